"""The push's square roots and quotients over their whole range: momenta of every
size from zero and denormals to infinite squares, particles on faces, next to
them and in the middle.  Particles equal the oracle's, whose roots and quotients
are the C library's and the CPU's, bit for bit."""
import numpy as np
import pytest

import states
from test_gpu_parity import DTYPES, _name, assert_particles_bitwise, sim_from_state

pytestmark = pytest.mark.gpu


# a wave per cell, a lane per cell, and columns that are packed (the first push)
@pytest.mark.parametrize("grid", [(9, 8, 7, 40), (33, 16, 17, 24), (64, 64, 33, 2)],
                         ids=lambda g: "x".join(map(str, g)))
@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
def test_roots_and_quotients(grid, dtype):
    nx, ny, nz, ppc = grid
    st, k = states.random_state(nx, ny, nz, ppc, dtype, seed=nx, cdt=(0.9, 0.85, 0.8))
    rng = np.random.default_rng(31)
    st.fields *= dtype(1e-3)
    tiny = np.finfo(dtype).smallest_subnormal
    edge = [1, -1, 0, 1 - np.finfo(dtype).epsneg, -1 + np.finfo(dtype).epsneg, tiny, -tiny]
    for m in ("x", "y", "z"):
        at = rng.random(st.np) < 0.2
        st.p[m][at] = rng.choice(np.array(edge, dtype), int(at.sum()))
    for m in ("ux", "uy", "uz"):
        # mostly the sizes at which particles move and meet faces
        e = np.where(rng.random(st.np) < 0.6, rng.uniform(-9, 2, st.np), rng.uniform(-45, 25, st.np))
        u = (rng.choice([-1.0, 1.0], st.np) * 10.0 ** e).astype(dtype)
        u[rng.random(st.np) < 0.05] = 0
        st.p[m][:] = u
    st.load_interpolator()
    with sim_from_state(st) as sim:
        sim.load_interpolator_array()
        for _ in range(2):
            sim.clear_accumulator_array()
            sim.push(**k)
            st.clear_accumulator()
            assert st.push(**k) > 0
        assert sim.device_errors() == 0
        assert_particles_bitwise(sim.download_particles(), st)
