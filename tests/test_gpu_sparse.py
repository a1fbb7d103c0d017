"""Few particles in many cells (fewer than 4 bytes a cell of them): downloads,
steps and snapshots hold every particle, and it equals the oracle's bit for bit."""
import numpy as np
import pytest

import oracle_lib
import states
from cabanapic_amd import Simulation
from test_gpu_parity import DTYPES, _name, assert_particles_bitwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
@pytest.mark.parametrize("grid,n", [((16, 16, 16), 1), ((20, 20, 20), 300), ((33, 32, 32), 7),
                                    ((64, 64, 33), 5000)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_few_particles(grid, n, dtype):
    nx, ny, nz = grid
    one, k = states.random_state(nx, ny, nz, 1, dtype, seed=n)
    keep = np.random.default_rng(n).permutation(one.np)[:n]
    st = oracle_lib.OracleState(nx, ny, nz, n, dtype)
    st.fields[:] = one.fields
    for m in states.MEMBERS:
        st.p[m][:] = one.p[m][keep]
    st.cell[:] = one.cell[keep]
    with Simulation(nx, ny, nz, n, dtype) as sim:
        sim.upload_fields(st.fields)
        sim.upload_particles(*[st.p[m] for m in states.MEMBERS], st.cell)
        assert_particles_bitwise(sim.download_particles(), st)
        assert sorted(sim.download_particle_tags()) == list(range(n))
        st.load_interpolator()
        sim.load_interpolator_array()
        for _ in range(3):
            sim.clear_accumulator_array()
            sim.push(**k)
            st.clear_accumulator()
            st.push(**k)
        got, tags = sim.download_particles(), sim.download_particle_tags()
        sim.snapshot_begin(0)
        snap = sim.snapshot_wait(0)
        assert sim.device_errors() == 0
    assert_particles_bitwise(got, st)
    assert np.array_equal(snap["x"][tags], got["x"]) and np.array_equal(snap["cell"][tags], got["cell"])
