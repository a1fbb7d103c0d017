"""Columns of more than 64 mask words without a hole (4500 particles at rest in one
cell): particles that enter the cell diagonally, whose last streak is a finish
pass's, find rows past them."""
import numpy as np
import pytest

import oracle_lib
import states
from test_gpu_parity import DTYPES, _name, assert_particles_bitwise, sim_from_state

pytestmark = pytest.mark.gpu


# the stages after the particle passes as launches of a wave per cell's passes, and
# of a lane's
@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
@pytest.mark.parametrize("grid", [(4, 4, 1), (20, 21, 22)], ids=lambda g: "x".join(map(str, g)))
def test_diagonal_arrivals(grid, dtype):
    nx, ny, nz = grid
    rest, moving = 4500, 40
    _, k = states.random_state(1, 1, 1, 1, dtype, seed=1, cdt=(0.9, 0.85, 0.8))
    st = oracle_lib.OracleState(nx, ny, nz, rest + moving, dtype)
    rng = np.random.default_rng(8)
    sy, sz = nx + 2, (nx + 2) * (ny + 2)
    st.cell[:rest] = 2 + 2 * sy + sz
    st.cell[rest:] = 1 + sy + sz  # across an edge
    for m in ("x", "y", "z"):
        st.p[m][:] = rng.uniform(-0.5, 0.5, rest + moving)
    for m in ("x", "y"):
        st.p[m][rest:] = rng.uniform(0.6, 0.9, moving)
    st.p["ux"][rest:] = st.p["uy"][rest:] = 1
    st.p["w"][:] = 1
    st.load_interpolator()
    with sim_from_state(st) as sim:
        sim.load_interpolator_array()
        sim.clear_accumulator_array()
        sim.push(**k)
        st.clear_accumulator()
        assert st.push(**k) == moving
        assert np.count_nonzero(st.cell == 2 + 2 * sy + sz) == rest + moving
        assert sim.device_errors() == 0
        assert_particles_bitwise(sim.download_particles(), st)
