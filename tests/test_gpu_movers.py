"""last_push_movers is the last push's count, whatever kernels ran before it on
the same columns and whatever became of the columns since: uploads of another
number of particles whose push takes other kernels (a wave per cell, or a lane,
on 4097 to 8192 cells), grown columns, columns laid out anew."""
import numpy as np
import pytest

import states
from test_gpu_parity import DTYPES, _name, sim_from_state

pytestmark = pytest.mark.gpu


def _pushed(sim, st, k):
    """One push of st's particles on the context and on the oracle: (count of
    the device, count of the oracle)."""
    sim.upload_fields(st.fields)
    sim.upload_particles(*[st.p[m] for m in states.MEMBERS], st.cell)
    st.load_interpolator()
    sim.load_interpolator_array()
    sim.clear_accumulator_array()
    st.clear_accumulator()
    sim.push(**k)
    return sim.last_push_movers(), st.push(**k)


# the groups of 64 cells fill the last block's 256 cells partly in the first
# three, wholly in the last
@pytest.mark.parametrize("grid", [(17, 17, 17), (20, 20, 20), (4160, 1, 1), (64, 16, 8)],
                         ids=lambda g: "x".join(map(str, g)))
def test_upload_that_changes_the_kernels(grid):
    many, k = states.random_state(*grid, 33, np.float32, seed=7)
    few, _ = states.random_state(*grid, 31, np.float32, seed=8)
    with sim_from_state(many) as sim:
        rows = sim.column_rows()
        for st in (many, few, many):
            got, want = _pushed(sim, st.copy(), k)
            assert want > 0 and got == want
            assert sim.column_rows() == rows
        assert sim.device_errors() == 0


@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
@pytest.mark.parametrize("grid", [(6, 5, 4, 8), (33, 16, 17, 9)],
                         ids=lambda g: "x".join(map(str, g)))
def test_count_outlives_the_columns(grid, dtype):
    nx, ny, nz, ppc = grid
    st, k = states.random_state(nx, ny, nz, 4 * ppc, dtype, seed=9)
    first = np.arange(nx * ny * nz * ppc)
    with sim_from_state(st) as sim:
        sim.upload_particles(*[st.p[m][first] for m in states.MEMBERS], st.cell[first])
        sim.load_interpolator_array()
        sim.push(**k)
        moved = sim.last_push_movers()
        assert moved > 0
        rows = sim.column_rows()
        sim.reserve_column_rows(rows + 64)
        assert sim.column_rows() > rows
        assert sim.last_push_movers() == moved
        # all particles: columns of other capacities
        sim.upload_particles(*[st.p[m] for m in states.MEMBERS], st.cell)
        assert sim.last_push_movers() == moved
        sim.upload_particles(*[st.p[m][:0] for m in states.MEMBERS], st.cell[:0])
        assert sim.last_push_movers() == moved
        # a push of no particles moves none
        sim.push(**k)
        assert sim.last_push_movers() == 0
