"""last_push_movers is the last push's count, whatever kernels ran before it on
the same columns: uploads of another number of particles whose push takes other
kernels (a wave per cell, or a lane, on 4097 to 8192 cells)."""
import numpy as np
import pytest

import states
from test_gpu_parity import sim_from_state

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
