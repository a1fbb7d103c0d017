"""cpic_forward's history holds the energies of the steps that the intervals name
counted over the run, whatever the checkpoint interval: those of cpic_step on the
same state, and nothing else."""
import numpy as np
import pytest

import states
from cabanapic_amd import Adjoint
from test_gpu_parity import DTYPES, _name, sim_from_state

pytestmark = pytest.mark.gpu


# steps, checkpoint interval, energy interval, kinetic interval
@pytest.mark.parametrize("steps,keep,energy,kinetic", [(7, 3, 2, 0), (7, 3, 2, 5), (10, 4, 3, 2),
                                                       (6, 1, 4, 3), (9, 9, 2, 2), (5, 2, 0, 2)])
@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
@pytest.mark.parametrize("grid", [(6, 5, 4, 8), (33, 16, 17, 2)],
                         ids=lambda g: "x".join(map(str, g)))
def test_energies_of_the_named_steps(grid, dtype, steps, keep, energy, kinetic):
    st, _ = states.random_state(*grid, dtype, seed=12)
    st.p["w"][:] *= dtype(1e-3)
    k = dict(states.step_consts(dtype), energy_interval=energy, kinetic_interval=kinetic)
    with sim_from_state(st) as sim:
        want = sim.step(k, steps)
    with sim_from_state(st) as sim, Adjoint(sim) as adj:
        for _ in range(2):  # buffers anew and in place
            got = adj.forward(k, steps, keep)
            sim.upload_fields(st.fields)
            sim.upload_particles(*[st.p[m] for m in states.MEMBERS], st.cell)
            assert np.array_equal(np.isnan(got), np.isnan(want))
            # the columns are laid out anew at every checkpoint, so that the
            # deposits' order, and the FP32 sums' last bits, differ
            assert np.allclose(got, want, rtol=1e-5 if dtype == np.float32 else 1e-12,
                               equal_nan=True)
