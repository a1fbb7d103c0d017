"""A particle whose squared momentum exceeds the single-precision range has an
infinite Lorentz factor and stays where it is.  Its derivatives are those of a
particle at rest in its cell, not NaN: without fields the outputs' tangents are
the inputs', and the inputs' adjoints the outputs', bit for bit."""
import numpy as np
import pytest

import states
from cabanapic_amd import Adjoint
from test_gpu_parity import DTYPES, _name, sim_from_state
from test_gpu_tangent import assert_same_bits, tangent_from_state

pytestmark = pytest.mark.gpu


def _state(dtype):
    st, k = states.random_state(4, 3, 5, 6, dtype, seed=21)
    st.fields[:] = 0
    fast = np.arange(0, st.np, 7)
    for n, m in enumerate(("ux", "uy", "uz")):
        st.p[m][fast[n::3]] = dtype(-3e19 if n == 1 else 3e19)
    return st, k, fast


@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
def test_tangent(dtype):
    st, k, fast = _state(dtype)
    t = np.random.default_rng(22).standard_normal((6, st.np))
    with tangent_from_state(st, tpart=t) as ts:
        for sim in (ts.primal, ts.tangent):
            sim.load_interpolator_array()
            sim.clear_accumulator_array()
        ts.push(**k)
        got = ts.download_particles()
        tacc = ts.tangent.download_accumulators()
        assert ts.primal.device_errors() == 0
    assert np.isfinite(got["tangent"]).all() and np.isfinite(tacc).all()
    assert_same_bits(got["tangent"][:, fast] + 0.0, t[:, fast], "tangents")
    for m in states.MEMBERS:
        assert_same_bits(got[m][fast], st.p[m][fast], m)


@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
def test_adjoint(dtype):
    st, _, fast = _state(dtype)
    seed = np.random.default_rng(23).standard_normal((6, st.np))
    with sim_from_state(st) as sim, Adjoint(sim) as adj:
        adj.forward(states.step_consts(dtype), 1, 1)
        gf, gp = adj.backward(np.zeros((9, st.ng)), seed)
        assert sim.device_errors() == 0
    assert np.isfinite(gp).all() and np.isfinite(gf).all()
    assert_same_bits(gp[:, fast] + 0.0, seed[:, fast], "adjoints")
