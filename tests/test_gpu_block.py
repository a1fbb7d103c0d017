"""Steps whose stages after the particle passes run in one workgroup, against the
launches of the general path (which a timed stage selects): everything that a run
leaves equals bit for bit.  Sizes at the limit of 1024 cells and one more, partly
filled waves and blocks, one cell, several calls, many steps, particles fast enough
for records of every crossing and for the overflow list."""
import numpy as np
import pytest

import states
from test_gpu_parity import DTYPES, _name, assert_bitwise, sim_from_state

pytestmark = pytest.mark.gpu

# nx, ny, nz, particles per cell, largest momentum, cdt, energy interval,
# kinetic interval, steps of the calls
SLOW, FAST = (0.45, 0.4, 0.35), (0.9, 0.85, 0.8)
CASES = [
    (1, 1, 1, 1, 0.6, SLOW, 1, 0, (1, 3)), (1, 1, 1, 12, 4.0, FAST, 1, 1, (3,)),
    (32, 1, 1, 64, 0.6, SLOW, 1, 0, (1, 1, 6)), (1, 37, 1, 20, 0.6, SLOW, 2, 3, (7, 6)),
    (16, 16, 1, 12, 4.0, FAST, 1, 3, (4,)), (257, 1, 1, 9, 0.6, SLOW, 3, 0, (5, 4)),
    (3, 2, 1, 300, 0.6, SLOW, 1, 0, (4,)), (6, 5, 4, 12, 4.0, FAST, 0, 2, (3,)),
    (17, 1, 1, 33, 0.6, SLOW, 1, 0, (300,)), (10, 10, 10, 9, 4.0, FAST, 1, 2, (3,)),
    (16, 16, 4, 5, 0.6, SLOW, 1, 0, (1, 4)), (1025, 1, 1, 5, 0.6, SLOW, 1, 0, (3,)),
]


def _run(st, case, dtype, compensated, timed):
    k = states.step_consts(dtype, cdt=case[5])
    with sim_from_state(st) as sim:
        sim.set_compensated_deposit(compensated)
        sim.set_timing(timed)
        hist = [sim.step(dict(k, energy_interval=case[6], kinetic_interval=case[7]), n)
                for n in case[8]]
        out = dict(history=np.nan_to_num(np.concatenate(hist), nan=-1.0),
                   fields=sim.download_fields(), accumulators=sim.download_accumulators(),
                   interpolators=sim.download_interpolators(), movers=sim.last_push_movers(),
                   errors=sim.device_errors())
        out.update(sim.download_particles())
        out["tags"] = sim.download_particle_tags()
    return out


@pytest.mark.parametrize("compensated", [False, True], ids=["plain", "compensated"])
@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:4])))
def test_steps_in_a_block(case, dtype, compensated):
    nx, ny, nz, ppc, umax, cdt = case[:6]
    st, _ = states.random_state(nx, ny, nz, ppc, dtype, seed=nx + ppc, umax=umax, cdt=cdt)
    # weak charges: the fields stay of the size they have
    st.p["w"][:] *= dtype(1e-4)
    got = _run(st, case, dtype, compensated, False)
    ref = _run(st, case, dtype, compensated, True)
    assert got["errors"] == ref["errors"] == 0
    assert np.isfinite(got["fields"]).all()
    assert got["movers"] == ref["movers"]
    for name, want in ref.items():
        if isinstance(want, np.ndarray):
            assert_bitwise(got[name], want, name)


@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
@pytest.mark.parametrize("case", [(1, 1, 1, 500), (3, 2, 1, 300), (10, 3, 11, 200)],
                         ids=lambda c: "x".join(map(str, c)))
def test_overflow_in_a_block(case, dtype):
    """One step whose records overflow the lists: their deposits are atomic, so
    the particles agree as a set and the accumulators within the bound of a
    reordered sum of the 12 streak contributions of at most 4 streaks."""
    nx, ny, nz, ppc = case
    st, _ = states.random_state(nx, ny, nz, ppc, dtype, seed=5, umax=4.0, cdt=FAST)
    got, ref = (_run(st, case + (4.0, FAST, 1, 0, (1,)), dtype, False, timed)
                for timed in (False, True))
    assert got["errors"] == ref["errors"] == 0
    assert got["movers"] == ref["movers"]
    a, b = states.canonical(got), states.canonical(ref)
    for m in states.MEMBERS + ("cell",):
        assert_bitwise(a[m], b[m], m)
    # |q| <= 1.5, displacement below 1, (1 +- mid) below 2, v5 below 1/3: no
    # contribution exceeds 7; a cell sees at most every streak of its row's
    # particles and of its neighbours'
    bound = 64 * np.finfo(dtype).eps * 7 * 4 * 7 * 2 * ppc
    assert np.abs(got["accumulators"].astype(float) - ref["accumulators"]).max() <= bound
