"""The passes whose rows and arrivals several waves share, and those with a wave
per cell, at the sizes where they can go wrong: groups of 64 cells that are
partly filled, columns around a mask word and past what one chunk of words
holds, columns too deep for LDS, both wave counts (up to 512 groups of cells, and more), 4096 cells and
4097, 8192 of 31 and 32 particles and 8193, more arrivals than lanes, and steps without some of the energies.  Particles equal the oracle's bit for bit;
accumulators agree within the bound of a reordered sum (as in
test_gpu_parity.py)."""
import numpy as np
import pytest

import states
from cabanapic_amd import Simulation
from test_gpu_parity import DTYPES, _name, assert_bitwise, assert_particles_bitwise, sim_from_state

pytestmark = pytest.mark.gpu

# nx, ny, nz, particles per cell, column rows asked for, pushes
CASES = [
    (1, 1, 1, 1, 0, 3), (63, 1, 1, 3, 0, 3), (64, 1, 1, 63, 0, 2), (65, 1, 1, 65, 0, 2),
    (5, 13, 1, 2, 0, 3), (3, 2, 1, 300, 0, 3), (4, 1, 1, 9, 4200, 3),
    (32, 32, 32, 2, 0, 2), (33, 32, 32, 2, 0, 2),
    (16, 16, 16, 9, 0, 2), (241, 17, 1, 9, 0, 2), (3, 2, 1, 900, 0, 3),
    (63, 1, 1, 3, 4200, 3), (3, 1, 1, 1500, 0, 3), (241, 17, 1, 1, 0, 3),
    (241, 17, 1, 65, 0, 2), (241, 17, 1, 300, 0, 2),
    (64, 16, 8, 31, 0, 2), (64, 16, 8, 32, 0, 2), (2731, 3, 1, 32, 0, 2), (2731, 3, 1, 65, 0, 2),
    (2731, 3, 1, 300, 0, 2),
]


@pytest.mark.parametrize("compensated", [False, True], ids=["plain", "compensated"])
@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])))
def test_shared_passes(case, dtype, compensated):
    nx, ny, nz, ppc, rows, pushes = case
    st, k = states.random_state(nx, ny, nz, ppc, dtype, seed=nx + ppc)
    st.load_interpolator()
    sim = Simulation(nx, ny, nz, st.np, dtype, column_rows=rows)
    sim.upload_fields(st.fields)
    sim.upload_particles(*[st.p[m] for m in ("x", "y", "z", "ux", "uy", "uz", "w")], st.cell)
    sim.set_compensated_deposit(compensated)
    with sim:
        assert sim.column_rows() >= rows
        sim.load_interpolator_array()
        movers = 0
        for _ in range(pushes):
            sim.clear_accumulator_array()
            sim.push(**k)
            st.clear_accumulator()
            absacc = np.zeros(st.acc.size)
            movers = st.push(**k, abs_acc=absacc)
        assert sim.last_push_movers() == movers
        assert sim.device_errors() == 0
        assert_particles_bitwise(sim.download_particles(), st)
        acc = sim.download_accumulators()
    eps = np.finfo(dtype).eps
    err = np.abs(acc.astype(np.float64) - st.acc.reshape(acc.shape).astype(np.float64))
    assert np.all(err <= 64 * eps * absacc.reshape(acc.shape) + np.finfo(dtype).tiny)


@pytest.mark.parametrize("dtype", DTYPES, ids=_name)
@pytest.mark.parametrize("energy,kinetic,steps", [(1, 0, 70), (3, 2, 7), (0, 3, 4), (5, 0, 4)])
def test_energy_rows_of_a_fused_run(dtype, energy, kinetic, steps):
    """The history of one call equals that of a call per step (whose rows are
    summed one at a time), bit for bit, whichever energies are asked for."""
    st, _ = states.random_state(6, 5, 4, 4, dtype, seed=3)
    k = states.step_consts(dtype)
    out = []
    for calls in (1, steps):
        with sim_from_state(st) as sim:
            if calls == 1:
                out.append(sim.step(dict(k, energy_interval=energy, kinetic_interval=kinetic), steps))
                continue
            rows = [sim.step(dict(k, energy_interval=1, kinetic_interval=1), 1) for _ in range(steps)]
            ref = np.concatenate(rows)
            for s in range(1, steps + 1):
                if not energy or s % energy:
                    ref[s - 1, :2] = np.nan
                if not kinetic or s % kinetic:
                    ref[s - 1, 2] = np.nan
            out.append(ref)
    assert_bitwise(np.nan_to_num(out[0], nan=-1.0), np.nan_to_num(out[1], nan=-1.0), "history")
