"""A large download does not wait for the GPU driver to clear memory given
back before it (it uses the copy engines for that): right after a context
of some GB is closed it takes the time that it takes at rest."""
import ctypes
import time

import numpy as np
import pytest

from cabanapic_amd import Simulation

pytestmark = pytest.mark.gpu


def _seconds(sim, out):
    t = time.perf_counter()
    assert sim.lib.cpic_download_fields(sim._h, out.ctypes.data_as(ctypes.c_void_p)) == 0
    return time.perf_counter() - t


def test_after_a_large_context_is_closed():
    with Simulation(101, 101, 101, 0, np.float64) as sim:
        f = np.random.default_rng(1).standard_normal((9, sim.ncells))
        sim.upload_fields(f)
        out = np.zeros_like(f)
        after = []
        for _ in range(3):
            time.sleep(0.5)
            rest = min(_seconds(sim, out) for _ in range(5))
            Simulation(320, 320, 320, 0, np.float32).close()  # 5 GB
            after.append(_seconds(sim, out) / rest)
        assert np.array_equal(out, f)
    # (3.7 times as long by the copy engines)
    assert min(after) < 2, after


# the piece's alignment (16, 8 and 4 bytes) and length: particle arrays of an odd
# number follow one another in the staging area
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1048577, 1100002, 2097155])
def test_arrays_of_any_alignment(n, dtype):
    rng = np.random.default_rng(n)
    p = [rng.standard_normal(n).astype(dtype) for _ in range(7)]
    cell = np.sort(rng.integers(0, 1000, n))
    cell = (cell % 10 + 1 + 12 * (cell // 10 % 10 + 1 + 12 * (cell // 100 + 1))).astype(np.int32)
    with Simulation(10, 10, 10, n, dtype) as sim:
        sim.upload_particles(*p, cell)
        got, tags = sim.download_particles(), sim.download_particle_tags()
    for want, have in zip(p + [cell], got.values()):
        assert np.array_equal(have, want[tags])
