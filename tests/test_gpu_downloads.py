"""Large downloads go through a pinned ring that several threads empty: the
sizes around its threshold, its pieces and its length come back whole, from
two contexts at once too."""
import threading

import numpy as np
import pytest

from cabanapic_amd import Simulation

pytestmark = pytest.mark.gpu


# grids whose nine field arrays are just under and over 4 MB (the threshold),
# over 16 MB (the ring) and an odd size beyond it
GRIDS = [(46, 46, 46), (47, 47, 47), (75, 75, 75), (101, 67, 83)]


def _fields(sim, seed):
    return np.random.default_rng(seed).standard_normal((9, sim.ncells)).astype(sim.dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_fields_come_back(grid, dtype):
    with Simulation(*grid, 0, dtype) as sim:
        for seed in (1, 2):
            f = _fields(sim, seed)
            sim.upload_fields(f)
            assert np.array_equal(sim.download_fields(), f)


def test_two_contexts_at_once():
    sims = [Simulation(75, 75, 75, 0, np.float64) for _ in range(2)]
    bad = []

    def work(k):
        f = _fields(sims[k], k)
        sims[k].upload_fields(f)
        for _ in range(4):
            if not np.array_equal(sims[k].download_fields(), f):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in sims:
        s.close()
    assert not bad
