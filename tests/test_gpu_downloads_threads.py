"""Two threads that download at the same time, one of them through the ring:
every download of both completes, and with the right values."""
import threading

import numpy as np
import pytest

from cabanapic_amd import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [50, 75])
def test_every_download_completes(n):
    done, errors = [], []

    def work(k):
        try:
            with Simulation(n, n, n, 0, np.float64) as sim:
                f = np.random.default_rng(k).standard_normal((9, sim.ncells))
                sim.upload_fields(f)
                for _ in range(4):
                    done.append((k, np.array_equal(sim.download_fields(), f)))
        except Exception as e:  # noqa: BLE001 (whatever it is, the test is to name it)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    assert sorted(done) == [(k, True) for k in range(2) for _ in range(4)]
