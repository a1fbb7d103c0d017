"""cpic_field_energies_noalloc equals cpic_energies bit for bit on grids of more
voxels than its 4096 blocks have threads, too."""
import numpy as np
import pytest

from cabanapic_amd import Simulation, load_library
from test_zz_no_alloc import Hip, _fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("grid", [(128, 128, 64), (129, 128, 64), (131, 127, 129)],
                         ids=lambda g: "x".join(map(str, g)))
def test_noalloc_energies_match_context(grid, dtype):
    hip = Hip()
    lib = load_library()
    f = _fields(*grid, dtype, seed=5)
    with Simulation(*grid, 0, dtype) as sim:
        sim.upload_fields(f)
        expect = np.array(sim.energies())
    dev_f, dev_out = hip.malloc(f.nbytes), hip.malloc(16)
    got = np.zeros(2)
    try:
        hip.upload(dev_f, f)
        assert lib.cpic_field_energies_noalloc(dev_f, np.dtype(dtype).itemsize, *grid, dev_out,
                                               None) == 0
        hip.sync()
        hip.download(got, dev_out)
    finally:
        hip.free(dev_f)
        hip.free(dev_out)
    assert np.array_equal(got, expect), (got, expect)
