"""Integrals of images whose last tile (32 rows by 256 columns) is ragged in each way, of unaligned
rows, of fewer than four columns, and of more tile rows than one pass of the carries holds in
registers (4096 rows).  Sums exact in FP64: 8- and 16-bit integers, and floats that are small
integers."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.gpu_util import say
from tests.test_gpu_integral import run_integral

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ocip():
    from openclipp_amd import ocip as mod
    ctx = mod.initialize()
    yield mod
    mod.lib.ocipUninitialize(ctx)


@pytest.mark.parametrize("dtype", [np.uint8, np.int16, np.float32])
@pytest.mark.parametrize("shape", [(31, 1), (33, 3), (32, 4), (40, 255), (64, 256), (65, 257),
                                   (17, 511), (4097, 5), (5000, 260)])
def test_ragged_tiles(ocip, dtype, shape):
    rng = np.random.default_rng(shape[0] + shape[1])
    src = rng.integers(0, 128, size=shape).astype(dtype)
    for sqr in (False, True):
        say("integral ragged", np.dtype(dtype).name, shape, sqr)
        exact = orc.integral_exact(src, sqr)
        np.testing.assert_array_equal(run_integral(ocip, src, sqr, np.float64), exact)
        np.testing.assert_array_equal(run_integral(ocip, src, sqr, np.float32),
                                      exact.astype(np.float32))
