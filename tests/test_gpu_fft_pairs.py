"""The FFT proximity path's row pairs and workgroup shapes: odd numbers of source and template rows
(a last pair of one row), one-row images, and padded widths on both sides of the 5112 points
up to which two workgroups share a CU.  Same bound as test_gpu_fft."""
import numpy as np
import pytest

from tests.gpu_util import say
from tests.test_gpu_fft import check_map, run_fft

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ocip():
    from openclipp_amd import ocip as mod
    ctx = mod.initialize()
    yield mod
    mod.lib.ocipUninitialize(ctx)


@pytest.mark.parametrize("op", ["CrossCorr", "CrossCorr_Norm", "SqrDistance_Norm"])
@pytest.mark.parametrize("shape,tshape", [((1, 40), (1, 9)), ((2, 33), (1, 33)), ((9, 64), (8, 3)),
                                          ((3, 5000), (3, 64)), ((5, 5100), (2, 40)),
                                          ((4, 8300), (3, 500)), ((4200, 3), (77, 2))])
def test_pairs_and_shapes(ocip, op, shape, tshape):
    rng = np.random.default_rng(shape[0] + shape[1])
    src = (rng.random(shape) - 0.3).astype(np.float32)
    tpl = (rng.random(tshape) - 0.3).astype(np.float32)
    say("fft pairs", op, shape, tshape)
    check_map(op, src, tpl, run_fft(ocip, op, src, tpl))
