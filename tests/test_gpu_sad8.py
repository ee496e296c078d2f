"""AbsDistance of 8-bit images on the byte-transposed tile: template widths around its 16-column
blocks, images narrower than one 16-byte load and across the tile's edges, tall templates (several
LDS bands), 1 to 4 channels.  Bit for bit the exact int64 sums of each channel."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.gpu_util import run_op, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ocip():
    from openclipp_amd import ocip as mod
    ctx = mod.initialize()
    yield mod
    mod.lib.ocipUninitialize(ctx)


@pytest.mark.parametrize("dtype", [np.uint8, np.int8])
@pytest.mark.parametrize("shape,tshape", [((1, 1), (1, 1)), ((9, 13), (3, 13)), ((65, 33), (5, 15)),
                                          ((70, 95), (4, 16)), ((64, 130), (7, 17)),
                                          ((129, 66), (31, 31)), ((200, 140), (190, 33)),
                                          ((80, 2050), (9, 6))])
def test_exact_sums(ocip, dtype, shape, tshape):
    rng = np.random.default_rng(shape[1] * 10 + tshape[1])
    info = np.iinfo(dtype)
    for channels in (1, 2, 3, 4) if shape[1] < 200 else (1,):
        src = rng.integers(info.min, info.max, size=shape + (channels,), endpoint=True).astype(dtype)
        tpl = rng.integers(info.min, info.max, size=tshape + (channels,), endpoint=True).astype(dtype)
        say("sad8", np.dtype(dtype).name, shape, tshape, channels)
        squeeze = (lambda a: a[..., 0].copy()) if channels == 1 else (lambda a: a)
        got = run_op(ocip, "AbsDistance", squeeze(src), squeeze(tpl)).reshape(src.shape)
        for c in range(channels):
            exact = orc.f64_from_i64(orc.SAD, src[..., c].copy(), tpl[..., c].copy())
            np.testing.assert_array_equal(got[..., c], exact.astype(np.float32))
