"""8-bit images of 2, 3 (colour) and 4 channels on the exact-integer MFMA path, every channel in
one launch from planes split off first, against the VALU kernel (OCIP_INT_MFMA=0) bit for bit
and the exact int64 sums of each channel."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.gpu_util import OP_CODE, run_op, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ocip():
    from openclipp_amd import ocip as mod
    ctx = mod.initialize()
    yield mod
    mod.lib.ocipUninitialize(ctx)


# widths around the 4-pixel groups and 16-byte planes, images around the 127 x 64 tiles, one pixel
@pytest.mark.parametrize("dtype", [np.uint8, np.int8])
@pytest.mark.parametrize("channels", [2, 3, 4])
@pytest.mark.parametrize("shape,tshape", [((1, 1), (1, 1)), ((30, 15), (4, 3)), ((128, 65), (17, 16)),
                                          ((140, 131), (24, 31)), ((254, 70), (97, 66))])
def test_channels_equal_the_valu_path(ocip, monkeypatch, dtype, channels, shape, tshape):
    rng = np.random.default_rng(shape[1] * 10 + channels)
    info = np.iinfo(dtype)
    src = rng.integers(info.min, info.max, size=shape + (channels,), endpoint=True).astype(dtype)
    tpl = rng.integers(info.min, info.max, size=tshape + (channels,), endpoint=True).astype(dtype)
    for op in ["CrossCorr", "SqrDistance", "CrossCorr_Norm", "SqrDistance_Norm"]:
        say("int channels", np.dtype(dtype).name, channels, shape, tshape, op)
        monkeypatch.delenv("OCIP_INT_MFMA", raising=False)
        got = run_op(ocip, op, src, tpl)
        monkeypatch.setenv("OCIP_INT_MFMA", "0")
        np.testing.assert_array_equal(got, run_op(ocip, op, src, tpl), err_msg=op)
        if not op.endswith("_Norm"):
            for c in range(channels):
                exact = orc.f64_from_i64(OP_CODE[op], src[..., c].copy(),
                                         tpl[..., c].copy()).astype(np.float32)
                np.testing.assert_array_equal(got[..., c], exact, err_msg=op)
