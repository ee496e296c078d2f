"""CrossCorr_Norm of F32 images on split-FP16 MFMA keeps at least the accuracy of the FP32 sums."""
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


# hi = 1 and lo = 2^-11 hold every value exactly, and the products of the two lo, all alike, are the
# whole difference between the exact sums and those of the other products
@pytest.mark.parametrize("tshape", [(5, 5), (8, 8), (11, 11), (16, 16), (24, 24)])
def test_products_of_the_low_parts(ocip, monkeypatch, tshape):
    src, tpl = (np.full(s, 1 + 2.0 ** -11, np.float32) for s in ((140, 150), tshape))
    say("split low parts", tshape)
    want = orc.prox_f64(orc.CC_NORM, src, tpl)
    worst = []
    for on in ("0", "1"):
        monkeypatch.setenv("OCIP_SPLIT_NCC", on)
        worst.append(np.max(np.abs(run_op(ocip, "CrossCorr_Norm", src, tpl) - want)))
    assert worst[1] <= worst[0], worst


@pytest.mark.parametrize("tshape", [(8, 8), (25, 8), (20, 5), (2, 50), (16, 16), (33, 64)])
@pytest.mark.parametrize("kind", ["noise", "signed", "levels"])
def test_no_further_from_fp64_than_fp32_sums(ocip, monkeypatch, kind, tshape):
    rng = np.random.default_rng(tshape[1])
    draw = {"noise": lambda s: rng.normal(0.5, 0.2, s).clip(0, 1), "signed": lambda s: rng.normal(0, 1, s),
            "levels": lambda s: rng.integers(0, 256, s) / 255}[kind]
    src, tpl = draw((220, 210)).astype(np.float32), draw(tshape).astype(np.float32)
    say("split accuracy", kind, tshape)
    want = orc.prox_f64(orc.CC_NORM, src, tpl)
    rms = []
    for on in ("0", "1"):
        monkeypatch.setenv("OCIP_SPLIT_NCC", on)
        rms.append(np.sqrt(np.mean((run_op(ocip, "CrossCorr_Norm", src, tpl) - want) ** 2)))
    assert rms[1] <= rms[0], rms
