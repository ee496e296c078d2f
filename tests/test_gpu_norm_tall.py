"""Norm ops on tall F32 images (8 Mpx and more, under 2048 columns): window sums of squares within the
tiles, so that a NaN or a far brighter pixel at the top stays there."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.gpu_util import band_oracle, run_op, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ocip():
    from openclipp_amd import ocip as mod
    ctx = mod.initialize()
    yield mod
    mod.lib.ocipUninitialize(ctx)


# sums of n terms of one sign, each step at most 2^-23 of them, and the result's rounding
@pytest.mark.parametrize("split", ["0", None])
@pytest.mark.parametrize("op,code", [("SqrDistance_Norm", orc.SSD_NORM), ("CrossCorr_Norm", orc.CC_NORM)])
def test_top_stays_at_the_top(ocip, monkeypatch, op, code, split):
    if split is None:
        monkeypatch.delenv("OCIP_SPLIT_NCC", raising=False)
    else:
        monkeypatch.setenv("OCIP_SPLIT_NCC", split)
    rng = np.random.default_rng(16)
    src = rng.random((4200, 2000), dtype=np.float32)
    tpl = rng.random((16, 16), dtype=np.float32)
    say("tall", op, split)
    src[5, 6] = 1e8
    got = run_op(ocip, op, src, tpl)[2000:2040]
    want = band_oracle(lambda crop: orc.prox_f64(code, crop, tpl), src, tpl, 2000, 2040)
    e = np.abs(got - want) / ((tpl.size + 4) * 2.0 ** -23 * np.abs(want))
    assert np.all(e <= 1), float(np.max(e))
    src[5, 6] = np.nan
    # its windows, and within the tile of 64 rows by 32 columns what the running sums carry it to
    nan = np.isnan(run_op(ocip, op, src, tpl))
    assert nan[:14, :15].all() and not nan[64:].any() and not nan[:, 32:].any()
