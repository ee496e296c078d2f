"""CrossCorr_Norm of F32 images on split-FP16 MFMA (OCIP_SPLIT_NCC=1) where one pixel is many orders of
magnitude above the others: values that the split rounds to zero are computed in FP32, exact
zeros are not.

Bound at windows without the pixel, which come before it in the image so that their sums of
squares have none of its rounding: operands to 2^-23 of themselves, n products and their
partial sums at 2^-23 each, the result's rounding:
    |got - f64| <= (n + 20) 2^-23 sum|s t| / sqrt(SS TT) + 2^-22 |f64|.
"""
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


def bound(src, tpl):
    """FP64 map and the bound."""
    s, t = src.astype(np.float64), tpl.astype(np.float64)
    want = orc.prox_f64(orc.CC_NORM, src, tpl)
    ss = orc.prox_f64(orc.CC, s * s, np.ones_like(t))
    with np.errstate(divide="ignore", invalid="ignore"):
        mag = orc.prox_f64(orc.CC, np.abs(s), np.abs(t)) / np.sqrt(ss * (t * t).sum())
    return want, (20 + t.size) * 2.0 ** -23 * mag + 2.0 ** -22 * np.abs(want)


# ratios below, at and far above the split's reach (2^40); the dark values positive, or a noise
# around zero whose sums cancel
@pytest.mark.parametrize("bright", [2.0 ** 15, 2.0 ** 25, 2.0 ** 39, 2.0 ** 45, 1e20])
@pytest.mark.parametrize("signed", [False, True])
def test_values_that_the_split_rounds_away(ocip, monkeypatch, bright, signed):
    rng = np.random.default_rng(45)
    src = rng.random((300, 280), dtype=np.float32) - np.float32(0.5 if signed else -0.1)
    src[299, 279] = bright
    tpl = rng.random((33, 31), dtype=np.float32)
    say("split wide range", bright, signed)
    monkeypatch.setenv("OCIP_SPLIT_NCC", "1")
    got = run_op(ocip, "CrossCorr_Norm", src, tpl)[:280, :260]
    want, tol = (m[:280, :260] for m in bound(src, tpl))
    assert np.all(np.abs(got - want) <= tol), float(np.max(np.abs(got - want) / tol))


def test_exact_zeros_stay_on_the_split(ocip, monkeypatch):
    """Zero windows beside bright ones: the split's own map (not the FP32 kernel's, bit for bit)."""
    rng = np.random.default_rng(46)
    src = np.zeros((300, 280), np.float32)
    src[20:120, 20:120] = rng.random((100, 100), dtype=np.float32) + np.float32(0.5)
    tpl = rng.random((33, 31), dtype=np.float32)
    say("split zeros")
    maps = []
    for on in ("0", "1"):
        monkeypatch.setenv("OCIP_SPLIT_NCC", on)
        maps.append(run_op(ocip, "CrossCorr_Norm", src, tpl)[20:120, 20:120])
    assert np.any(maps[0] != maps[1])
    want, tol = (m[20:120, 20:120] for m in bound(src, tpl))
    assert np.all(np.abs(maps[1] - want) <= tol)
