"""CrossCorr_Norm of F32 images on split-FP16 MFMA (OCIP_SPLIT_NCC=1 has it take every call that
it can, 0 turns it off) against FP64.

Bound: each operand is held to 2^-24 of itself (2^-40 of the image's largest value, which the dark
windows below do not see: they are computed again in FP32), lo lo is left out (2^-24), and the
n products and their partial sums round in FP32, each step at most 2^-23 of the sum so far
(the matrix cores align their addends to the largest):
    |got - f64| <= (4 + n + 16) 2^-23 sum|s t| / sqrt(SS TT) + 2^-22 |f64|.
"""
import os

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


@pytest.fixture
def split(monkeypatch):
    return lambda on: monkeypatch.setenv("OCIP_SPLIT_NCC", "1" if on else "0")


def reference(src, tpl):
    """FP64 map and the bound."""
    s, t = src.astype(np.float64), tpl.astype(np.float64)
    want = orc.prox_f64(orc.CC_NORM, src, tpl)
    ss = orc.prox_f64(orc.CC, s * s, np.ones_like(t))
    den = np.sqrt(ss * (t * t).sum())
    with np.errstate(divide="ignore", invalid="ignore"):
        mag = orc.prox_f64(orc.CC, np.abs(s), np.abs(t)) / den
    return want, (20 + t.size) * 2.0 ** -23 * mag + 2.0 ** -22 * np.abs(want), ss


# widths around the 16-column chunks, heights around the row pairs, images around the 127 x 64
# tiles, aligned and unaligned rows
@pytest.mark.parametrize("shape,tshape", [
    ((1, 1), (1, 1)), ((127, 64), (2, 16)), ((128, 65), (3, 17)), ((129, 63), (1, 33)),
    ((140, 200), (64, 64)), ((255, 131), (31, 49)), ((200, 130), (97, 97)), ((260, 90), (256, 5)),
    ((300, 260), (5, 5))])
def test_against_fp64(ocip, split, shape, tshape):
    rng = np.random.default_rng(shape[0] * 1000 + tshape[1])
    src = rng.normal(0.2, 1.0, shape).astype(np.float32)
    tpl = rng.normal(0.2, 1.0, tshape).astype(np.float32)
    say("split ncc", shape, tshape)
    split(True)
    got = run_op(ocip, "CrossCorr_Norm", src, tpl)
    want, tol, _ = reference(src, tpl)
    assert np.all(np.abs(got - want) <= tol), float(np.max(np.abs(got - want) / tol))


@pytest.mark.parametrize("scale", [2.0 ** -50, 1.0, 2.0 ** 45])
def test_dark_windows_keep_their_accuracy(ocip, split, scale):
    """One bright pixel, 2^21 times the rest: the windows without it are as accurate as any."""
    rng = np.random.default_rng(21)
    src = rng.random((300, 280), dtype=np.float32) + np.float32(0.1)
    src[150, 200] = 2.0 ** 21
    src = (src * np.float32(scale)).astype(np.float32)
    tpl = rng.random((33, 31), dtype=np.float32)
    split(True)
    got = run_op(ocip, "CrossCorr_Norm", src, tpl)
    want, tol, ss = reference(src, tpl)
    # the FP64 integral behind SS: 2^-50 of the image's energy
    tol = tol + np.abs(want) * 2.0 ** -50 * (src.astype(np.float64) ** 2).sum() / ss
    assert np.all(np.abs(got - want) <= tol), float(np.max(np.abs(got - want) / tol))


@pytest.mark.parametrize("where", ["source nan", "source inf", "template inf", "huge", "tiny", "zero"])
def test_what_the_split_cannot_hold_is_the_plain_path(ocip, split, where):
    rng = np.random.default_rng(5)
    src = rng.random((200, 140), dtype=np.float32)
    tpl = rng.random((40, 35), dtype=np.float32)
    if where == "source nan":
        src[60, 70] = np.nan
    elif where == "source inf":
        src[60, 70] = np.inf
    elif where == "template inf":
        tpl[3, 4] = -np.inf
    elif where == "huge":
        src *= np.float32(2.0 ** 100)
        tpl *= np.float32(2.0 ** 27)
    elif where == "tiny":
        src *= np.float32(2.0 ** -70)
        tpl *= np.float32(2.0 ** -60)
    else:
        src[:] = 0
    split(False)
    plain = run_op(ocip, "CrossCorr_Norm", src, tpl)
    split(True)
    np.testing.assert_array_equal(run_op(ocip, "CrossCorr_Norm", src, tpl), plain)
