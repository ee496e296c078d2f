"""Cross terms of 8- and 16-bit integer images as products of signed bytes: against exact integer
sums.  The largest and smallest values of each type are among the data (they reach every digit, the
both halves of 16-bit values included)."""
import numpy as np
import pytest

from tests.gpu_util import run_op, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ocip():
    from openclipp_amd import ocip as mod
    ctx = mod.initialize()
    yield mod
    mod.lib.ocipUninitialize(ctx)


def exact_sums(src, tpl):
    """int64 sum s t and sum s^2 over each output's window, zeros outside the image."""
    (H, W), (th, tw) = src.shape, tpl.shape
    pad = np.pad(src.astype(np.int64), ((th // 2, th), (tw // 2, tw)))
    win = np.lib.stride_tricks.sliding_window_view(pad, (th, tw))[:H, :W]
    t = tpl.astype(np.int64)
    cross = np.stack([np.tensordot(row, t, 2) for row in win])
    return cross, np.stack([(row * row).sum((1, 2)) for row in win])


def image(rng, dtype, shape):
    info = np.iinfo(dtype)
    edge = np.array([info.min, info.min + 1, info.max - 1, info.max, 0, 127, 128 & info.max], dtype)
    a = rng.integers(info.min, info.max, size=shape, endpoint=True).astype(dtype)
    return np.where(rng.random(shape) < 0.4, rng.choice(edge, size=shape), a).astype(dtype)


# widths around the 32-column chunks (tw 17, 18, 49, 50, 81, 82, 113), odd and even rows, images around
# the 127-row tiles of 32 (16-bit) and 64 columns, one pixel
@pytest.mark.parametrize("dtype", [np.uint8, np.int8, np.uint16, np.int16])
@pytest.mark.parametrize("shape,tshape", [((1, 1), (1, 1)), ((20, 19), (5, 17)), ((126, 33), (8, 18)),
                                          ((128, 65), (31, 49)), ((255, 96), (1, 50)),
                                          ((130, 131), (64, 81)), ((97, 129), (97, 82)),
                                          ((140, 117), (128, 113)), ((131, 120), (129, 114))])
def test_sums_are_exact(ocip, dtype, shape, tshape):
    rng = np.random.default_rng(shape[1] + tshape[1])
    src, tpl = image(rng, dtype, shape), image(rng, dtype, tshape)
    cross, ss = exact_sums(src, tpl)
    tt = int((tpl.astype(np.int64) ** 2).sum())
    say("int8 products", np.dtype(dtype).name, shape, tshape)
    np.testing.assert_array_equal(run_op(ocip, "CrossCorr", src, tpl), cross.astype(np.float32))
    np.testing.assert_array_equal(run_op(ocip, "SqrDistance", src, tpl),
                                  (ss - 2 * cross + tt).astype(np.float32))
    # one rounding to float after FP64 work short of its last bits: one unit in the last place
    with np.errstate(divide="ignore", invalid="ignore"):
        want = cross / np.sqrt(ss.astype(np.float64) * tt)
    np.testing.assert_allclose(run_op(ocip, "CrossCorr_Norm", src, tpl), want, rtol=2.0 ** -23, atol=0)


# constant images at both ends of each type: the largest sums of every digit
@pytest.mark.parametrize("dtype", [np.uint8, np.int8, np.uint16, np.int16])
@pytest.mark.parametrize("s,t", [("min", "min"), ("min", "max"), ("max", "min"), ("max", "max")])
def test_extreme_constants(ocip, dtype, s, t):
    info = np.iinfo(dtype)
    tshape = (97, 97) if np.dtype(dtype).itemsize == 1 else (128, 113)
    src = np.full((130, 140), getattr(info, s), dtype)
    tpl = np.full(tshape, getattr(info, t), dtype)
    cross, ss = exact_sums(src, tpl)
    say("int8 extremes", np.dtype(dtype).name, s, t)
    np.testing.assert_array_equal(run_op(ocip, "CrossCorr", src, tpl), cross.astype(np.float32))
    tt = int((tpl.astype(np.int64) ** 2).sum())
    np.testing.assert_array_equal(run_op(ocip, "SqrDistance", src, tpl),
                                  (ss - 2 * cross + tt).astype(np.float32))
