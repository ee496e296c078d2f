"""CrossCorr_Norm of F32 images on split-FP16 MFMA at template sizes whose FP32 kernel forms the
window sums of squares within its tiles: a pixel far above the others, a NaN or infinity and zero
margins reach no further than they do there.

Bound: as in test_gpu_split_wide_range.py, and 2^-22 of the value for a sum of squares that is a
difference of prefixes at most 2^27 times itself (2^-53 each, a few of them)."""
import numpy as np
import pytest

from tests.gpu_util import run_op, say
from tests.test_gpu_split_wide_range import bound

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ocip():
    from openclipp_amd import ocip as mod
    ctx = mod.initialize()
    yield mod
    mod.lib.ocipUninitialize(ctx)


# windows at least 96 columns or rows from the pixel: outside its tile of 32 x 64 outputs
@pytest.mark.parametrize("tshape", [(24, 24), (3, 31), (30, 7)])
@pytest.mark.parametrize("bright", [1e4, 1e6, 1e8, 1e9, 1e12])
def test_bright_pixel(ocip, monkeypatch, tshape, bright):
    rng = np.random.default_rng(int(bright) % 1000 + tshape[1])
    src = rng.random((300, 280), dtype=np.float32) + np.float32(0.1)
    src[5, 6] = bright
    tpl = rng.random(tshape, dtype=np.float32)
    say("split bright", tshape, bright)
    monkeypatch.setenv("OCIP_SPLIT_NCC", "1")
    got = run_op(ocip, "CrossCorr_Norm", src, tpl)
    want, tol = bound(src, tpl)
    far = np.ones(src.shape, bool)
    far[:101, :102] = False
    e = np.abs(got - want)[far] / (tol + 2.0 ** -22 * np.abs(want))[far]
    assert np.all(e <= 1), float(np.max(e))


# zero windows (7 x 7 outputs) between the samples of split_prep, and the whole of one 127 x 64 tile
@pytest.mark.parametrize("rows,cols", [((117, 147), (101, 131)), ((100, 300), (40, 160))])
def test_hole(ocip, monkeypatch, rows, cols):
    rng = np.random.default_rng(9)
    src = rng.random((330, 260), dtype=np.float32)
    src[slice(*rows), slice(*cols)] = 0
    tpl = rng.random((24, 24), dtype=np.float32)
    say("split hole", rows, cols)
    maps = []
    for on in ("0", "1"):
        monkeypatch.setenv("OCIP_SPLIT_NCC", on)
        maps.append(run_op(ocip, "CrossCorr_Norm", src, tpl))
    assert np.isnan(maps[0]).sum() == (rows[1] - rows[0] - 23) * (cols[1] - cols[0] - 23)
    np.testing.assert_array_equal(np.isnan(maps[1]), np.isnan(maps[0]))
    np.testing.assert_allclose(maps[1], maps[0], rtol=0, atol=2 * (20 + tpl.size) * 2.0 ** -23)


# the default rule takes the split at 1920x1080 / 24x24
@pytest.mark.parametrize("what", [np.nan, np.inf, -np.inf, "margins"])
@pytest.mark.parametrize("shape,forced", [((200, 190), True), ((1080, 1920), False)])
def test_reach(ocip, monkeypatch, what, shape, forced):
    rng = np.random.default_rng(7)
    src = rng.random(shape, dtype=np.float32)
    if what == "margins":
        src[:, :shape[1] // 3] = 0
        src[2 * shape[0] // 3:] = 0
    else:
        src[60, 70] = what
    tpl = rng.random((24, 24), dtype=np.float32)
    say("split reach", what, shape)
    monkeypatch.setenv("OCIP_SPLIT_NCC", "0")
    plain = run_op(ocip, "CrossCorr_Norm", src, tpl)
    if forced:
        monkeypatch.setenv("OCIP_SPLIT_NCC", "1")
    else:
        monkeypatch.delenv("OCIP_SPLIT_NCC")
    got = run_op(ocip, "CrossCorr_Norm", src, tpl)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(plain))
    np.testing.assert_allclose(got, plain, rtol=0, atol=2 * (20 + tpl.size) * 2.0 ** -23)
