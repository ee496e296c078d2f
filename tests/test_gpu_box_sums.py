"""Window sums of the gradient path, exactly: with an all-zero template the gradient of SqrDistance in
the source is 2 s times the flipped window sum of G, and whole numbers make every sum exact, so
the result is that product rounded once."""
import numpy as np
import pytest

from tests.gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ocip():
    from openclipp_amd import ocip as mod
    ctx = mod.initialize()
    yield mod
    mod.lib.ocipUninitialize(ctx)


# heights around the 8 rows that one wavefront's columns run down (1 row, 8, 9, 10, 16, 17, 18), widths
# around the 64 lanes, images around the 32 x 64 tiles, and both sides of the 256 rows from which
# the sums come from an integral
@pytest.mark.parametrize("shape,tshape", [((1, 1), (1, 1)), ((33, 65), (8, 1)), ((31, 64), (9, 2)),
                                          ((64, 130), (10, 65)), ((70, 67), (16, 66)),
                                          ((65, 200), (17, 130)), ((40, 63), (18, 31)),
                                          ((270, 70), (256, 3)), ((270, 70), (257, 3))])
def test_window_sums_are_exact(ocip, shape, tshape):
    (H, W), (th, tw) = shape, tshape
    rng = np.random.default_rng(th * 10 + tw)
    s = rng.integers(-15, 16, size=shape).astype(np.float32)
    g = rng.integers(-3, 4, size=shape).astype(np.float32)
    say("box sums", shape, tshape)
    S, G = ocip.Image(s), ocip.Image(g)
    T = ocip.Image(np.zeros(tshape, np.float32))
    dS, dT = ocip.Image(shape=shape, dtype=np.float32), ocip.Image(shape=tshape, dtype=np.float32)
    ocip.check(ocip.lib.ocipSqrDistanceBackward(S.handle, T.handle, G.handle, dS.handle, dT.handle),
               "backward")
    cx, cy = tw // 2, th // 2
    pad = np.pad(g.astype(np.int64), ((th - 1 - cy, cy), (tw - 1 - cx, cx)))
    I = np.pad(pad.cumsum(0).cumsum(1), ((1, 0), (1, 0)))
    box = I[th:, tw:] - I[:-th, tw:] - I[th:, :-tw] + I[:-th, :-tw]
    np.testing.assert_array_equal(dS.read(), (2.0 * s.astype(np.float64) * box).astype(np.float32))
