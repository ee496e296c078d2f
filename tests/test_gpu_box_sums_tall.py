"""Window sums of the gradient path for tall narrow templates: one weight far above the others, or a
NaN among them, leaves every other window's sum exact."""
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


def gradient(ocip, s, g, tshape):
    """dS of SqrDistance for an all-zero template: 2 s times the flipped window sum of G."""
    S, G = ocip.Image(s), ocip.Image(g)
    T = ocip.Image(np.zeros(tshape, np.float32))
    dS, dT = ocip.Image(shape=s.shape, dtype=np.float32), ocip.Image(shape=tshape, dtype=np.float32)
    ocip.check(ocip.lib.ocipSqrDistanceBackward(S.handle, T.handle, G.handle, dS.handle, dT.handle),
               "backward")
    return dS.read()


def exact(s, g, tshape):
    th, tw = tshape
    cx, cy = tw // 2, th // 2
    pad = np.pad(g.astype(np.int64), ((th - 1 - cy, cy), (tw - 1 - cx, cx)))
    I = np.pad(pad.cumsum(0).cumsum(1), ((1, 0), (1, 0)))
    box = I[th:, tw:] - I[:-th, tw:] - I[th:, :-tw] + I[:-th, :-tw]
    return (2.0 * s.astype(np.float64) * box).astype(np.float32)


def whole_numbers(rng, shape):
    return (rng.integers(-15, 16, size=shape).astype(np.float32),
            rng.integers(-3, 4, size=shape).astype(np.float32))


# rows whose windows, and those of the rows above in their 32-row tile, begin below the weight
@pytest.mark.parametrize("bright", [2.0 ** 60, np.nan])
@pytest.mark.parametrize("tshape", [(257, 3), (400, 8), (481, 5), (520, 1)])
def test_one_bright_weight(ocip, tshape, bright):
    s, g = whole_numbers(np.random.default_rng(tshape[0]), (700, 90))
    want = exact(s, g, tshape)
    g[1, 2] = bright
    say("tall box sums", tshape, bright)
    top = (tshape[0] - 1 - tshape[0] // 2) + 2 + 32
    np.testing.assert_array_equal(gradient(ocip, s, g, tshape)[top:], want[top:])


# tall and wide: sums from an integral
def test_integral_sums_are_exact(ocip):
    s, g = whole_numbers(np.random.default_rng(270), (300, 130))
    say("integral sums")
    np.testing.assert_array_equal(gradient(ocip, s, g, (270, 62)), exact(s, g, (270, 62)))
