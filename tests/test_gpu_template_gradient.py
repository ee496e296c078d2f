"""The template gradient of SqrDistance with small whole numbers, whose products and sums are all exact:
    dT(u, v) = -2 sum G(x, y) P(x + u - cx, y + v - cy) + 2 t(u, v) sum G."""
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


# images around the 32 x 128 tasks and their chunks of 16 columns (whole tasks, whole and partial ones side
# by side, one column over), templates from one tap to 32 x 32
@pytest.mark.parametrize("shape,tshape", [((1, 1), (1, 1)), ((32, 128), (32, 32)), ((33, 129), (5, 31)),
                                          ((31, 112), (31, 5)), ((40, 113), (32, 1)), ((65, 241), (9, 17)),
                                          ((70, 300), (31, 31)), ((34, 272), (1, 32))])
def test_template_gradient_is_exact(ocip, shape, tshape):
    (H, W), (th, tw) = shape, tshape
    rng = np.random.default_rng(W + tw)
    s = rng.integers(-7, 8, size=shape)
    g = rng.integers(-3, 4, size=shape)
    t = rng.integers(1, 8, size=tshape)
    say("template gradient", shape, tshape)
    S, G, T = (ocip.Image(a.astype(np.float32)) for a in (s, g, t))
    dS, dT = ocip.Image(shape=shape, dtype=np.float32), ocip.Image(shape=tshape, dtype=np.float32)
    ocip.check(ocip.lib.ocipSqrDistanceBackward(S.handle, T.handle, G.handle, dS.handle, dT.handle),
               "backward")
    cx, cy = tw // 2, th // 2
    P = np.pad(s, ((cy, th), (cx, tw)))
    want = np.array([[-2 * (g * P[v:v + H, u:u + W]).sum() + 2 * t[v, u] * g.sum() for u in range(tw)]
                     for v in range(th)])
    np.testing.assert_array_equal(dT.read(), want.astype(np.float32))
