"""F32 tiles that read the template in place: pitched templates, images and columns at every
alignment of the 16-byte staging loads and stores, tiles at the right edge, and templates on both
sides of the 1024 taps up to which the workgroups sum t^2 themselves.  Raw ops bit for bit
against the reference order, Norm ops within 1e-5 of it (1e-6 floor)."""
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


@pytest.mark.parametrize("tshape", [(1, 1), (3, 2), (5, 7), (32, 32), (33, 32), (4, 40)])
@pytest.mark.parametrize("shape,pitch", [((70, 64), 64), ((66, 97), 101), ((64, 131), 133),
                                         ((129, 46), 46)])
def test_in_place_templates(ocip, shape, pitch, tshape):
    rng = np.random.default_rng(pitch * 100 + tshape[1])
    src = rng.random((shape[0], pitch), dtype=np.float32)[:, :shape[1]]
    tpl = rng.random((tshape[0], tshape[1] + 3), dtype=np.float32)[:, :tshape[1]]
    for op in ["SqrDistance", "AbsDistance", "CrossCorr", "SqrDistance_Norm", "CrossCorr_Norm"]:
        say("in place", shape, pitch, tshape, op)
        got = run_op(ocip, op, src, tpl)
        want = orc.prox_ref(OP_CODE[op], src, tpl)
        if op.endswith("_Norm"):
            assert np.all(np.abs(got - want) <= 1e-5 * np.abs(want) + 1e-6), op
        else:
            np.testing.assert_array_equal(got, want, err_msg=op)


def test_map_over_its_own_template(ocip):
    """Dest may be the template's image (of the source's size): the template is read first."""
    rng = np.random.default_rng(3)
    src = rng.random((70, 90), dtype=np.float32)
    tpl = rng.random((70, 90), dtype=np.float32)
    want = orc.prox_ref(OP_CODE["SqrDistance"], src, tpl)
    S, T = ocip.Image(src), ocip.Image(tpl.copy())
    ocip.check(ocip.proximity("SqrDistance", S, T, T), "SqrDistance")
    np.testing.assert_array_equal(T.read(), want)
