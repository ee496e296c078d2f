"""One-column templates of hundreds of rows: the band that fills the tile kernels' LDS to the last row
(392 rows and more of tiles 36 floats wide)."""
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


# sums of positive terms: n steps of 2^-23 each at most, and the result's rounding
@pytest.mark.parametrize("th", [391, 392, 393, 470])
@pytest.mark.parametrize("dtype", [np.float32, np.uint32, np.int32])
@pytest.mark.parametrize("op", ["SqrDistance_Norm", "CrossCorr_Norm"])
def test_one_column(ocip, op, dtype, th):
    rng = np.random.default_rng(th)
    draw = rng.random if dtype == np.float32 else lambda n: rng.integers(1, 1000, n)
    src, tpl = draw((480, 40)).astype(dtype), draw((th, 1)).astype(dtype)
    say("one column", op, np.dtype(dtype).name, th)
    got, want = run_op(ocip, op, src, tpl), orc.prox_f64(OP_CODE[op], src, tpl)
    assert np.all(np.abs(got - want) <= (th + 4) * 2.0 ** -23 * np.abs(want))
