"""Cross terms of 8- and 16-bit integer images as products of signed bytes, at the edges of the output
tiles (127 rows of 16 columns for 16-bit values, of 32 for 8-bit ones): against exact integer sums."""
import numpy as np
import pytest

from tests.gpu_util import run_op, say
from tests.test_gpu_int8_products import exact_sums, image

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ocip():
    from openclipp_amd import ocip as mod
    ctx = mod.initialize()
    yield mod
    mod.lib.ocipUninitialize(ctx)


@pytest.mark.parametrize("dtype", [np.uint8, np.int8, np.uint16, np.int16])
@pytest.mark.parametrize("height", [126, 127, 128])
@pytest.mark.parametrize("width", [15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65])
def test_tile_edges(ocip, dtype, height, width):
    rng = np.random.default_rng(1000 * height + width)
    src, tpl = image(rng, dtype, (height, width)), image(rng, dtype, (6, 9))
    cross, ss = exact_sums(src, tpl)
    tt = int((tpl.astype(np.int64) ** 2).sum())
    say("int8 tile edges", np.dtype(dtype).name, height, width)
    np.testing.assert_array_equal(run_op(ocip, "CrossCorr", src, tpl), cross.astype(np.float32))
    np.testing.assert_array_equal(run_op(ocip, "SqrDistance", src, tpl),
                                  (ss - 2 * cross + tt).astype(np.float32))
