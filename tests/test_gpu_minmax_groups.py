"""ocipMinIndx / ocipMaxIndx on both sides of the 1024 work-groups whose results the host combines
(256 x 16 pixels each): values, ties between groups and NaN as the reference-order oracle."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.test_gpu_integral import _min_max

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ocip():
    from openclipp_amd import ocip as mod
    ctx = mod.initialize()
    yield mod
    mod.lib.ocipUninitialize(ctx)


@pytest.mark.parametrize("rows", [16 * 1024, 16 * 1024 + 1])
def test_groups_on_the_host_and_on_the_device(ocip, rows):
    rng = np.random.default_rng(rows)
    ties = rng.integers(0, 3, (rows, 40)).astype(np.float32)
    holes = rng.random((rows, 40), dtype=np.float32)
    holes[5000] = np.nan
    for src in (ties, holes):
        for want_max in (True, False):
            assert _min_max(ocip, src, want_max) == orc.min_max_indx(src, want_max)
    holes[0, 0] = np.nan
    for want_max in (True, False):
        v, x, y = _min_max(ocip, holes, want_max)
        assert np.isnan(v) and (x, y) == (0, 0)
