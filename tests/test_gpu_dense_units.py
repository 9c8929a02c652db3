"""Units of more than 64 poses: lists long enough for the cap of 256 (n Q at least 256
times the blocks of four full launches), crowded on a few gamma2 rows, so that a
unit's poses run in up to four batches, the last one partial.  A pose's sums do
not depend on its unit: both forms give a pose of the long list the bits of the
FP64 cross terms, respectively of the FP32 ones, that it has in a short list, whose
units hold at most 64 poses."""
import numpy as np
import pytest

from tests.problem import build_problem
from tests.test_gpu_parity import _gpu_problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F():
    import libfmftsaxs_amd as F
    if F.device_count() < 1:
        pytest.fail("no HIP device visible")
    return F


@pytest.mark.parametrize("mixed", [False, True])
def test_long_list_equals_short_lists(F, mixed):
    nb, na, ng, n, Q = 4, 12, 14, 40000, 40
    pb = build_problem(200, 150, 5, 0.3, Q, np.array([22.0, 25.0]), 20, seed=77, nbeta=nb, na=na,
                       ng=ng)
    rng = np.random.default_rng(78)
    idx = rng.choice(2 * nb * nb * na * ng * ng, size=n, replace=False).astype(np.int64)
    gp = _gpu_problem(F, pb)
    print(f"{n} poses, mixed={mixed}", flush=True)
    r = F.score(gp, idx, want_cross=True, mixed=mixed)
    assert not np.isnan(r["score"]).any()
    for k0 in (0, 17000, n - 700):
        s = F.score(gp, idx[k0:k0 + 700], want_cross=True, mixed=mixed)
        assert np.array_equal(r["cross"][k0:k0 + 700], s["cross"])
