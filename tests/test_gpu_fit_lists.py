"""A pose's result does not depend on the length of its list: score, c1 and c2 of a
long list (more fits than the device runs at once) are bit for bit those of its
poses scored in lists of 1, 700 and 5,000, in both forms, with 2, 25, 41 and 70 q (four,
eight and sixteen lanes per fit in the mixed form; more lanes than q among them)."""
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
@pytest.mark.parametrize("Q,n", [(2, 3000), (25, 70000), (41, 40000), (70, 20000)])
def test_long_list_equals_short_lists(F, Q, n, mixed):
    nb, na, ng = 5, 12, 14
    pb = build_problem(200, 150, 5, 0.4, Q, np.array([22.0, 25.0, 28.0]), 20, seed=177, nbeta=nb,
                       na=na, ng=ng)
    rng = np.random.default_rng(178)
    idx = rng.choice(3 * nb * nb * na * ng * ng, size=n, replace=False).astype(np.int64)
    gp = _gpu_problem(F, pb)
    print(f"{n} poses, Q={Q}, mixed={mixed}", flush=True)
    r = F.score(gp, idx, mixed=mixed)
    # two q are fitted exactly: chi^2 is rounding, its root NaN where that is negative
    # (so in the oracle too)
    assert Q == 2 or not np.isnan(r["score"]).any()
    for k0, m in ((0, 1), (n // 2, 700), (n - 5000 if n > 5000 else 0, 5000)):
        s = F.score(gp, idx[k0:k0 + m], mixed=mixed)
        for k in ("score", "c1", "c2"):
            assert np.array_equal(r[k][k0:k0 + m], s[k], equal_nan=True), (k, k0, m)


def test_both_orders_of_the_records(F):
    """One pose more than start at once: the records are then sorted by (z, beta2)
    instead of (beta2, z).  A list on either side, poses of all z and beta2."""
    nb, na, ng, Q = 4, 9, 8, 12
    pb = build_problem(200, 150, 4, 0.4, Q, np.linspace(21.0, 33.0, 70), 20, seed=179, nbeta=nb,
                       na=na, ng=ng)
    rng = np.random.default_rng(180)
    gp = _gpu_problem(F, pb)
    total = 70 * nb * nb * na * ng * ng
    idx = rng.choice(total, size=min(total, 120000), replace=False).astype(np.int64)
    print(f"{idx.size} poses", flush=True)
    for mixed in (False, True):
        r = F.score(gp, idx, mixed=mixed)
        s = F.score(gp, idx[:30000], want_cross=True, mixed=mixed)
        assert not np.isnan(s["cross"]).any()
        for k in ("score", "c1", "c2"):
            assert np.array_equal(r[k][:30000], s[k], equal_nan=True), k
