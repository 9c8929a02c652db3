"""More complexes than the batch has streams, of different sizes, so that each stream's
shared buffers serve several of them in turn, some larger than the one before: every
complex's results are bit for bit those of its own call, eager and replayed, in both
forms."""
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
def test_more_complexes_than_streams(F, mixed):
    pbs = [build_problem(200, 150, L, 0.3, Q, np.arange(22.0, 22.0 + zn), n, seed=700 + L + Q)
           for L, Q, zn, n in ((6, 9, 3, 40), (10, 21, 4, 300), (4, 7, 2, 15), (12, 15, 5, 500),
                               (6, 30, 2, 900), (9, 11, 3, 1), (11, 12, 6, 700))]
    gps = [_gpu_problem(F, pb) for pb in pbs]
    poses = [pb["index"] for pb in pbs]
    singles = [F.score(g, p, want_cross=True, mixed=mixed) for g, p in zip(gps, poses)]
    for rep in range(3):
        print(f"mixed={mixed}, call {rep}", flush=True)
        got = F.score_batch(gps, poses, want_cross=True, mixed=mixed)
        for r, s in zip(got, singles):
            for k in ("score", "c1", "c2", "cross"):
                assert np.array_equal(r[k], s[k], equal_nan=True), (rep, k)
        # other work between the replays
        F.score(gps[rep], poses[rep], mixed=not mixed)
