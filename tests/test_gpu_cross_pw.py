"""One and two poses per wavefront of the cross-term pairing (FSX_CROSS_PW): the two
forms add the same products in the same order, so a pose's profile has the same
bits.  Orders with one to four slots per lane of 32 (L = 6, 7, 8, 10, 11, 12, 13, 15:
25, 32, 41, 61, 72, 85, 98 and 128 slots), with mirrored tables (even gamma grid) and
without; units of odd numbers of poses, so that a wavefront's second half runs past
the last one.  The default against the oracle at the two smallest orders."""
import numpy as np
import pytest

import oracle as O
from tests.problem import build_problem
from tests.test_gpu_edges import _check_fp64, _check_mixed
from tests.test_gpu_parity import _gpu_problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F():
    import libfmftsaxs_amd as F
    if F.device_count() < 1:
        pytest.fail("no HIP device visible")
    return F


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("L", [6, 7, 8, 10, 11, 12, 13, 15])
def test_same_bits_with_one_and_two_poses(F, monkeypatch, L, mixed):
    for ng in (12, 13):
        pb = build_problem(200, 150, L, 0.3, 7, np.array([22.0, 25.0]), 701, seed=300 + L, nbeta=5,
                           na=11, ng=ng)
        gp = _gpu_problem(F, pb)
        print(f"L={L} ng={ng} mixed={mixed}", flush=True)
        got = []
        for pw in ("1", "2"):
            monkeypatch.setenv("FSX_CROSS_PW", pw)
            got.append(F.score(gp, pb["index"], want_cross=True, mixed=mixed)["cross"])
        assert not np.isnan(got[0]).any()
        assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("n", [1, 2, 3, 67])
@pytest.mark.parametrize("L", [6, 7])
def test_short_lists_vs_oracle(F, L, n):
    pb = build_problem(200, 150, L, 0.3, 7, np.array([22.0, 25.0]), n, seed=400 + L, nbeta=4, na=7,
                       ng=8)
    ro = O.compute_saxs_scores(pb["index"], pb["A_re"], pb["A_im"], pb["B_re"], pb["B_im"],
                               pb["params"], pb["qvals"], pb["zvals"], L, nbeta=4, na=7, ng=8,
                               want_cross=True)
    gp = _gpu_problem(F, pb)
    print(f"L={L} n={n}", flush=True)
    _check_fp64(F.score(gp, pb["index"], want_cross=True), ro)
    _check_mixed(F.score(gp, pb["index"], want_cross=True, mixed=True), ro)
