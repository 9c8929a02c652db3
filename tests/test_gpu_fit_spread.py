"""Fewer fits than the device has lanes for.

FP64 form: the fits are spread over the wavefronts, fpw = ceil(n / wavefronts)
in each, and evaluated wavefront-wide from the start; the operations are those of
the lane-per-fit order (FSX_FIT_WIDE=0, 64 fits per wavefront), so every result
has the same bits, for one fit, for one and two per wavefront, and where the last
wavefront starts with fewer.  Mixed form: twice the lanes per fit, which changes
only the order of the FP64 sums over q: chi within 1e-9 relative, c1 and c2 within
1e-5 of those of four lanes per fit, as between the device's and the host's order."""
import numpy as np
import pytest

from tests.problem import build_problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F():
    import libfmftsaxs_amd as F
    if F.device_count() < 1:
        pytest.fail("no HIP device visible")
    return F


@pytest.fixture(scope="module")
def problem(F):
    pb = build_problem(300, 200, 6, 0.5, 25, np.arange(18.0, 30.0), 4100, seed=64)
    gp = F.ScoringProblem(pb["L"], pb["qvals"], pb["zvals"], pb["A_re"], pb["A_im"], pb["B_re"],
                          pb["B_im"], pb["a"], pb["params"].mult, pb["peak"],
                          nbeta=pb["nbeta"], nalpha=pb["na"], ngamma=pb["ng"])
    return gp, pb["index"]


@pytest.mark.parametrize("n", [1, 3, 1024, 1025, 2047, 4100])
def test_spread_fits_bit_identical(F, monkeypatch, problem, n):
    gp, index = problem
    print(f"{n} fits", flush=True)
    r = F.score(gp, index[:n])
    monkeypatch.setenv("FSX_FIT_WIDE", "0")
    base = F.score(gp, index[:n])
    for k in ("score", "c1", "c2"):
        assert np.array_equal(r[k], base[k], equal_nan=True), k
    assert r["stats"]["fit_evals"] == base["stats"]["fit_evals"]


@pytest.mark.parametrize("n", [1, 33, 4100])
def test_twice_the_lanes_per_fit(F, monkeypatch, problem, n):
    gp, index = problem
    print(f"{n} fits", flush=True)
    r = F.score(gp, index[:n], mixed=True)
    monkeypatch.setenv("FSX_FIT_GROUP_LANES", "2")
    base = F.score(gp, index[:n], mixed=True)
    ok = ~np.isnan(base["score"])
    assert ok.sum() >= 0.9 * n and np.array_equal(ok, ~np.isnan(r["score"]))
    assert (np.abs(r["score"] - base["score"])[ok] / base["score"][ok]).max() <= 1e-9
    assert np.abs(r["c1"] - base["c1"])[ok].max() <= 1e-5
    assert np.abs(r["c2"] - base["c2"])[ok].max() <= 1e-5
