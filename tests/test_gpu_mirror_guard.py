"""Which mixed calls take the mirrored tables (beta <= pi / 2 only): coefficients of a
real density on even gamma grids, and no others.  FSX_MIRROR=0 keeps every beta.  With
the reference's pi both tables round to nearly the same FP32 values; with a pi 9e-11
off (the mirror image is taken up to 1e-10) the mirrored half is that of a grid 9e-11
beside, which shows in the last bit of about 1 % of the sums of a molecule of 2,000
atoms and stays far below the bar.

Coefficients without A_l-m = (-1)^(l+m) conj(A_lm), receptor's or ligand's, on even
grids against the oracle at the mixed form's bar: mirrored tables would be wrong for
half the betas there (the change made here is 1e-3 of the largest coefficient)."""
import numpy as np
import pytest

import oracle as O
from tests.problem import build_problem
from tests.test_gpu_edges import _check_mixed
from tests.test_gpu_parity import _gpu_problem

pytestmark = pytest.mark.gpu
L, NB, NA = 9, 5, 8


@pytest.fixture(scope="module")
def F():
    import libfmftsaxs_amd as F
    if F.device_count() < 1:
        pytest.fail("no HIP device visible")
    return F


def _problem(ng):
    return build_problem(2000, 1500, L, 0.5, 21, np.array([24.0, 25.5]), 160, seed=340, nbeta=NB,
                         na=NA, ng=ng)


def _with_and_without(F, monkeypatch, pb, pi=None):
    gp = _gpu_problem(F, pb)
    if pi is not None:
        gp.s.pi = pi
    r = F.score(gp, pb["index"], want_cross=True, mixed=True)
    monkeypatch.setenv("FSX_MIRROR", "0")
    g = F.score(gp, pb["index"], want_cross=True, mixed=True)
    monkeypatch.delenv("FSX_MIRROR")
    return r, g


@pytest.mark.parametrize("side", ["A_im", "B_im", "B_re"])
def test_asymmetric_coefficients(F, monkeypatch, side):
    ng = 10
    pb = _problem(ng)
    rng = np.random.default_rng(5)
    pb[side] = pb[side] + 1e-3 * np.abs(pb[side]).max() * rng.normal(size=pb[side].shape)
    ro = O.compute_saxs_scores(pb["index"], pb["A_re"], pb["A_im"], pb["B_re"], pb["B_im"],
                               pb["params"], pb["qvals"], pb["zvals"], L, nbeta=NB, na=NA, ng=ng,
                               want_cross=True)
    print(side, flush=True)
    _check_mixed(F.score(_gpu_problem(F, pb), pb["index"], want_cross=True, mixed=True), ro)
    r, g = _with_and_without(F, monkeypatch, pb, pi=np.pi - 9e-11)
    assert r["stats"]["cross_entries"] == (L + 1) ** 2
    assert np.array_equal(r["cross"], g["cross"])


@pytest.mark.parametrize("ng,mirrored", [(10, True), (11, False)])
def test_symmetric_coefficients(F, monkeypatch, ng, mirrored):
    pb = _problem(ng)
    print(f"ng={ng}", flush=True)
    r, g = _with_and_without(F, monkeypatch, pb, pi=np.pi - 9e-11)
    assert r["stats"]["cross_entries"] == (L + 1) * (L + 2) // 2
    assert np.array_equal(r["cross"], g["cross"]) != mirrored
    scale = np.abs(g["cross"]).max(axis=2, keepdims=True)
    assert (np.abs(r["cross"] - g["cross"]) / scale).max() <= 1e-5


def test_another_pi(F, monkeypatch):
    """A beta grid that does not end at pi has no mirror image."""
    pb = _problem(10)
    gp = _gpu_problem(F, pb)
    gp.s.pi = 3.1
    r = F.score(gp, pb["index"], want_cross=True, mixed=True)
    monkeypatch.setenv("FSX_MIRROR", "0")
    g = F.score(gp, pb["index"], want_cross=True, mixed=True)
    assert np.array_equal(r["cross"], g["cross"])
    d = F.score(gp, pb["index"], want_cross=True)
    scale = np.abs(d["cross"]).max(axis=2, keepdims=True)
    assert (np.abs(r["cross"] - d["cross"]) / scale).max() <= 1e-5
