"""The cross-term stage's units, tiles and mirrored tables against the oracle.

Sizes at which the packing changes: translation tiles of 16 l (L = 15, 16, 17)
and blocks of 4 l1, expansions of more than one m-chunk with rows split
between two summation orders (L = 23: 300 entries, 256 + 44 in FP64), more
than 8 gamma2 rows of one (z, beta2) and more than 64 poses on one row (a
unit's limits), a unit of one pose, and the tables of beta <= pi / 2 only, which
even gamma grids of conjugate-symmetric coefficients take, with odd and even
numbers of betas, alpha = 0, odd alpha grids, and the general tables of odd
gamma grids and of coefficients without that symmetry.

Bars as in the parity and mixed-form tests: the arithmetic is FP64 with sums of
at most a few thousand terms (1e-10 in I(q)), respectively FP32 tables and sums
(1e-5)."""
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


def _poses(rng, zn, nb, na, ng):
    """Distinct poses: 130 on one gamma2 row, one on every gamma2 of another
    (z, beta2), one alone, every (beta1, beta2) pair at alpha = 0, and some
    drawn at random."""
    def index(z, b1, b2, a2, g1, g2):
        return ((((z * nb + b1) * nb + b2) * na + a2) * ng + g1) * ng + g2
    got = [index(0, *rng.integers(0, (nb, 1), 2) + (0, nb - 1), rng.integers(na), rng.integers(ng), 1)
           for _ in range(400)]
    got = list(dict.fromkeys(int(i) for i in got))[:130]
    assert len(got) > 64
    got += [index(zn - 1, rng.integers(nb), nb // 2, rng.integers(na), rng.integers(ng), g2)
            for g2 in range(ng)]
    got += [index(zn - 1, nb - 1, 0, na - 1, ng - 1, ng - 1)]
    got += [index(0, b1, b2, 0, rng.integers(ng), rng.integers(ng))
            for b1 in range(nb) for b2 in range(nb - 1)]
    got += list(rng.integers(0, zn * nb * nb * na * ng * ng, 40))
    got = np.array(list(dict.fromkeys(int(i) for i in got)), dtype=np.int64)
    return rng.permutation(got)


def _both_forms(F, pb):
    ro = O.compute_saxs_scores(pb["index"], pb["A_re"], pb["A_im"], pb["B_re"], pb["B_im"],
                               pb["params"], pb["qvals"], pb["zvals"], pb["L"], nbeta=pb["nbeta"],
                               na=pb["na"], ng=pb["ng"], want_cross=True)
    gp = _gpu_problem(F, pb)
    print("FP64 form", flush=True)
    _check_fp64(F.score(gp, pb["index"], want_cross=True), ro)
    print("mixed form", flush=True)
    _check_mixed(F.score(gp, pb["index"], want_cross=True, mixed=True), ro)


@pytest.mark.parametrize("L,nb,na,ng", [(7, 7, 12, 12), (7, 6, 12, 12), (8, 5, 9, 10),
                                        (7, 6, 12, 13), (6, 7, 1, 2)])
def test_units_and_mirrored_tables(F, L, nb, na, ng):
    pb = build_problem(200, 150, L, 0.3, 7, np.array([22.0, 25.0]), 20, seed=300 + L + nb,
                       nbeta=nb, na=na, ng=ng)
    rng = np.random.default_rng(41 * nb + ng)
    if na * ng < 8:
        pb["index"] = np.arange(2 * nb * nb * na * ng * ng, dtype=np.int64)
    else:
        pb["index"] = _poses(rng, 2, nb, na, ng)
    _both_forms(F, pb)


@pytest.mark.parametrize("L", [15, 16, 17, 23])
def test_tile_edges(F, L):
    pb = build_problem(200, 150, L, 0.3, 5, np.array([24.0, 25.5]), 60, seed=320 + L,
                       nbeta=4, na=6, ng=10)
    _both_forms(F, pb)


def test_coefficients_without_symmetry(F):
    """A receptor that is not the expansion of a real density: all m entries,
    general tables also on an even grid."""
    L = 9
    pb = build_problem(200, 150, L, 0.3, 7, np.array([24.0, 25.5]), 80, seed=340,
                       nbeta=5, na=8, ng=10)
    rng = np.random.default_rng(5)
    pb["A_im"] = pb["A_im"] + 1e-3 * np.abs(pb["A_im"]).max() * rng.normal(size=pb["A_im"].shape)
    ro = O.compute_saxs_scores(pb["index"], pb["A_re"], pb["A_im"], pb["B_re"], pb["B_im"],
                               pb["params"], pb["qvals"], pb["zvals"], L, nbeta=5, na=8, ng=10,
                               want_cross=True)
    r = F.score(_gpu_problem(F, pb), pb["index"], want_cross=True)
    assert r["stats"]["cross_entries"] == (L + 1) ** 2
    cg, co = r["cross"], ro["cross"]
    assert (np.abs(cg - co) / np.abs(co).max(axis=2, keepdims=True)).max() <= 1e-10
