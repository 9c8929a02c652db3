"""The bucketing of poses over many (z, beta2) groups: on both sides of the count from
which the groups' sums have a launch of their own (700), of that launch's steps of
4,096 groups, and at 180,000 groups, where the stage has to stay far below the
milliseconds that summing all earlier groups in every wavefront takes (14 ms; 0.2
with the launch)."""
import numpy as np
import pytest

import oracle as O
from tests.problem import build_problem
from tests.test_gpu_edges import _check_fp64
from tests.test_gpu_parity import _gpu_problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F():
    import libfmftsaxs_amd as F
    if F.device_count() < 1:
        pytest.fail("no HIP device visible")
    return F


@pytest.mark.parametrize("nb,zn,ng", [(7, 100, 6), (27, 26, 5), (64, 64, 3), (17, 241, 4), (91, 91, 2)])
def test_groups_vs_oracle(F, nb, zn, ng):
    L, n = 3, 400
    pb = build_problem(200, 150, L, 0.3, 5, np.linspace(20.0, 30.0, zn), n, seed=500 + nb, nbeta=nb,
                       na=6, ng=ng)
    rng = np.random.default_rng(nb)
    # first and last groups, one crowded group, the rest spread
    total = zn * nb * nb * 6 * ng * ng
    pb["index"] = np.unique(np.concatenate([rng.integers(0, total, n - 102), np.arange(100), [total - 1]])
                            ).astype(np.int64)
    ro = O.compute_saxs_scores(pb["index"], pb["A_re"], pb["A_im"], pb["B_re"], pb["B_im"],
                               pb["params"], pb["qvals"], pb["zvals"], L, nbeta=nb, na=6, ng=ng,
                               want_cross=True)
    print(f"{nb * zn} groups", flush=True)
    _check_fp64(F.score(_gpu_problem(F, pb), pb["index"], want_cross=True), ro)


def test_stage_time_of_180000_groups(F):
    nb, zn, ng, L = 200, 900, 4, 3
    pb = build_problem(200, 150, L, 0.3, 5, np.linspace(20.0, 40.0, zn), 500, seed=77, nbeta=nb,
                       na=12, ng=ng)
    gp = _gpu_problem(F, pb)
    idx = np.random.default_rng(3).integers(0, zn * nb * nb * 12 * ng * ng, 500).astype(np.int64)
    print(f"{nb * zn} groups", flush=True)
    ms = [F.score(gp, idx)["stats"]["ms_group"] for _ in range(4)]
    assert min(ms) < 3.0
