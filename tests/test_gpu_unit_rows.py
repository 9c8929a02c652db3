"""Cross-term units of one (z, beta2) whose gamma2 rows don't divide by a unit's eight:
the rows are cut in even shares (9 as 5 and 4, 25 as 7, 6, 6, 6; 65 and 130 rows span
the 64 buckets a wavefront looks at together), rows of one pose and of more poses
than a unit holds among them, against the oracle at the parity and mixed-form bars."""
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


@pytest.mark.parametrize("ng", [1, 8, 9, 17, 25, 65, 130])
def test_rows_vs_oracle(F, ng):
    L, nb, na, zn = 5, 3, 8, 2
    pb = build_problem(200, 150, L, 0.3, 6, np.array([24.0, 25.5]), 20, seed=600 + ng, nbeta=nb,
                       na=na, ng=ng)
    rng = np.random.default_rng(ng)

    def index(z, b1, b2, a2, g1, g2):
        return ((((z * nb + b1) * nb + b2) * na + a2) * ng + g1) * ng + g2
    got = [index(0, rng.integers(nb), 1, rng.integers(na), rng.integers(ng), g2) for g2 in range(ng)]
    got += [index(1, rng.integers(nb), 2, rng.integers(na), rng.integers(ng), g2)
            for g2 in range(0, ng, 3) for _ in range(4)]
    got += [index(1, rng.integers(nb), 0, rng.integers(na), rng.integers(ng), ng // 2) for _ in range(90)]
    pb["index"] = rng.permutation(np.array(list(dict.fromkeys(int(i) for i in got)), dtype=np.int64))
    ro = O.compute_saxs_scores(pb["index"], pb["A_re"], pb["A_im"], pb["B_re"], pb["B_im"],
                               pb["params"], pb["qvals"], pb["zvals"], L, nbeta=nb, na=na, ng=ng,
                               want_cross=True)
    gp = _gpu_problem(F, pb)
    print(f"ng={ng}, {len(pb['index'])} poses", flush=True)
    _check_fp64(F.score(gp, pb["index"], want_cross=True), ro)
    _check_mixed(F.score(gp, pb["index"], want_cross=True, mixed=True), ro)
