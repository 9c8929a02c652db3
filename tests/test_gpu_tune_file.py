"""The batch tuner's table file (FSX_TUNE_FILE): a line as it is written now is taken
as it stands; lines of earlier versions (without the last word: their rows meant
single rows of another kernel) and damaged ones are passed over, so that their bucket
is tuned and appended anew.  Results do not depend on the table."""
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


@pytest.mark.parametrize("lines,tuned", [("0 0 1 0 0.1000 pairs\n", False),
                                         ("0 0 1 0 0.1000\n", True),
                                         ("nothing\n0 0 9 0 0.1 pairs\n0 0 2 0\n", True),
                                         ("nothing\n0 0 2 0 0.1 pairs\n", False)])
def test_table_lines(F, tmp_path, monkeypatch, lines, tuned):
    path = tmp_path / "tune.txt"
    path.write_text(lines)
    monkeypatch.setenv("FSX_TUNE_FILE", str(path))
    pb = build_problem(200, 150, 6, 0.3, 9, np.array([22.0, 25.0]), 60, seed=91)
    gp = _gpu_problem(F, pb)
    print(repr(lines), flush=True)
    F.release()   # a fresh table
    try:
        r = F.score_batch([gp], [pb["index"]])[0]
        s = F.score(gp, pb["index"])
    finally:
        F.release()
    for k in ("score", "c1", "c2"):
        assert np.array_equal(r[k], s[k])
    got = path.read_text()
    assert got.startswith(lines)
    added = [l.split() for l in got[len(lines):].splitlines()]
    if tuned:
        assert len(added) == 1 and added[0][:2] == ["0", "0"] and added[0][5:] == ["pairs"]
    else:
        assert added == []
