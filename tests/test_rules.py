"""The size rules of csrc/fsx_rules.h, compiled for the host with gcc."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "fsx_rules.h"
int cross_pw(int mixed, int ns) { return fsx_cross_pw(mixed, ns); }
int cross_blocks(int mixed, int rows3, int ns, int pw, long nrows, double per_bucket)
{
    return fsx_cross_blocks(mixed, rows3, ns, pw, nrows, per_bucket);
}
int fit_lanes(int Q) { return fsx_fit_lanes(Q); }
int unit_scan(long groups) { return fsx_unit_scan(groups); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, so = d / "rules.c", d / "librules.so"
    src.write_text(SRC)
    subprocess.run(["gcc", "-std=c11", "-O2", "-Wall", "-Werror", "-shared", "-fPIC",
                    "-I" + os.path.join(ROOT, "libfmftsaxs_amd", "csrc"), str(src), "-o",
                    str(so)], check=True)
    return C.CDLL(str(so))


def test_two_poses_per_wavefront_at_small_orders(rules):
    """Slots of one chunk at order L: (L + 1)(L + 2) / 2 less the packed m = 0
    pairs.  Orders 6 to 12 leave lanes of a one-pose wavefront without a slot or
    its last slots half empty."""
    for L in range(6, 13):
        ns = (L + 1) * (L + 2) // 2 - (L + 1) // 2
        assert rules.cross_pw(1, ns) == 2 and rules.cross_pw(0, ns) == 2, L
    assert rules.cross_pw(1, 128) == 1 and rules.cross_pw(0, 128) == 2
    assert rules.cross_pw(1, 176) == 1 and rules.cross_pw(0, 176) == 1


def test_group_sums_of_their_own_for_many_groups(rules):
    """Summed by every wavefront they cost the square of the number of groups."""
    rules.unit_scan.argtypes = [C.c_long]
    assert not rules.unit_scan(1) and not rules.unit_scan(684)
    assert rules.unit_scan(3737) and rules.unit_scan(2 ** 30)


def test_lanes_per_fit(rules):
    got = [rules.fit_lanes(Q) for Q in (2, 32, 33, 51, 64, 65, 81, 128, 129, 512, 513, 1024, 4000)]
    assert got == [4, 4, 8, 8, 8, 16, 16, 16, 32, 64, 64, 64, 64]


def test_blocks_of_crowded_fp64_lists(rules):
    f = rules.cross_blocks
    f.argtypes = [C.c_int] * 4 + [C.c_long, C.c_double]
    # 64 x 19 rows at L = 15: 1,000,000 and 210,000 poses on 43,776 buckets
    assert f(0, 8, 128, 2, 1216, 22.8) == 2 and f(0, 8, 128, 2, 1216, 4.8) == 5
    # 128 x 37 rows at L = 25: 2,500,000 and 200,000 poses on 478,336 buckets
    assert f(0, 6, 171, 1, 4736, 5.23) == 2 and f(0, 6, 171, 1, 4736, 0.42) == 5
    # few rows per unit with three blocks
    assert f(0, 4, 181, 1, 703, 0.4) == 2 and f(0, 4, 221, 1, 861, 0.4) == 5
    assert f(0, 4, 181, 1, 468, 0.009) == 5   # 95 poses: too few units for two blocks
    assert f(0, 4, 221, 1, 861, 35.0) == 2
    # small tables, FP32 tables
    assert f(0, 8, 61, 2, 231, 88.0) == 5 and f(1, 8, 128, 1, 1216, 22.8) == 5
