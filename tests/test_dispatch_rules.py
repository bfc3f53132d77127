"""Which variant of a kernel a size takes (csrc/lf_rules.h, compiled for the host): both sides of every line.  The times behind
the lines stand at the rules."""
import ctypes

import pytest

from helpers import host_library

SOURCE = """
#include "lf_rules.h"
extern "C" int csr_rows(long long rows, long long entries, long long longest, int panels) { return lf::csr_rows_of_group(rows, entries, longest, panels); }
extern "C" int bsr_features(int feat, int block, long long rows, long long blocks) { return lf::bsr_lane_features(feat, block, rows, blocks); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    return host_library(tmp_path_factory.mktemp("rules"), SOURCE)


@pytest.mark.parametrize("rows,average,longest,group", [
    (2461, 367, 2301, 2), (4972, 271, 4533, 2), (2975, 162, 751, 2), (5120, 96, 240, 2),
    (6149, 286, 4223, 2), (12_288, 208, 520, 2), (12_289, 208, 520, 4), (24_575, 400, 5000, 4),
    (4137, 377, 703, 2), (6144, 300, 300, 2), (6144, 299, 400, 8), (6145, 300, 400, 8),         # rows of about one length
    (10_026, 276, 502, 8), (2840, 214, 287, 8), (5120, 96, 239, 8), (12_289, 208, 519, 8),
    (9140, 107, 1051, 8), (5121, 207, 5000, 8),                                # more rows
    (2000, 60, 800, 8), (5120, 95, 288, 8), (3000, 200, 0, 8),                 # short rows; the longest one is not known
    (24_576, 400, 5000, 16), (2_000_000, 2, 100, 16)])
def test_rows_of_a_csr_workgroup(rules, rows, average, longest, group):
    size = ctypes.c_longlong
    assert rules.csr_rows(size(rows), size(rows * average), size(longest), 1) == group
    assert rules.csr_rows(size(rows), size(0), size(longest), 1) in (8, 16)    # (how many entries there are is not known)


def test_rows_of_a_csr_workgroup_in_panels(rules):
    size = ctypes.c_longlong
    assert [rules.csr_rows(size(5000), size(5000 * 200), size(2000), panels) for panels in (1, 2, 3)] == [2, 2, 8]


@pytest.mark.parametrize("feat,block,rows,blocks,features", [
    (8, 16, 50_000, 500_000, 2), (32, 64, 12_500, 120_000, 2), (40, 16, 50_000, 500_000, 4), (48, 64, 12_500, 120_000, 4), (72, 16, 100, 300, 8), (128, 64, 100, 1000, 8),
    (56, 64, 1397, 9_761, 4), (56, 64, 2048, 12_288, 4), (56, 64, 2048, 12_289, 8), (64, 64, 2049, 4_100, 8), (56, 64, 1936, 17_390, 8),
    (56, 32, 21_398, 192_515, 4), (64, 32, 6553, 65_536, 4), (64, 32, 6553, 65_537, 8), (64, 32, 18_331, 91_639, 8),
    (64, 16, 10_176, 61_041, 4), (56, 16, 16_384, 65_536, 4), (56, 16, 16_385, 40_000, 8), (56, 16, 16_384, 65_537, 8), (64, 16, 14_770, 132_930, 8),
    (56, 16, 1000, 0, 8), (56, 32, 1000, 0, 4), (64, 64, 100, 0, 8)])                       # 0: their number is not known
def test_features_of_a_bsr_lane(rules, feat, block, rows, blocks, features):
    assert rules.bsr_features(feat, block, ctypes.c_longlong(rows), ctypes.c_longlong(blocks)) == features
