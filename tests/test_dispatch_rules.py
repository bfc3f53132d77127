"""Which variant of a kernel a size takes (csrc/lf_rules.h, compiled for the host): both sides of every line.  The times behind
the lines stand at the rules."""
import ctypes

import pytest

from helpers import host_library

SOURCE = """
#include "lf_rules.h"
extern "C" int csr_rows(long long rows, long long entries, long long longest, int panels) { return lf::csr_rows_of_group(rows, entries, longest, panels); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    return host_library(tmp_path_factory.mktemp("rules"), SOURCE)


@pytest.mark.parametrize("rows,average,longest,group", [
    (2461, 367, 2301, 2), (4972, 271, 4533, 2), (2975, 162, 751, 2), (5120, 96, 288, 2),
    (10_026, 276, 502, 8), (2840, 214, 287, 8), (5120, 96, 287, 8),            # rows of about one length
    (5817, 266, 4201, 8), (9140, 107, 1051, 8), (5121, 96, 288, 8),            # more rows
    (2000, 60, 800, 8), (5120, 95, 288, 8), (3000, 200, 0, 8),                 # short rows; the longest one is not known
    (24_575, 400, 5000, 8), (24_576, 400, 5000, 16), (2_000_000, 2, 100, 16)])
def test_rows_of_a_csr_workgroup(rules, rows, average, longest, group):
    size = ctypes.c_longlong
    assert rules.csr_rows(size(rows), size(rows * average), size(longest), 1) == group
    assert rules.csr_rows(size(rows), size(0), size(longest), 1) in (8, 16)    # (how many entries there are is not known)


def test_rows_of_a_csr_workgroup_in_panels(rules):
    size = ctypes.c_longlong
    assert [rules.csr_rows(size(5000), size(5000 * 200), size(2000), panels) for panels in (1, 2, 3)] == [2, 2, 8]
