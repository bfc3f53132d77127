"""The index arithmetic of the kernels (csrc/lf_index.h), compiled for the host, at the largest arrays that are accepted:
no GPU, and no array of that size, is needed to see a 32-bit sum pass 2^31."""
import pytest

from helpers import host_library

MOST = 2**31 - 1                       # entries of a matrix

SOURCE = """
#include "lf_index.h"
extern "C" int group_source(int start, int q, int n) { return lf::group_source(start, q, n); }
extern "C" int chunks_of(int len, int chunk) { return lf::chunks_of(len, chunk); }
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    return host_library(tmp_path_factory.mktemp("index"), SOURCE)


@pytest.mark.parametrize("start,fill,width,entries", [(MOST - 16, 16, 32, MOST), (2**31 - 20, 17, 32, MOST), (MOST - 1, 1, 1024, MOST), (MOST - 3, 3, 4, MOST),
                                                      (MOST - 1025, 1025, 1024, MOST), (0, MOST, 1024, MOST), (0, 5, 8, 9), (0, 4, 8, 4), (7, 2, 8, 9)])
def test_groups_of_the_last_rows_are_loaded_inside_the_arrays(host, start, fill, width, entries):
    """Groups of four slots of a segment's ELL rows, its padding among them."""
    slots = -(-fill // width) * width
    for q in sorted({*range(0, min(slots, 2048), 4), *range(max(slots - 2048, 0), slots, 4)}):
        assert host.group_source(start, q, entries) == min(start + q, entries - 4)


@pytest.mark.parametrize("length", [1, 511, 512, 513, 1024, 2**31 - 513, 2**31 - 511, MOST])
def test_chunks_of_the_longest_rows(host, length):
    assert host.chunks_of(length, 512) == -(-length // 512)
