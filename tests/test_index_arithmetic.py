"""The index arithmetic of the kernels (csrc/lf_index.h), compiled for the host, at the largest arrays that are accepted:
no GPU, and no array of that size, is needed to see a 32-bit sum pass 2^31."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MOST = 2**31 - 1                       # entries of a matrix

SOURCE = """
#include "lf_index.h"
extern "C" int group_source(int start, int fill, int q) { return lf::group_source(start, fill, q); }
extern "C" int fours_inside(int j, int ahead, int fill) { return lf::fours_inside(j, ahead, fill); }
extern "C" int fours_source(int j, int ahead, int fill) { return lf::fours_source(j, ahead, fill); }
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    where = tmp_path_factory.mktemp("index")
    (where / "index.cpp").write_text(SOURCE)
    lib = str(where / "index.so")
    # (sums that wrap, as the GPU's do)
    subprocess.run([cxx, "-std=c++17", "-O1", "-fwrapv", "-shared", "-fPIC", "-I", os.path.join(ROOT, "liteform_ae_amd", "csrc"),
                    str(where / "index.cpp"), "-o", lib], check=True)
    return ctypes.CDLL(lib)


@pytest.mark.parametrize("start,fill,width", [(MOST - 16, 16, 32), (2**31 - 20, 17, 32), (MOST - 1, 1, 1024), (MOST - 3, 3, 4), (MOST - 1025, 1025, 1024),
                                              (0, 5, 8), (7, 0, 8), (MOST, 0, 4)])
def test_padding_of_the_last_rows_reads_inside_the_arrays(host, start, fill, width):
    """Groups of four slots of a segment's ELL rows: the ones that hold entries start at theirs, the others somewhere
    in the segment."""
    slots = -(-fill // width) * width
    for q in range(0, max(slots, 4), 4):
        source = host.group_source(start, fill, q)
        if q < fill:
            assert source == start + q
        else:
            assert start <= source <= max(start + fill - 1, start)


@pytest.mark.parametrize("fill", [4, 5, 255, 256, 257, 1023, 1024, 1025, 8193, 2**31 - 1024, 2**31 - 1023, MOST - 1, MOST])
def test_the_end_of_a_long_segment_is_walked_inside_it(host, fill):
    """The last pieces of 1024 entries of a segment, four to a lane: every entry is loaded, nothing past the end is."""
    for j in {max((fill - 1) // 1024 * 1024 - k * 1024, 0) for k in range(2)}:
        for ahead in range(0, 1024, 4):
            inside = j + ahead < fill
            assert host.fours_inside(j, ahead, fill) == inside
            assert host.fours_source(j, ahead, fill) == min(j + ahead, fill - 4)
