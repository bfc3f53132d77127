"""When a CSR product asks for work space: the rules by which it is cut into panels of columns and long rows into chunks.  They
are the host's alone, so no GPU is needed; the times behind the cases stand at the rules (csrc/lf_csr.hip)."""
import numpy as np
import pytest

from liteform_ae_amd import _lib


def work_bytes(rows, cols, degree, feat, longest=0, counts=None):
    """Bytes of work space; -1: the product wants the list of long rows."""
    counts = None if counts is None else np.array(counts, dtype=np.int64)
    return _lib.load().lf_csr_spmm_work_bytes(rows, cols, rows * degree, 0, None if counts is None else counts.ctypes.data, longest, feat,
                                              _lib.LF_DTYPE_F32)


@pytest.mark.parametrize("rows,cols,degree,feat", [(5790, 9198, 170, 704), (6785, 8064, 263, 960), (9138, 6953, 197, 672), (16700, 18782, 197, 288),
                                                   (11060, 20326, 164, 480), (57000, 57000, 28, 64), (120000, 120000, 28, 64)])
def test_no_panels_where_one_launch_is_faster(rows, cols, degree, feat):
    assert work_bytes(rows, cols, degree, feat) == 0


@pytest.mark.parametrize("rows,cols,degree,feat", [(82_900, 82_900, 91, 480), (154_000, 154_000, 144, 160), (65_457, 124_653, 153, 64), (52_653, 64_065, 239, 128),
                                                   (15_953, 21_959, 68, 608), (8_834, 12_228, 127, 992), (18_984, 29_149, 256, 320), (11_316, 14_603, 133, 608)])
def test_panels_where_they_are_faster(rows, cols, degree, feat):
    panels, rest = divmod(work_bytes(rows, cols, degree, feat), 4 * rows)
    assert 1 <= panels <= 7 and rest == 0


# rows, columns, entries a row, N, longest row
@pytest.mark.parametrize("rows,cols,degree,feat,longest", [(15_976, 30_245, 3, 64, 2636), (20_968, 25_716, 3, 256, 5468), (23_998, 33_355, 3, 256, 6192),
                                                           (4000, 4141, 3, 96, 1500), (2000, 1377, 21, 672, 591),
                                                           (2391, 4700, 47, 192, 1900), (57_000, 57_000, 28, 64, 1000), (6500, 6500, 5, 64, 1200)])
def test_long_rows_stay_whole_where_that_is_faster(rows, cols, degree, feat, longest):
    assert work_bytes(rows, cols, degree, feat, longest) == 0
    assert work_bytes(rows, cols, degree, feat, counts=(7, 3, longest)) == 0


@pytest.mark.parametrize("rows,cols,degree,feat,longest", [(116_000, 116_000, 4, 352, 6613), (150_000, 176_328, 4, 320, 13_000), (60_000, 74_951, 3, 96, 4000),
                                                           (9000, 10_951, 3, 672, 10_951), (9000, 10_178, 3, 128, 10_178), (2932, 5251, 311, 128, 5251)])
def test_long_rows_in_chunks_where_that_is_faster(rows, cols, degree, feat, longest):
    assert work_bytes(rows, cols, degree, feat, longest) == -1
    assert work_bytes(rows, cols, degree, feat, counts=(31, 5, longest)) == 31 * 4 * feat


def test_chunks_that_fill_the_cus_unevenly():
    """250 workgroups of rows and two slices of B are two to a CU; 41 chunks make them three."""
    assert work_bytes(2000, 2000, 90, 800, 1528) == -1         # how many chunks there are is not known yet
    assert work_bytes(2000, 2000, 90, 800, counts=(5, 2, 1528)) == 5 * 4 * 800
    assert work_bytes(2000, 2000, 90, 800, counts=(41, 19, 1528)) == 0
