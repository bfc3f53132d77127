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
                                                   (15_953, 21_959, 68, 608), (8_834, 12_228, 127, 992)])
def test_panels_where_they_are_faster(rows, cols, degree, feat):
    panels, rest = divmod(work_bytes(rows, cols, degree, feat), 4 * rows)
    assert 1 <= panels <= 7 and rest == 0
