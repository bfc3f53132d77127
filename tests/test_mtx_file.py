"""MTX(path): the MatrixMarket ingest of the reference's container
(playground_pipline/format_matrix_market.py:58-65): the file is read with scipy.io.mmread,
every stored value is replaced by 1, the name is the file's stem.  The CPU part checks the
container; the GPU part takes the same files through the device ingest, the search, the
builder and the product."""
import numpy as np
import pytest
import scipy.sparse as sp

from liteform_ae_amd.format_matrix_market import MTX
from oracle import liteform_oracle as O

# 5 x 6, coordinate entries unsorted; (2,3) and (4,1) appear twice (MatrixMarket allows repeated
# coordinates in a general matrix; scipy keeps them as separate COO triplets)
REAL_GENERAL = """%%MatrixMarket matrix coordinate real general
% unsorted, with repeated coordinates
5 6 9
4 1 2.5
1 1 -1.0
2 3 0.25
5 6 7.0
2 3 4.0
3 2 1e-3
1 5 3.0
4 1 -2.5
2 1 9.0
"""

PATTERN_GENERAL = """%%MatrixMarket matrix coordinate pattern general
4 7 6
3 7
1 2
1 1
4 4
2 6
3 1
"""

INTEGER_SYMMETRIC = """%%MatrixMarket matrix coordinate integer symmetric
4 4 4
1 1 5
3 1 2
4 2 -3
4 4 8
"""

FILES = {"real_general": REAL_GENERAL, "pattern_general": PATTERN_GENERAL, "integer_symmetric": INTEGER_SYMMETRIC}
# stored triplets after reading (row, col), 0-based, in file order; symmetric files are expanded by mmread
TRIPLETS = {
    "real_general": ((5, 6), [(3, 0), (0, 0), (1, 2), (4, 5), (1, 2), (2, 1), (0, 4), (3, 0), (1, 0)]),
    "pattern_general": ((4, 7), [(2, 6), (0, 1), (0, 0), (3, 3), (1, 5), (2, 0)]),
    "integer_symmetric": ((4, 4), [(0, 0), (2, 0), (3, 1), (3, 3), (0, 2), (1, 3)]),
}


@pytest.fixture(params=sorted(FILES))
def mtx_file(request, tmp_path):
    path = tmp_path / f"{request.param}.mtx"
    path.write_text(FILES[request.param])
    return request.param, str(path)


def test_mtx_path_reads_pattern_and_forces_ones(mtx_file):
    name, path = mtx_file
    g = MTX(path)
    shape, trip = TRIPLETS[name]
    assert g.name == name
    assert g.coo_mtx.shape == shape
    assert g.num_src_nodes() == shape[0] and g.num_dst_nodes() == shape[1]
    assert g.num_edges() == len(trip)
    assert sorted(zip(g.coo_mtx.row.tolist(), g.coo_mtx.col.tolist())) == sorted(trip)
    assert (g.coo_mtx.data == 1).all() and g.coo_mtx.data.dtype == np.float64     # format_matrix_market.py:63-64
    indptr, indices, data = g.adj_tensors("csr")
    want = sp.coo_matrix((np.ones(len(trip)), tuple(zip(*trip))), shape=shape).tocsr()
    np.testing.assert_array_equal(indptr, want.indptr)
    np.testing.assert_array_equal(indices, want.indices)
    np.testing.assert_array_equal(data, want.data)        # repeated coordinates add up to 2
    # the container's product is the scipy one
    B = np.arange(shape[1] * 3, dtype=np.float64).reshape(shape[1], 3)
    np.testing.assert_array_equal(g.dot(B), want @ B)


def _sent_to_the_gpu(monkeypatch, g):
    """What _DeviceCSR would upload for g: ("csr" or "coo", its arrays, its entry count)."""
    import types
    from liteform_ae_amd import format_algos as fa

    class Recorder(fa._DeviceCSR):
        def _from_csr(self, csr, unit_values):
            self.sent = tuple(np.array(x) for x in (csr.indptr, csr.indices, csr.data))
            return True

        def _from_coo(self, row, col, data):
            self.sent = tuple(np.array(x) for x in (row, col, data))

    stream = types.SimpleNamespace(synchronize=lambda: None)
    monkeypatch.setattr(fa, "_torch", lambda: types.SimpleNamespace(cuda=types.SimpleNamespace(current_stream=lambda: stream)))
    dev = Recorder(g)
    return dev.path, dev.sent, dev.coo_nnz


def _edits():
    """In-place changes of a COO matrix, each through what scipy offers for it."""
    def new_data(coo):
        coo.data = np.full(len(coo.data), 3.0, dtype=np.float32)
    return [lambda coo: coo.sum_duplicates(), lambda coo: coo.eliminate_zeros(), new_data]


@pytest.mark.parametrize("edit", _edits(), ids=["sum_duplicates", "eliminate_zeros", "data"])
def test_changes_of_the_coo_view_reach_the_gpu(monkeypatch, edit):
    """A container made from triplets: what is done to its COO view before the first use counts."""
    row, col = np.array([0, 0, 2], dtype=np.int32), np.array([1, 1, 0], dtype=np.int32)
    data = np.array([1.0, 2.0, 0.0], dtype=np.float32)
    g = MTX.from_coo(row, col, (3, 2), data=data)
    assert _sent_to_the_gpu(monkeypatch, g)[1][2] is not None
    edit(g.coo_mtx)
    want = sp.coo_matrix((data, (row, col)), shape=(3, 2))
    edit(want)
    path, sent, nnz = _sent_to_the_gpu(monkeypatch, g)
    assert path == "coo" and nnz == g.num_edges() == want.nnz
    for got, ref in zip(sent, (want.row, want.col, want.data)):
        np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("edit", _edits(), ids=["sum_duplicates", "eliminate_zeros", "data"])
def test_changes_of_the_coo_view_of_csr_arrays_reach_the_gpu(monkeypatch, edit):
    """The same for a container made from CSR arrays, which go up as they are only while its COO view
    has not been handed out; the host's CSR view follows the change as well."""
    indptr, indices = np.array([0, 2, 2, 3], dtype=np.int32), np.array([1, 1, 0], dtype=np.int32)
    data = np.array([1.0, 2.0, 0.0], dtype=np.float32)
    g = MTX.from_csr(indptr, indices, (3, 2), data=data)
    g.adj_tensors("csr")
    path, sent, _ = _sent_to_the_gpu(monkeypatch, g)
    assert path == "csr"
    np.testing.assert_array_equal(sent[2], data)
    edit(g.coo_mtx)
    want = sp.csr_matrix((data, indices, indptr), shape=(3, 2)).tocoo()
    edit(want)
    path, sent, nnz = _sent_to_the_gpu(monkeypatch, g)
    assert path == "coo" and nnz == g.num_edges() == want.nnz
    for got, ref in zip(sent, (want.row, want.col, want.data)):
        np.testing.assert_array_equal(got, ref)
    unedited = MTX.from_csr(np.array([0, 1]), indices[:1], (1, 2), data=data[:1])     # (canonical: the CSR view is the source)
    unedited.adj_tensors("csr")
    edit(unedited.coo_mtx)
    np.testing.assert_array_equal(unedited.adj_tensors("csr")[2], unedited.coo_mtx.tocsr().data)


def test_a_copy_on_the_gpu_is_kept_until_the_matrix_is_replaced():
    """Looking at the COO view is no new matrix; assigning one is."""
    from liteform_ae_amd import format_algos as fa
    g = MTX.from_coo(np.array([0, 1], dtype=np.int32), np.array([1, 0], dtype=np.int32), (2, 2))
    before = fa._matrix_identity(g)
    assert g.coo_mtx.nnz == 2 and g.dot(np.eye(2)).shape == (2, 2) and fa._matrix_identity(g) is before
    g.coo_mtx = sp.identity(2, format="coo")
    assert fa._matrix_identity(g) is not before


@pytest.mark.gpu
def test_mtx_path_through_the_gpu_pipeline(mtx_file):
    import torch
    from liteform_ae_amd import format_algos as fa
    name, path = mtx_file
    g = MTX(path)
    shape, trip = TRIPLETS[name]
    dev = fa._DeviceCSR(g)
    want = g.coo_mtx.tocsr()
    want.sum_duplicates()
    assert dev.coo_nnz == len(trip) and dev.nnz == want.nnz
    np.testing.assert_array_equal(dev.indptr.cpu().numpy(), want.indptr)
    np.testing.assert_array_equal(dev.indices.cpu().numpy(), want.indices)
    np.testing.assert_array_equal(dev.values.cpu().numpy(), want.data.astype(np.float32))
    assert dev.all_ones == (want.nnz == len(trip))
    # search and builder against the oracle (degrees come from the raw triplets, fills from the CSR)
    cfg = fa.search_bucket_config(g, 1, fa.CostModelSettings(32, 1))
    assert cfg == O.search_bucket_config(g, 1, O.OracleCostModelSettings(32, 1))
    got = fa.build_hyb_format(g, cfg)
    ref = O.build_hyb_format_closed_form(g, cfg)
    for a_parts, b_parts in zip(got, ref):
        for ab, bb in zip(a_parts, b_parts):
            for x, y in zip(ab, bb):
                assert x.shape == y.shape and np.array_equal(x, y)
    # product with the summed values against the container's own scipy product
    B = np.arange(shape[1] * 32, dtype=np.float32).reshape(shape[1], 32) % 7
    out = fa.spmm_hyb(fa.build_hyb_format_device(g, cfg), torch.from_numpy(B).cuda()).cpu().numpy()
    np.testing.assert_array_equal(out, g.dot(B.astype(np.float64)).astype(np.float32))
