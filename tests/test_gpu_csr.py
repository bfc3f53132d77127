"""CSR products in panels of columns and with long rows in chunks, against scipy in float64.

Tolerance: |C - ref| <= 1e-5 * sum|a||b|, the bound of every product of this package."""
import copy

import numpy as np
import pytest

from liteform_ae_amd import _lib
from liteform_ae_amd.format_matrix_market import MTX
from oracle import liteform_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fa():
    from liteform_ae_amd import format_algos
    return format_algos


@pytest.fixture(scope="module")
def torch():
    import torch
    return torch


def matrix(rng, lens, cols):
    """CSR arrays with `lens` distinct ascending columns per row."""
    def row(n):
        if 4 * n >= cols:
            return np.sort(rng.choice(cols, size=n, replace=False))
        some = np.unique(rng.integers(0, cols, size=2 * n + 8))
        return some[np.sort(rng.choice(len(some), size=n, replace=False))]
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    indices = np.concatenate([row(n) for n in lens]).astype(np.int32)
    return indptr, indices, rng.uniform(-1, 1, size=len(indices)).astype(np.float32)


def operand(torch, rng, cols, feat, b_dtype):
    B = torch.from_numpy(rng.uniform(-1, 1, size=(cols, feat)).astype(np.float32)).cuda()
    return B.to(torch.bfloat16) if b_dtype == "bf16" else B


def work_bytes(fa, g, feat, b_dtype):
    return fa._device_csr(g).csr_work(feat, {"f32": _lib.LF_DTYPE_F32, "bf16": _lib.LF_DTYPE_BF16}[b_dtype])[-1]


@pytest.mark.parametrize("feat,b_dtype,longest", [(512, "f32", 0), (512, "f32", 60_003), (480, "f32", 13_000), (1024, "bf16", 600)])
def test_panels_of_columns(fa, torch, feat, b_dtype, longest):
    """Rows of 0 to 300 entries, rows that lie in one panel only, and rows that the panels leave to the chunks."""
    rng = np.random.default_rng(feat + longest)
    rows, cols = 24_001, 60_003
    lens = rng.integers(0, 300, size=rows)
    lens[::97] = 0
    if longest:
        lens[5::4001] = longest
    indptr, indices, values = matrix(rng, lens, cols)
    for r in range(3, rows, 501):                              # in the last columns, in the first ones
        n = lens[r]
        if n <= 2500:
            indices[indptr[r]:indptr[r + 1]] = (cols - 2500 if r % 2 else 0) + np.sort(rng.choice(2500, size=n, replace=False))
    g = MTX.from_csr(indptr, indices, (rows, cols), data=values)
    B = operand(torch, rng, cols, feat, b_dtype)
    got = fa.spmm_csr(g, B, b_dtype)
    chunks = 4 * feat * sum(-(-n // 512) for n in lens.tolist() if n > 512)
    both = work_bytes(fa, g, feat, b_dtype)
    assert both % (4 * rows) == 0 and both > 0 if longest < cols else both > chunks and (both - chunks) % (4 * rows) == 0
    assert torch.equal(got, fa.spmm_csr(g, B, b_dtype))
    some = np.unique(np.concatenate([np.arange(0, rows, 23), np.arange(3, rows, 501), np.arange(5, rows, 4001), [rows - 1]]))
    ip = np.concatenate([[0], np.cumsum(lens[some])]).astype(np.int64)
    at = np.concatenate([np.arange(indptr[r], indptr[r + 1]) for r in some])
    Bh = B.float().cpu().numpy()
    ref = O.spmm_csr_f64(ip, indices[at], values[at], (len(some), cols), Bh)
    bound = 1e-5 * O.spmm_abs_bound(ip, indices[at], values[at], (len(some), cols), Bh)
    assert (np.abs(got.cpu().numpy()[some] - ref) <= bound).all()


@pytest.mark.parametrize("b_dtype", ["f32", "bf16"])
@pytest.mark.parametrize("feat", [32, 64, 96, 352, 1024])
def test_long_rows_in_chunks(fa, torch, feat, b_dtype):
    """Rows around the length and the multiples of a chunk, next to short and empty ones; also recorded into a graph."""
    rng = np.random.default_rng(feat)
    cols = 30_000
    lens = rng.integers(0, 6, size=700)
    lens[[0, 5, 6, 7, 40, 41, 42, 100, 350, 699]] = [511, 512, 513, 1023, 1024, 1025, 1536, 29_000, 30_000, 2000]
    indptr, indices, values = matrix(rng, lens, cols)
    g = MTX.from_csr(indptr, indices, (len(lens), cols), data=values)
    B = operand(torch, rng, cols, feat, b_dtype)
    got = fa.spmm_csr(g, B, b_dtype)
    chunks = sum(-(-n // 512) for n in lens.tolist() if n > 512)
    assert work_bytes(fa, g, feat, b_dtype) == 4 * chunks * feat
    Bh = B.float().cpu().numpy()
    ref = O.spmm_csr_f64(indptr, indices, values, (len(lens), cols), Bh)
    bound = 1e-5 * O.spmm_abs_bound(indptr, indices, values, (len(lens), cols), Bh)
    assert (np.abs(got.cpu().numpy() - ref) <= bound).all()
    twin = copy.deepcopy(g)                                    # with its own list of long rows
    assert torch.equal(got, fa.spmm_csr(twin, B, b_dtype))
    fresh = MTX.from_csr(indptr, indices, (len(lens), cols), data=values)
    fa._device_csr(fresh)                                      # on the GPU, but without a product yet
    for m in (g, fresh):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = fa.spmm_csr(m, B, b_dtype)
        for _ in range(3):
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            if m is g:
                assert torch.equal(out, got)
            assert (np.abs(out.cpu().numpy() - ref) <= bound).all()


@pytest.mark.parametrize("rows,average", [(1, 95), (1, 96), (3, 207), (5, 208), (700, 300), (12_288, 96), (12_288, 208), (12_289, 96), (12_289, 208),
                                          (24_575, 208), (24_576, 208)])
def test_rows_of_a_workgroup(fa, torch, rows, average):
    """Where 2, 4, 8 or 16 rows go to a workgroup; rows of the average, empty ones and some of twice as much."""
    rng = np.random.default_rng(rows + average)
    cols = 3_001
    lens = np.full(rows, average)
    if rows > 3:
        lens[1:rows - rows % 4:4], lens[2:rows - rows % 4:4] = 0, 2 * average
    assert lens.sum() == average * rows
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    first = rng.integers(0, cols, size=rows)
    at = np.arange(indptr[-1]) - np.repeat(indptr[:-1], lens)
    step = np.maximum(1, (cols - 1) // np.maximum(lens, 1))
    indices = (np.repeat(first % step, lens) + at * np.repeat(step, lens)).astype(np.int32)
    assert indices.max() < cols
    values = rng.uniform(-1, 1, size=len(indices)).astype(np.float32)
    g = MTX.from_csr(indptr, indices, (rows, cols), data=values)
    B = operand(torch, rng, cols, 64, "f32")
    got = fa.spmm_csr(g, B).cpu().numpy()
    Bh = B.cpu().numpy()
    ref = O.spmm_csr_f64(indptr, indices, values, (rows, cols), Bh)
    bound = 1e-5 * O.spmm_abs_bound(indptr, indices, values, (rows, cols), Bh)
    assert (np.abs(got - ref) <= bound).all()


@pytest.mark.parametrize("rows,average", [(4, 96), (7, 100), (1001, 97), (5120, 96), (5119, 250), (5121, 150), (12_288, 250), (12_289, 250), (24_573, 210)])
def test_few_uneven_rows(fa, torch, rows, average):
    """Two rows to a workgroup and four, and the least numbers of rows that take four and eight: rows of the average, empty ones, some of twice
    as much and a long one."""
    rng = np.random.default_rng(rows + average)
    cols = 3_001
    lens = np.full(rows, average)
    lens[1::4], lens[3::4] = 0, 2 * average                    # the average still, or a little below it
    lens[0] = 1600
    indptr, indices, values = matrix(rng, lens, cols)
    assert indptr[-1] >= 96 * rows and lens.max() * rows >= 3 * indptr[-1]
    g = MTX.from_csr(indptr, indices, (rows, cols), data=values)
    B = operand(torch, rng, cols, 96, "f32")
    got = fa.spmm_csr(g, B).cpu().numpy()
    Bh = B.cpu().numpy()
    ref = O.spmm_csr_f64(indptr, indices, values, (rows, cols), Bh)
    bound = 1e-5 * O.spmm_abs_bound(indptr, indices, values, (rows, cols), Bh)
    assert (np.abs(got - ref) <= bound).all()


def triplets(rng, lens, cols, twice=0):
    """Triplets of rows of `lens` distinct columns in random order, `twice` of them given again."""
    indptr, indices, values = matrix(rng, lens, cols)
    row = np.repeat(np.arange(len(lens)), lens)
    order = rng.permutation(len(row))
    order = np.concatenate([order, order[:twice]])
    return row[order].astype(np.int32), indices[order], values[order]


@pytest.mark.parametrize("rows,cols,average,longest,twice", [
    (1, 60, 40, 40, 0), (3001, 4001, 20, 700, 0), (3001, 4001, 20, 700, 9), (70_001, 3000, 12, 40, 0),
    (4, 9000, 1200, 5000, 0),                                  # a bin of more than 4096 entries
    (2_000_003, 2_000_003, 1, 1000, 0), (255, 8_400_000, 30, 90, 0), (256, 8_400_000, 30, 90, 3), (511, 8_400_000, 30, 90, 0)])      # not in bins
def test_triplets_know_their_longest_row(fa, torch, rows, cols, average, longest, twice):
    """The first product of a matrix made from triplets is the one call that it is for CSR arrays: no list of long rows unless they are cut."""
    rng = np.random.default_rng(rows + twice)
    lens = rng.integers(0, average + 1, size=rows)
    lens[rows // 2] = longest
    if rows == 511:
        lens[254], lens[rows // 2] = longest, 1                # the last row of a workgroup's
    row, col, data = triplets(rng, lens, cols, twice)
    g = MTX.from_coo(row, col, (rows, cols), data=data)
    dev = fa._device_csr(g)
    assert dev.path == "coo" and (dev._longest == longest if not twice else longest <= dev._longest <= longest + twice)
    B = torch.rand((cols, 32), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)) - 0.5
    got = fa.spmm_csr(g, B)
    assert dev._long_rows is None and not dev._csr_work
    at, inverse = np.unique(col, return_inverse=True)          # the rows of B that are met
    ref = torch.zeros((rows, 32), dtype=torch.float64, device="cuda")
    bound = torch.zeros_like(ref)
    rows_at, met = torch.from_numpy(row).cuda().long(), B[torch.from_numpy(at).cuda().long()].double()[torch.from_numpy(inverse).cuda()]
    products = torch.from_numpy(data).cuda().double()[:, None] * met
    ref.index_add_(0, rows_at, products)
    bound.index_add_(0, rows_at, products.abs())
    assert bool(((got - ref).abs() <= 1e-5 * bound).all())


def test_no_triplets(fa, torch):
    none = np.zeros(0, dtype=np.int32)
    g = MTX.from_coo(none, none, (5, 7), data=np.zeros(0, dtype=np.float32))
    assert fa._device_csr(g)._longest == 0
    assert not fa.spmm_csr(g, torch.rand((7, 32), device="cuda")).any()


@pytest.mark.parametrize("twice", [0, 300])
def test_panels_and_chunks_of_a_matrix_from_triplets(fa, torch, twice):
    rng = np.random.default_rng(twice)
    rows, cols, feat = 24_577, 30_011, 512
    lens = rng.integers(0, 180, size=rows)
    lens[7] = cols
    row, col, data = triplets(rng, lens, cols, twice)
    g = MTX.from_coo(row, col, (rows, cols), data=data)
    B = operand(torch, rng, cols, feat, "f32")
    got = fa.spmm_csr(g, B)
    chunks = 4 * feat * sum(-(-n // 512) for n in lens.tolist() if n > 512)
    both = work_bytes(fa, g, feat, "f32")
    assert both > chunks and (both - chunks) % (4 * rows) == 0
    some = np.unique(np.concatenate([np.arange(0, rows, 37), [7, rows - 1]]))
    mine = np.isin(row, some)
    A = np.searchsorted(some, row[mine])
    Bh = B.cpu().numpy()
    import scipy.sparse as sp
    S = sp.coo_matrix((data[mine].astype(np.float64), (A, col[mine])), shape=(len(some), cols)).tocsr()
    bound = 1e-5 * (abs(S) @ np.abs(Bh.astype(np.float64)))
    assert (np.abs(got.cpu().numpy()[some] - S @ Bh.astype(np.float64)) <= bound).all()


@pytest.mark.parametrize("b_dtype,cols", [("f32", 1_060_003), ("bf16", 2_110_003)])
def test_long_rows_in_chunks_of_a_b_past_4_gb(fa, torch, b_dtype, cols):
    rng = np.random.default_rng(cols)
    feat = 1024
    lens = rng.integers(0, 6, size=300)
    lens[[0, 7, 150, 299]] = [513, 60_000, 1025, 20_000]
    indptr, indices, values = matrix(rng, lens, cols)
    indices[indptr[8] - 1] = cols - 1                          # the last row of B
    g = MTX.from_csr(indptr, indices, (len(lens), cols), data=values)
    gen = torch.Generator(device="cuda").manual_seed(cols)
    B = torch.rand((cols, feat), device="cuda", generator=gen, dtype=torch.float32 if b_dtype == "f32" else torch.bfloat16).sub_(0.5)
    assert B.numel() * B.element_size() > 2**32
    got = fa.spmm_csr(g, B, b_dtype).double()
    assert work_bytes(fa, g, feat, b_dtype) == 4 * feat * sum(-(-n // 512) for n in lens.tolist() if n > 512)
    for r, n in enumerate(lens):
        if n == 0:
            assert not got[r].any()
            continue
        at = torch.from_numpy(indices[indptr[r]:indptr[r + 1]]).cuda().long()
        x = torch.from_numpy(values[indptr[r]:indptr[r + 1]]).cuda().double()
        rows_of_b = B[at].double()
        assert bool(((got[r] - x @ rows_of_b).abs() <= 1e-5 * (x.abs() @ rows_of_b.abs())).all()), r
