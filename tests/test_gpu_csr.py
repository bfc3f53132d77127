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


@pytest.mark.parametrize("rows,average", [(4, 96), (7, 100), (1001, 97), (5120, 96), (5119, 250), (5121, 250)])
def test_few_uneven_rows(fa, torch, rows, average):
    """Two rows to a workgroup, and the least number of rows that takes eight again: rows of the average, empty ones, some of twice
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
