"""GPU parity of the format pass (statistics, search, hyb composition) with the oracle.

Everything goes through the C ABI (ctypes) behind the reference-shaped Python functions.
Format structures must match bit for bit."""
import numpy as np
import pytest

from liteform_ae_amd.format_matrix_market import MTX
from oracle import liteform_oracle as O

from helpers import assert_hyb_equal, mtx_from_rows, skewed_matrix, stats_from_oracle

pytestmark = pytest.mark.gpu

HAND = [[0, 1, 2, 5], [1], [], [0, 1, 2, 3, 4, 6], [2, 7], [0, 3, 4, 5, 6]]


@pytest.fixture(scope="module")
def fa():
    from liteform_ae_amd import format_algos
    return format_algos


def test_hand_example_end_to_end(fa):
    g = mtx_from_rows(HAND, (6, 8))
    cfg = fa.search_bucket_config(g, 2, fa.CostModelSettings(32, 2))
    assert cfg == [[1, 4], [1, 2]]
    rows, cols, mask = fa.build_hyb_format(g, cfg)
    assert rows[0][1].tolist() == [0, 3, 5]
    assert cols[0][1].tolist() == [[0, 1, 2, 0], [0, 1, 2, 3], [0, 3, 0, 0]]
    assert mask[0][1].tolist() == [[1, 1, 1, 0], [1, 1, 1, 1], [1, 1, 0, 0]]
    assert rows[1][1].tolist() == [3, 5, 5]
    assert cols[1][1].tolist() == [[4, 6], [4, 5], [6, 0]]
    assert mask[1][1].tolist() == [[1, 1], [1, 1], [1, 0]]
    assert rows[0][0].dtype == np.int64 and cols[0][1].shape == (3, 4)
    assert_hyb_equal((rows, cols, mask), O.build_hyb_format_sequential(g, cfg))


@pytest.mark.parametrize("seed", range(8))
def test_bucket_stats_match_oracle(fa, seed):
    rng = np.random.default_rng(40 + seed)
    nr, nc = int(rng.integers(100, 3000)), int(rng.integers(100, 3000))
    parts = int(rng.choice([1, 2, 3, 7, 16]))
    g = skewed_matrix(rng, nr, nc, mean_deg=float(rng.choice([3, 8, 20])), heavy_rows=3, values=False)
    stats, hist = fa.bucket_statistics(g, parts)
    wstats, whist = stats_from_oracle(g, parts)
    np.testing.assert_array_equal(stats, wstats)
    np.testing.assert_array_equal(hist, whist)


@pytest.mark.parametrize("nr,nc,parts,limit", [
    (131072, 70_001, 1, 1024),          # the smallest matrix whose column sets are LDS bitmaps
    (131071, 70_001, 1, 1024),          # ... and the largest below it
    (131073, 1_245_184, 1, 1024),       # the largest single slice
    (131073, 1_245_185, 1, 1024),       # two slices
    (140_000, 2_600_011, 2, 1024),      # two partitions of two slices
    (140_000, 31, 2, 1024),             # a bitmap of one word
    (131072, 9000, 46, 1024),           # the most (partition, class) pairs
    (131072, 9000, 47, 1024),           # one more: byte planes
    (131072, 40_000, 3, 16),            # most entries in segments beyond the last class's width
])
def test_column_sets_of_large_matrices(fa, nr, nc, parts, limit):
    rng = np.random.default_rng(nr + nc + parts)
    deg = np.minimum(rng.geometric(0.2, size=nr) - 1, nc)
    deg[rng.integers(0, nr, size=40)] = np.minimum(rng.integers(60, 1100, size=40), nc)
    deg[[0, nr // 2, nr - 1]] = min(nc, 8193), min(nc, 8192), min(nc, 30_000)
    row = np.repeat(np.arange(nr), deg)
    key = np.unique(row * nc + rng.integers(0, nc, size=len(row)))
    row, col = key // nc, key % nc
    g = MTX.from_coo(row, col, (nr, nc))
    stats, hist = fa.bucket_statistics(g, parts, width_limit=limit)

    psize = -(-nc // parts)
    seg = (col // psize) * nr + row
    fill = np.bincount(seg, minlength=parts * nr)
    pow2 = np.where(fill > 0, 2 ** np.ceil(np.log2(np.maximum(fill, 1))).astype(np.int64), 0)
    k = np.log2(np.maximum(np.minimum(pow2, limit), 1)).astype(np.int64)
    touched = np.unique(k[seg] * nc + col)                        # every (class, column) once
    masks = np.zeros(nc, np.int64)
    np.add.at(masks, touched % nc, 1 << (touched // nc))
    for p in range(parts):
        lo, hi = p * psize, min(nc, (p + 1) * psize)
        want = np.bincount(masks[lo:hi], minlength=2048) if hi > lo else np.zeros(2048, np.int64)
        np.testing.assert_array_equal(hist[p], want)
        mine, f = k[p * nr:(p + 1) * nr], fill[p * nr:(p + 1) * nr]
        for c in range(11):
            on = (f > 0) & (mine == c)
            rows = np.maximum(1, pow2[p * nr:(p + 1) * nr][on] // limit).sum()
            assert stats[p, c].tolist() == [rows, f[on].sum(), on.sum(), 0]


@pytest.mark.parametrize("nc,parts", [(30_000, 1), (1_300_000, 1), (2_600_000, 1), (2_600_000, 3)])       # slices: 1, 2, 3, 1
@pytest.mark.parametrize("copies", [1, 3])       # of every entry: the class follows the degree, the columns are there once
def test_column_sets_by_length(fa, nc, parts, copies):
    nr = 131072
    rng = np.random.default_rng(nc + copies)
    edges = np.array([1, 2, 3, 4, 5, 7, 8, 9, 12, 13, 16, 17, 31, 32, 33, 63, 64, 65, 128, 129, 255, 256, 257, 260, 512, 513, 1025, 1300])
    deg = rng.choice([1, 2, 3, 4, 6], size=nr)
    deg[-2 * len(edges):] = np.concatenate([edges, edges[::-1]])  # among them the last segments of the index array, of one entry
    row = np.repeat(np.arange(nr), deg)
    col = (rng.integers(0, nc, size=nr)[row] + np.arange(len(row))) % nc if parts == 1 else rng.integers(0, nc, size=len(row))
    key = np.unique(row * nc + col)
    row, col = key // nc, key % nc
    g = MTX.from_coo(np.tile(row, copies), np.tile(col, copies), (nr, nc))
    stats, hist = fa.bucket_statistics(g, parts)
    psize = -(-nc // parts)
    seg = (col // psize) * nr + row
    fill = np.bincount(seg, minlength=parts * nr) * copies
    k = np.minimum(np.ceil(np.log2(np.maximum(fill, 1))).astype(np.int64), 10)
    touched = np.unique(k[seg] * nc + col)
    masks = np.zeros(nc, np.int64)
    np.add.at(masks, touched % nc, 1 << (touched // nc))
    for p in range(parts):
        np.testing.assert_array_equal(hist[p], np.bincount(masks[p * psize:(p + 1) * psize], minlength=2048))


@pytest.mark.parametrize("seed", range(8))
def test_search_matches_oracle(fa, seed):
    rng = np.random.default_rng(60 + seed)
    nr, nc = int(rng.integers(200, 2500)), int(rng.integers(200, 2500))
    parts = int(rng.choice([1, 2, 4, 8]))
    feat = int(rng.choice([32, 128, 512]))
    g = skewed_matrix(rng, nr, nc, mean_deg=8, heavy_rows=2, values=False)
    try:
        want = O.search_bucket_config(g, parts, O.OracleCostModelSettings(feat, parts))
    except ValueError:
        with pytest.raises(ValueError):
            fa.search_bucket_config(g, parts, fa.CostModelSettings(feat, parts))
        return
    assert fa.search_bucket_config(g, parts, fa.CostModelSettings(feat, parts)) == want


def test_single_nonzero_partition_raises_value_error(fa):
    g = mtx_from_rows([[3]], (1, 8))
    with pytest.raises(ValueError, match="only having 1 non-zero element"):
        fa.search_bucket_config(g, 1, fa.CostModelSettings(32, 1))


@pytest.mark.parametrize("seed", range(10))
def test_builder_matches_sequential_oracle(fa, seed):
    rng = np.random.default_rng(80 + seed)
    nr, nc = int(rng.integers(30, 700)), int(rng.integers(30, 700))
    parts = int(rng.choice([1, 2, 3, 5]))
    g = skewed_matrix(rng, nr, nc, mean_deg=6, heavy_rows=2, values=False)
    all_w = [1 << i for i in range(8)]
    widths = [sorted(rng.choice(all_w, size=int(rng.integers(1, 6)), replace=False).tolist())
              for _ in range(parts)]
    got = fa.build_hyb_format(g, widths)
    assert_hyb_equal(got, O.build_hyb_format_sequential(g, widths))


def test_builder_with_searched_config_mid_size(fa):
    rng = np.random.default_rng(7)
    g = skewed_matrix(rng, 20000, 20000, mean_deg=12, heavy_rows=5, heavy_len=6000, values=False)
    for parts in (1, 4):
        cfg = fa.search_bucket_config(g, parts, fa.CostModelSettings(128, parts))
        assert cfg == O.search_bucket_config(g, parts, O.OracleCostModelSettings(128, parts))
        assert_hyb_equal(fa.build_hyb_format(g, cfg), O.build_hyb_format_closed_form(g, cfg))


def test_builder_edge_cases(fa):
    # empty matrix rows, an empty partition, a single bucket of width 1 holding a long row
    g = mtx_from_rows([[], [0, 1, 2, 3, 4], [], [1]], (4, 16))
    for widths in ([[1], []], [[8], []], [[1, 2, 4, 8], []]):
        assert_hyb_equal(fa.build_hyb_format(g, widths), O.build_hyb_format_sequential(g, widths))
    with pytest.raises(IndexError):
        fa.build_hyb_format(g, [[], [4]])                 # nonzeros in a partition without widths
    with pytest.raises(AssertionError):
        fa.build_hyb_format(g, [[3], []])                 # not a power of two
    # empty buckets are kept with shapes (0,), (0, W)   (format_algos.py:365-368)
    rows, cols, mask = fa.build_hyb_format(g, [[1, 2, 4, 8], []])
    assert rows[0][1].shape == (0,) and cols[0][1].shape == (0, 2) and mask[0][2].shape == (0, 4)


@pytest.mark.parametrize("lists", [[[2]], [[], [0, 3], []], [[5], [1, 2]], [[0], [1], [2]], [[1], [0, 2, 3]], [[0, 1, 2, 3, 4], [6]], [[3], list(range(9)), [0, 1]]])
@pytest.mark.parametrize("widths", [[1], [2, 8], [4], [16]])
def test_builder_of_few_entries(fa, lists, widths):
    # groups of four slots end where the index array ends, or hold all of it
    row, col = np.array([(i, j) for i, cols in enumerate(lists) for j in cols]).T
    g = MTX.from_coo(row, col, (len(lists), 10), data=np.arange(1, len(row) + 1, dtype=np.float32))
    assert_hyb_equal(fa.build_hyb_format(g, [widths]), O.build_hyb_format_sequential(g, [widths]))
    fmt = fa.build_hyb_format_device(g, [widths])
    seen = []
    for k in range(fmt.num_buckets):
        rows, cols, vals = (x.cpu().numpy() for x in fmt.slab(k)[:3])
        at = np.flatnonzero(vals)
        seen += zip(vals[at].tolist(), rows[at // widths[k]].tolist(), cols[at].tolist())
    assert sorted(seen) == [(i + 1.0, r, c) for i, (r, c) in enumerate(zip(row.tolist(), col.tolist()))]


def test_duplicate_coo_entries(fa):
    """COO duplicates raise the degree but not the fill (format_algos.py:250-254)."""
    from liteform_ae_amd.format_matrix_market import MTX
    rng = np.random.default_rng(11)
    r = rng.integers(0, 50, size=600)
    c = rng.integers(0, 64, size=600)
    g = MTX.from_coo(r, c, (50, 64))
    assert g.num_edges() != g.adj_tensors("csr")[1].shape[0]      # there are duplicates
    for parts in (1, 2):
        widths = [[2, 8, 16]] * parts
        assert_hyb_equal(fa.build_hyb_format(g, widths), O.build_hyb_format_sequential(g, widths))
        stats, hist = fa.bucket_statistics(g, parts)
        wstats, whist = stats_from_oracle(g, parts)
        np.testing.assert_array_equal(stats, wstats)
        np.testing.assert_array_equal(hist, whist)


def test_workload_shapes_scaled(fa):
    from liteform_ae_amd.synthetic import make_workload
    for name, scale, parts in (("cfg1", 1.0, 1), ("cfg2", 0.05, 2), ("cfg3", 0.005, 1), ("cfg3", 0.005, 4),
                               ("cfg4", 0.004, 1), ("cfg5", 0.01, 2)):
        wl = make_workload(name, scale)
        g = wl.matrix
        cfg = fa.search_bucket_config(g, parts, fa.CostModelSettings(wl.feat_size, parts))
        assert cfg == O.search_bucket_config(g, parts, O.OracleCostModelSettings(wl.feat_size, parts)), name
        assert_hyb_equal(fa.build_hyb_format(g, cfg), O.build_hyb_format_closed_form(g, cfg))


def test_device_ingest_matches_scipy_tocsr(fa):
    """lf_coo_to_csr against coo.tocsr() (format_matrix_market.py:74-76): unsorted triplets,
    duplicates, empty rows, rectangular shapes."""
    import scipy.sparse as sp
    from liteform_ae_amd.format_matrix_market import MTX
    rng = np.random.default_rng(17)
    for (nr, nc, n, weighted) in ((1, 1, 1, False), (300, 500, 4000, False), (2000, 70, 30000, True),
                                  (5, 100000, 2000, True), (100000, 3, 50000, False)):
        r = rng.integers(0, nr, size=n)
        c = rng.integers(0, nc, size=n)
        d = rng.uniform(-1, 1, size=n) if weighted else None
        g = MTX.from_coo(r, c, (nr, nc), data=d)
        dev = fa._DeviceCSR(g)
        want = g.coo_mtx.tocsr()
        want.sum_duplicates()
        assert dev.nnz == want.nnz and dev.coo_nnz == n
        np.testing.assert_array_equal(dev.indptr.cpu().numpy(), want.indptr)
        np.testing.assert_array_equal(dev.indices.cpu().numpy(), want.indices)
        np.testing.assert_allclose(dev.values.cpu().numpy(), want.data, rtol=1e-5, atol=1e-6)
        assert dev.all_ones == (not weighted and want.nnz == n)
    g = MTX.from_coo(np.zeros(0, np.int64), np.zeros(0, np.int64), (7, 9))
    dev = fa._DeviceCSR(g)
    assert dev.nnz == 0 and dev.indptr.cpu().numpy().tolist() == [0] * 8


def coo_case(name):
    """(rows, columns, shape) of triplets in no order, each place once."""
    rng = np.random.default_rng(sum(map(ord, name)))
    if name.startswith("n="):                              # entries around a chunk, a handful of rows to a bin
        n, (nr, nc) = int(name[2:]), (700, 900)
        key = rng.choice(nr * nc, size=n, replace=False)
        return key // nc, key % nc, (nr, nc)
    shapes = {"giant rows": (600, 40_000, [1024, 1025, 4096, 4097, 9000, 32_768]), "a row past the limit": (40, 90_000, [32_769, 5000]),
              "crowded columns": (64, 1 << 21, [3000, 900, 2000, 1500]), "one column": (5000, 1, []), "one row": (1, 3000, [2500]),
              "few entries": (2_100_000, 50, []), "wide keys": (300_000, 1 << 23, []), "long bins": (512 * 40, 30_000, [4000] * 60)}
    if name in shapes:
        nr, nc, lens = shapes[name]
    else:                                                  # 256 rows to a bin: what stands in the bins named
        nr, nc = 200_000, 150_000
        long_rows = [0, 2, 1100, 0, 3000, 1, 1025, 2048, 0, 5]
        bins = {"adjacent long rows": {100: [*long_rows * 6, 4097, 0, 4500, 9000], 101: [1100] * 60, 781: long_rows},
                # sums of whole windows with empty rows behind them, the last bin (64 rows) among them, and one more or less
                "whole windows": {3: [4096], 4: [4097], 5: [4096, 4096], 6: [0, 4097, 4095], 7: [4095, 4098], 8: [8191, 1], 9: [8192], 10: [1, 8191, 0, 1],
                                  11: [12_288, 0, 0, 1], 12: [1, 12_288], 13: [100] * 81 + [92], 14: [100] * 82, 15: [32] * 256, 781: [0, 5000, 3192]},
                "rows by length": {i: rng.integers(max(1, 400 // (i + 1)), 500 // (i + 1) + 1, size=256) for i in range(60)},
                "a bin of the most": {50: [70_000, 3, 0, 30_000, *[250] * 124, 69]}, "a bin past the limit": {50: [70_000, 3, 0, 30_000, *[250] * 124, 70]},
                "a crowded long row": {50: [9000, 20]}}[name]
        deg = np.zeros(nr, np.int64) if name == "whole windows" else (rng.random(nr) < 0.2).astype(np.int64)
        for b, lens in bins.items():
            deg[256 * b:256 * b + 256] = 0
            deg[256 * b:256 * b + len(lens)] = lens
        row = np.repeat(np.arange(nr), deg)
        col = np.concatenate([rng.choice(10_000 if name == "a crowded long row" and d > 20 else nc, size=d, replace=False) for d in deg if d])
        return row, col, (nr, nc)
    deg = np.minimum(rng.integers(0, 9, size=nr), nc) if nr < 1_000_000 else (rng.random(nr) < 0.01).astype(np.int64)
    deg[rng.choice(nr, size=len(lens), replace=False)] = lens
    row = np.repeat(np.arange(nr), deg)
    col = np.concatenate([rng.choice(min(nc, 4000) if name == "crowded columns" else nc, size=d, replace=False) for d in deg if d]
                         or [np.zeros(0, np.int64)])
    return row, col, (nr, nc)


@pytest.mark.parametrize("twice", ["none", "some", "many"])
@pytest.mark.parametrize("name", ["n=1", "n=63", "n=4095", "n=4096", "n=4097", "n=130000", "giant rows", "a row past the limit", "crowded columns",
                                  "one column", "one row", "few entries", "wide keys", "long bins", "adjacent long rows", "whole windows", "rows by length",
                                  "a bin of the most", "a bin past the limit", "a crowded long row"])
def test_triplets_through_bins_of_rows(fa, name, twice):
    """Every way an entry can take: bins sorted by buckets or bitonically, large bins in windows, rows that are sorted a
    range of columns at a time, bins past the limits, shapes that are left to the library's sort; without
    duplicates (the values' bits are kept, not only numbers), with some and with 300 of one entry."""
    import scipy.sparse as sp
    from liteform_ae_amd.format_matrix_market import MTX
    row, col, shape = coo_case(name)
    rng = np.random.default_rng(len(row))
    if twice != "none":
        again = rng.integers(0, len(row), size=max(1, len(row) // 10))
        if twice == "many":
            again = np.concatenate([again, np.full(300, rng.integers(0, len(row)))])
        row, col = np.concatenate([row, row[again]]), np.concatenate([col, col[again]])
    order = rng.permutation(len(row))
    row, col = row[order].astype(np.int32), col[order].astype(np.int32)
    val = rng.uniform(-1, 1, size=len(row)).astype(np.float32)
    if twice == "none":
        val[:4] = np.array([np.inf, -0.0, np.nan, 1e-42], dtype=np.float32)[:len(val)]
    dev = fa._DeviceCSR(MTX.from_coo(row, col, shape, data=val))
    want = sp.coo_matrix((val.astype(np.float64), (row, col)), shape=shape).tocsr()
    want.sort_indices()
    assert dev.nnz == want.nnz
    np.testing.assert_array_equal(dev.indptr.cpu().numpy(), want.indptr)
    np.testing.assert_array_equal(dev.indices.cpu().numpy(), want.indices)
    got = dev.values.cpu().numpy()
    if twice == "none":
        np.testing.assert_array_equal(got.view(np.int32), want.data.astype(np.float32).view(np.int32))
    else:
        # the shapes of the library's sort: float32 sums in some order, a rounding of at most the sum of the magnitudes
        # for each addition; the others: sums in 64 bits, rounded once
        of_size = sp.coo_matrix((np.abs(val).astype(np.float64), (row, col)), shape=shape).tocsr()
        times = sp.coo_matrix((np.ones(len(val)), (row, col)), shape=shape).tocsr()
        of_size.sort_indices()
        times.sort_indices()
        in_float = name in ("few entries", "wide keys", "a bin of the most", "a bin past the limit", "a crowded long row")      # (most: and duplicates)
        bound = (times.data - 1) * 2.0 ** -24 * of_size.data if in_float else 2.0 ** -24 * np.abs(want.data) + 2.0 ** -52 * times.data * of_size.data
        assert (np.abs(got - want.data) <= bound).all()
    again = fa._DeviceCSR(MTX.from_coo(row, col, shape, data=val))
    assert np.array_equal(again.values.cpu().numpy().view(np.int32), got.view(np.int32))        # run to run the same bits


@pytest.mark.parametrize("name", ["n=4097", "giant rows", "a row past the limit", "crowded columns", "long bins", "few entries", "whole windows"])
def test_triplets_in_place(fa, name):
    """The results in the triplets' own arrays: the same as in others, also where the bins cannot take the matrix."""
    import ctypes as C
    import torch
    from liteform_ae_amd import _lib
    row, col, shape = coo_case(name)
    rng = np.random.default_rng(3)
    again = rng.integers(0, len(row), size=len(row) // 10)
    row, col = np.concatenate([row, row[again]]).astype(np.int32), np.concatenate([col, col[again]]).astype(np.int32)
    val = rng.integers(-1000, 1000, size=len(row)).astype(np.float32)           # (sums that are exact in any order)
    lib, n = _lib.load(), len(row)
    nbytes = lib.lf_coo_to_csr_workspace_bytes(n, *shape)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    results = []
    for in_place in (False, True):
        r, c, v = (torch.from_numpy(x).cuda() for x in (row, col, val))
        indptr = torch.empty(shape[0] + 1, dtype=torch.int32, device="cuda")
        indices, values = (c, v) if in_place else (torch.empty_like(c), torch.empty_like(v))
        left = C.c_int64(0)
        _lib.check(lib.lf_coo_to_csr(_lib.ptr(r), _lib.ptr(c), _lib.ptr(v), n, *shape, _lib.ptr(ws), nbytes, _lib.ptr(indptr),
                                     _lib.ptr(indices), _lib.ptr(values), C.byref(left), None))
        results.append([x.cpu().numpy() for x in (indptr, indices[:left.value], values[:left.value])])
    for x, y in zip(*results):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("times", [2, 3, 17, 18, 27, 64, 81, 300, 4000, 8000])
def test_sums_of_triplets_of_one_place(fa, times):
    """Sums of 2 to 8000 triplets are at most one rounding off, in whatever order they come: the entries of
    several places, beside each other and with the last one of the matrix among them."""
    from liteform_ae_amd.format_matrix_market import MTX
    rng = np.random.default_rng(times)
    rows, cols = 400, 300
    places = np.unique(np.concatenate([rng.choice(rows * cols, size=max(1, 8000 // times), replace=False), [rows * cols - 1]]))
    once = np.setdiff1d(rng.choice(rows * cols, size=900, replace=False), places)
    key = np.concatenate([np.repeat(places, times), once])
    val = rng.uniform(-1, 1, size=len(key)).astype(np.float32)
    order = rng.permutation(len(key))
    dev = fa._DeviceCSR(MTX.from_coo((key // cols)[order].astype(np.int32), (key % cols)[order].astype(np.int32), (rows, cols), data=val[order]))
    assert dev.nnz == len(places) + len(once)
    got = dev.values.cpu().numpy().astype(np.float64)
    at = np.searchsorted(np.sort(np.concatenate([places, once])), places)
    sums = val[:len(places) * times].astype(np.float64).reshape(len(places), times)
    want, of_size = sums.sum(1), np.abs(sums).sum(1)
    # rounded once to 24 bits; either sum of `times` values in 53 bits
    assert (np.abs(got[at] - want) <= 2.0 ** -24 * np.abs(want) + 2.0 ** -52 * times * of_size).all()


def test_canonical_csr_input_goes_in_as_it_is(fa):
    """A container made from canonical CSR arrays is uploaded and checked (lf_csr_check), not
    converted to COO and sorted: same device arrays, statistics and slabs as the COO route."""
    import scipy.sparse as sp
    from liteform_ae_amd.format_matrix_market import MTX
    rng = np.random.default_rng(19)
    for (nr, nc, deg, weighted) in ((1, 1, 1, False), (700, 900, 9, True), (3000, 40, 5, False), (40, 30000, 200, True)):
        src = skewed_matrix(rng, nr, nc, mean_deg=deg, heavy_rows=1, values=weighted)
        indptr, indices, data = src.adj_tensors("csr")
        g = MTX.from_csr(indptr, indices, (nr, nc), data=data if weighted else None)
        assert g._coo is None                                   # no COO view was built
        dev = fa._DeviceCSR(g)
        assert dev.path == "csr" and g._coo is None
        ref = fa._DeviceCSR(MTX.from_coo(src.coo_mtx.row, src.coo_mtx.col, (nr, nc), data=data if weighted else None))
        assert ref.path == "coo"
        assert dev.nnz == ref.nnz == dev.coo_nnz and dev.all_ones == ref.all_ones == (not weighted)
        np.testing.assert_array_equal(dev.indptr.cpu().numpy(), ref.indptr.cpu().numpy())
        np.testing.assert_array_equal(dev.indices.cpu().numpy(), ref.indices.cpu().numpy())
        np.testing.assert_array_equal(dev.values.cpu().numpy(), ref.values.cpu().numpy())
        if nr > 1:
            widths = [[1, 4, 16]] * 2
            assert_hyb_equal(fa.build_hyb_format(g, widths), O.build_hyb_format_sequential(src, widths))
            np.testing.assert_array_equal(fa.bucket_statistics(g, 2)[0], stats_from_oracle(src, 2)[0])
    # float32 ones given as data are recognised on the GPU
    g = MTX.from_csr(indptr, indices, (nr, nc), data=np.ones(len(indices), dtype=np.float32))
    assert fa._DeviceCSR(g).all_ones
    # an empty matrix
    dev = fa._DeviceCSR(MTX.from_csr(np.zeros(8, np.int32), np.zeros(0, np.int32), (7, 9)))
    assert dev.path == "csr" and dev.nnz == 0


def test_csr_input_that_is_not_canonical_takes_the_sort(fa):
    """Unsorted columns or duplicates inside a row: the check says so and the arrays go the
    COO route, ending as scipy's tocsr() has them (format_matrix_market.py:74-76).  Arrays that
    are no CSR structure at all are refused."""
    import scipy.sparse as sp
    from liteform_ae_amd.format_matrix_market import MTX
    rng = np.random.default_rng(23)
    nr, nc = 400, 300
    deg = rng.integers(0, 12, size=nr)
    indptr = np.concatenate(([0], np.cumsum(deg))).astype(np.int32)
    for kind in ("unsorted", "duplicates"):
        if kind == "unsorted":
            indices = np.concatenate([rng.permutation(nc)[:d] for d in deg]).astype(np.int32)
        else:
            indices = np.concatenate([np.sort(rng.integers(0, 6, size=d)) for d in deg]).astype(np.int32)
        data = rng.uniform(-1, 1, size=len(indices)).astype(np.float32)
        g = MTX.from_csr(indptr, indices, (nr, nc), data=data)
        dev = fa._DeviceCSR(g)
        assert dev.path == "coo"
        want = sp.csr_matrix((data, indices, indptr), shape=(nr, nc)).tocoo().tocsr()
        want.sum_duplicates()
        assert dev.nnz == want.nnz and dev.coo_nnz == len(indices)
        np.testing.assert_array_equal(dev.indptr.cpu().numpy(), want.indptr)
        np.testing.assert_array_equal(dev.indices.cpu().numpy(), want.indices)
        np.testing.assert_allclose(dev.values.cpu().numpy(), want.data, rtol=1e-5, atol=1e-6)
        widths = [[2, 8]]
        assert_hyb_equal(fa.build_hyb_format(g, widths), O.build_hyb_format_sequential(g, widths))
    bad = np.sort(rng.integers(0, nc, size=int(indptr[-1]))).astype(np.int32)
    bad[5] = nc                                                    # a column outside the matrix
    m = MTX(None)
    m._csr_source = sp.csr_matrix((nr, nc), dtype=np.float32)      # placeholder, arrays replaced below
    m._csr_source.indptr, m._csr_source.indices = indptr, bad
    m._csr_source.data = np.ones(len(bad), dtype=np.float32)
    with pytest.raises(ValueError, match="outside"):
        fa._DeviceCSR(m)
