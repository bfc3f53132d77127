"""Edge cases through the reference-shaped API on the GPU: empty and degenerate shapes,
many partitions, HIP-graph replay of the fused kernel."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from liteform_ae_amd.format_matrix_market import MTX
from oracle import liteform_oracle as O

from helpers import assert_hyb_equal, mtx_from_rows, skewed_matrix

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fa():
    from liteform_ae_amd import format_algos
    return format_algos


@pytest.fixture(scope="module")
def torch():
    import torch
    return torch


def product(fa, torch, g, cfg, feat=32, seed=0):
    rng = np.random.default_rng(seed)
    B = rng.uniform(-1, 1, size=(g.num_dst_nodes(), feat)).astype(np.float32)
    C = fa.spmm_hyb(fa.build_hyb_format_device(g, cfg), torch.from_numpy(B).cuda()).cpu().numpy()
    indptr, indices, data = g.adj_tensors("csr")
    ref = O.spmm_csr_f64(indptr, indices, data, g.coo_mtx.shape, B)
    bound = O.spmm_abs_bound(indptr, indices, data, g.coo_mtx.shape, B)
    assert C.shape == ref.shape
    assert (np.abs(C - ref) <= 1e-5 * bound).all()
    return C


def test_matrix_without_nonzeros(fa, torch):
    g = MTX.from_coo(np.zeros(0, dtype=np.int64), np.zeros(0, dtype=np.int64), (17, 9))
    cfg = fa.search_bucket_config(g, 2, fa.CostModelSettings(32, 2))
    assert cfg == [[], []] == O.search_bucket_config(g, 2, O.OracleCostModelSettings(32, 2))
    assert_hyb_equal(fa.build_hyb_format(g, cfg), O.build_hyb_format_sequential(g, cfg))
    C = product(fa, torch, g, cfg)
    assert (C == 0).all()


def test_single_entry_and_single_column(fa, torch):
    g = mtx_from_rows([[0, 0][:1], [0]], (2, 1))           # two rows, one column
    cfg = fa.search_bucket_config(g, 1, fa.CostModelSettings(32, 1))
    assert cfg == O.search_bucket_config(g, 1, O.OracleCostModelSettings(32, 1))
    assert_hyb_equal(fa.build_hyb_format(g, cfg), O.build_hyb_format_sequential(g, cfg))
    product(fa, torch, g, cfg)
    g = mtx_from_rows([[2]], (1, 5))                       # a single nonzero: the search refuses it
    with pytest.raises(ValueError):
        fa.search_bucket_config(g, 1, fa.CostModelSettings(32, 1))
    product(fa, torch, g, [[1]])                           # but a given config still works


def test_rectangular_both_ways(fa, torch):
    rng = np.random.default_rng(3)
    for shape in ((50, 4000), (4000, 50)):
        g = skewed_matrix(rng, shape[0], shape[1], mean_deg=4, heavy_rows=1, heavy_len=shape[1])
        for parts in (1, 3):
            try:
                want = O.search_bucket_config(g, parts, O.OracleCostModelSettings(64, parts))
            except ValueError:
                continue
            cfg = fa.search_bucket_config(g, parts, fa.CostModelSettings(64, parts))
            assert cfg == want
            assert_hyb_equal(fa.build_hyb_format(g, cfg), O.build_hyb_format_closed_form(g, cfg))
            product(fa, torch, g, cfg, feat=64)


def test_many_partitions(fa, torch):
    rng = np.random.default_rng(8)
    g = skewed_matrix(rng, 2000, 3000, mean_deg=30, heavy_rows=3, heavy_len=5000, values=True)
    for parts in (16, 37, 64):
        try:
            want = O.search_bucket_config(g, parts, O.OracleCostModelSettings(128, parts))
        except ValueError:
            with pytest.raises(ValueError):
                fa.search_bucket_config(g, parts, fa.CostModelSettings(128, parts))
            want = [[1, 4, 16, 64]] * parts
        else:
            assert fa.search_bucket_config(g, parts, fa.CostModelSettings(128, parts)) == want
        assert_hyb_equal(fa.build_hyb_format(g, want), O.build_hyb_format_closed_form(g, want))
        product(fa, torch, g, want, feat=128)


def test_more_partitions_than_columns(fa, torch):
    g = mtx_from_rows([[0, 1, 2], [1, 2], [0, 2], [0, 1]], (4, 3))
    widths = [[1, 2]] * 5                                  # partition size ceil(3/5) = 1; two empty partitions
    assert_hyb_equal(fa.build_hyb_format(g, widths), O.build_hyb_format_sequential(g, widths))
    product(fa, torch, g, widths)


def test_graph_replay_matches_eager(fa, torch):
    """The run entry point only launches kernels, so it can be captured in a HIP graph.
    Replays are interleaved with eager work and every replay is compared with the eager result."""
    rng = np.random.default_rng(12)
    g = skewed_matrix(rng, 6000, 20000, mean_deg=9, heavy_rows=3, heavy_len=60000)
    for parts in (1, 3):
        cfg = fa.search_bucket_config(g, parts, fa.CostModelSettings(128, parts, cost_model="gfx950"))
        fmt = fa.build_hyb_format_device(g, cfg)
        plan = fa.HybSpMM(fmt, 128)
        assert plan.info["heavy_rows"] >= 1, (cfg, plan.info, fmt.ell_rows)   # the partial-row kernel is in the graph
        B = torch.rand((20000, 128), device="cuda") - 0.5
        out = torch.empty((6000, 128), device="cuda")
        eager = plan.run(B).clone()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            plan.run(B, out)                            # warm-up on the capture stream
            side.synchronize()
            with torch.cuda.graph(graph, stream=side):
                plan.run(B, out)
        torch.cuda.current_stream().wait_stream(side)
        for i in range(4):
            out.fill_(float("nan"))
            junk = (torch.rand((512, 512), device="cuda") @ torch.rand((512, 512), device="cuda")).sum()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager), f"replay {i} differs"
            assert torch.isfinite(junk)
        # new operand values through the same graph
        B.mul_(2.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, plan.run(B))
        plan.close()


def test_runs_of_one_plan_on_several_streams(fa, torch):
    """The runs of a plan share its partial rows and counters: on several streams, with operands of
    their own, each gives what it gives alone - also behind a run that was recorded into a graph."""
    rng = np.random.default_rng(31)
    g = skewed_matrix(rng, 3000, 30000, mean_deg=6, heavy_rows=40, heavy_len=9000)
    plan = fa.HybSpMM(fa.build_hyb_format_device(g, [[1, 4, 16, 64]]), 64)
    assert plan.info["heavy_rows"] >= 30
    streams = [torch.cuda.current_stream()] + [torch.cuda.Stream() for _ in range(3)]
    Bs = [torch.rand((30000, 64), device="cuda") - 0.5 for _ in streams]
    alone = [plan.run(B).clone() for B in Bs]
    outs = [[torch.full_like(alone[0], float("nan")) for _ in range(12)] for _ in streams]
    graph, in_graph = torch.cuda.CUDAGraph(), torch.full_like(alone[0], float("nan"))
    torch.cuda.synchronize()
    for i in range(12):
        for stream, B, out in zip(streams, Bs, outs):
            with torch.cuda.stream(stream):
                plan.run(B, out[i])
        if i == 5:
            torch.cuda.synchronize()
            with torch.cuda.graph(graph):
                plan.run(Bs[1], in_graph)
    torch.cuda.synchronize()
    for ref, out in zip(alone, outs):
        assert all(torch.equal(ref, x) for x in out)
    for _ in range(3):
        in_graph.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(in_graph, alone[1])


def test_runs_of_one_plan_from_several_threads(fa, torch):
    """The same with a thread to each stream: what a run waits for has been launched, not just begun."""
    rng = np.random.default_rng(32)
    g = skewed_matrix(rng, 3000, 30000, mean_deg=6, heavy_rows=40, heavy_len=9000)
    plan = fa.HybSpMM(fa.build_hyb_format_device(g, [[1, 4, 16, 64]]), 64)
    assert plan.info["heavy_rows"] >= 30
    streams = [torch.cuda.Stream() for _ in range(4)]
    Bs = [torch.rand((30000, 64), device="cuda") - 0.5 for _ in streams]
    alone = [plan.run(B).clone() for B in Bs]
    outs = [[torch.full_like(alone[0], float("nan")) for _ in range(12)] for _ in streams]
    torch.cuda.synchronize()

    def runs(stream, B, out):
        with torch.cuda.stream(stream):
            for C in out:
                plan.run(B, C)

    with ThreadPoolExecutor(len(streams)) as pool:
        list(pool.map(runs, streams, Bs, outs))
    torch.cuda.synchronize()
    for ref, out in zip(alone, outs):
        assert all(torch.equal(ref, x) for x in out)


def test_matrix_features_on_device(fa, torch):
    """Integer fields exact, float fields to 1e-9 relative against the host routine
    (numpy's two-pass standard deviation against sqrt(E[d^2] - E[d]^2) on exact sums)."""
    rng = np.random.default_rng(11)
    g = skewed_matrix(rng, 5000, 3000, mean_deg=7.0, heavy_rows=3, heavy_len=2500)
    # duplicated COO entries: "nnz" counts stored entries, row lengths come from the CSR
    row = np.concatenate([g.coo_mtx.row, g.coo_mtx.row[:100]])
    col = np.concatenate([g.coo_mtx.col, g.coo_mtx.col[:100]])
    for m in (g, MTX.from_coo(row, col, g.coo_mtx.shape), mtx_from_rows([[], [1], []], (3, 4))):
        want = m.matrix_features()
        got = fa.matrix_features_device(m)
        assert list(got) == list(want)
        for key in ("name", "num_rows", "num_cols", "nnz", "min_nnz_per_row", "max_nnz_per_row"):
            assert got[key] == want[key], key
        for key in want:
            if key.startswith(("avg", "std", "min_nnz_density", "max_nnz_density")):
                assert got[key] == pytest.approx(want[key], rel=1e-9, abs=1e-15), key


@pytest.mark.parametrize("n", [1, 524_287, 524_288, 524_289, 7 * 524_288 + 5, 16_777_216 + 3])
def test_staged_transfers_round_trip(fa, n):
    """One piece, whole pieces, a remainder, more pieces than buffers, the large buffers."""
    import torch
    ints = np.arange(n, dtype=np.int64) - n // 2
    reals = np.linspace(-1.0, 1.0, n)
    up = fa._upload(ints, np.int32), fa._upload(reals, np.float32), fa._upload(ints.astype(np.int16), np.int32)
    assert [t.dtype for t in up] == [torch.int32, torch.float32, torch.int32]
    with fa._Downloads([(up[0], torch.int64), (up[1], torch.float32), (up[2], torch.int64)]) as down:
        back = [down.get(i).numpy() for i in range(3)]
    np.testing.assert_array_equal(back[0], ints)
    np.testing.assert_array_equal(back[1], reals.astype(np.float32))
    np.testing.assert_array_equal(back[2], ints.astype(np.int16))


@pytest.mark.parametrize("nr,feat,b_dtype", [
    *((nr, feat, b) for nr in (1, 31, 33, 65) for feat, b in ((32, "f32"), (64, "f32"), (96, "f32"), (128, "f32"), (256, "f32"),
                                                              (512, "f32"), (1024, "f32"), (64, "bf16"), (320, "bf16"), (1024, "bf16"))),
    (524_288, 64, "f32"), (524_289, 64, "f32"),          # many groups
])
def test_csr_product_at_group_edges(fa, torch, nr, feat, b_dtype):
    """Rows that end a group of 32 or 64, empty rows at both ends and in a row, rows at and past the
    length that a whole workgroup sums."""
    import scipy.sparse as sp
    rng = np.random.default_rng(nr + feat)
    nc = 700
    deg = rng.integers(0, 12, size=nr)
    deg[rng.random(nr) < 0.3] = 0
    deg[(7 * np.arange(5) + nr // 2) % nr] = (128, 129, 700, 127, 300)
    deg[-1] = 0 if nr > 1 else 129
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    row = np.repeat(np.arange(nr), deg)
    key = np.sort(row * nc + (row * 13 + 31 * (np.arange(len(row)) - indptr[row])) % nc)      # 31 and 700 share no factor
    vals = rng.uniform(-1, 1, size=len(key)).astype(np.float32)
    A = sp.csr_matrix((vals.astype(np.float64), key % nc, indptr), shape=(nr, nc))
    B = torch.from_numpy(rng.uniform(-1, 1, size=(nc, feat)).astype(np.float32)).cuda().to(torch.bfloat16 if b_dtype == "bf16" else torch.float32)
    got = fa.spmm_csr(MTX.from_csr(indptr, (key % nc).astype(np.int32), (nr, nc), data=vals), B, b_dtype).cpu().numpy()
    Bh = B.float().cpu().numpy().astype(np.float64)
    assert (np.abs(got - A @ Bh) <= 1e-5 * (abs(A) @ np.abs(Bh)) + 1e-30).all()


@pytest.mark.parametrize("nr,feat,b_dtype,usual,longest", [
    *((nr, feat, b, *rows) for nr in (3, 4, 5, 9, 16, 17, 32, 63)
      for feat, b in ((32, "f32"), (64, "f32"), (224, "f32"), (448, "f32"), (1024, "f32"), (128, "bf16"), (512, "bf16"), (1024, "bf16"))
      for rows in ((0, 128), (0, 129), (80, 270), (80, 299))),
    *((nr, feat, "f32", 0, longest) for longest in (32, 33, 128, 129) for nr, feat in (
        (4096, 224), (4097, 224),                            # the most rows in groups of 16, the fewest in groups of 32
        (1 << 20, 32), ((1 << 20) + 1, 32))),                # ... in groups of as many as sub-waves, in groups of 64
])
def test_csr_product_of_short_rows(fa, torch, nr, feat, b_dtype, usual, longest):
    """Groups whose longest row has 128 entries (32 where a sub-wave has two rows) or three average rows,
    summed a row to a sub-wave, and groups with more than that, cut into runs; rows of every remainder of a
    batch of eight gathers; infinite rows of B give Inf, not NaN."""
    import scipy.sparse as sp
    rng = np.random.default_rng(nr + feat)
    nc = 300
    deg = usual + np.arange(nr) * 5 % 34
    deg[nr // 2] = longest
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    row = np.repeat(np.arange(nr), deg)
    key = np.sort(row * nc + (row * 13 + 31 * (np.arange(len(row)) - indptr[row])) % nc)      # 31 and 300 share no factor
    vals = rng.uniform(0.25, 1, size=len(key)).astype(np.float32)
    A = sp.csr_matrix((vals.astype(np.float64), key % nc, indptr), shape=(nr, nc))
    B = torch.from_numpy(rng.uniform(-1, 1, size=(nc, feat)).astype(np.float32)).cuda().to(torch.bfloat16 if b_dtype == "bf16" else torch.float32)
    g = MTX.from_csr(indptr, (key % nc).astype(np.int32), (nr, nc), data=vals)
    finite = B.float().cpu().numpy().astype(np.float64)
    want, bound = A @ finite, 1e-5 * (abs(A) @ np.abs(finite)) + 1e-30
    assert (np.abs(fa.spmm_csr(g, B, b_dtype).cpu().numpy() - want) <= bound).all()
    for col in (0, 31, 93):
        Binf = B.clone()
        Binf[col] = float("inf")
        got = fa.spmm_csr(g, Binf, b_dtype).cpu().numpy()
        hit = np.diff(A[:, [col]].indptr) > 0
        assert np.isposinf(got[hit]).all()
        assert (np.abs(got[~hit] - want[~hit]) <= bound[~hit]).all()


@pytest.mark.parametrize("nr,nc,feat,b_dtype", [
    *((nr, 3000, feat, b) for nr in (1, 7, 9, 300) for feat, b in ((32, "f32"), (64, "f32"), (96, "f32"), (128, "f32"), (256, "f32"),
                                                                   (512, "f32"), (1024, "f32"), (128, "bf16"), (256, "bf16"), (512, "bf16"))),
    *((nr, 9001, feat, b) for nr in (7, 300) for feat, b in ((160, "f32"), (224, "f32"), (288, "f32"), (352, "f32"), (448, "bf16"))),
    (24_575, 3000, 32, "f32"), (24_576, 3000, 64, "f32"), (24_577, 3000, 256, "f32"),          # the two group sizes
    (300, 1_060_000, 1024, "f32"),                           # 4.3 GB of B: past what 32-bit offsets reach
    (40, 2_200_000, 992, "bf16"),
])
def test_csr_product_of_uneven_rows(fa, torch, nr, nc, feat, b_dtype):
    """Long rows between short ones (a wavefront's teams hold rows of both kinds), rows of every remainder of a
    batch, first and last column, features split over the XCDs (small matrices and whole multiples of 128 bytes
    are), with and without values; twice the same bits."""
    import scipy.sparse as sp
    rng = np.random.default_rng(nr + feat)
    deg = np.arange(nr) * 7 % 19
    deg[nr // 3::11] = 33
    deg[(np.arange(6) * 3 + nr // 2) % nr] = (257, 300, 1025, 0, 2999, 256)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(nc, size=n, replace=False)) if n > 40 else np.sort((rng.integers(nc) + 61 * np.arange(n)) % nc)
                          for n in deg]).astype(np.int32)
    if deg[-1]:
        col[-1] = nc - 1
    if deg[0]:
        col[0] = 0
    vals = rng.uniform(-1, 1, size=len(col)).astype(np.float32)
    gen = torch.Generator(device="cuda").manual_seed(nr)
    B = torch.rand((nc, feat), device="cuda", generator=gen, dtype=torch.float32 if b_dtype == "f32" else torch.bfloat16)
    used, at = np.unique(col, return_inverse=True)
    Bh = B[torch.from_numpy(used.astype(np.int64)).cuda()].float().cpu().numpy().astype(np.float64)
    g = MTX.from_csr(indptr, col, (nr, nc), data=vals)
    for use_values in (True, False):
        A = sp.csr_matrix((vals.astype(np.float64) if use_values else np.ones(len(col)), at, indptr), shape=(nr, len(used)))
        got = fa.spmm_csr(g, B, b_dtype, use_values=use_values)
        assert torch.equal(got, fa.spmm_csr(g, B, b_dtype, use_values=use_values))
        assert (np.abs(got.cpu().numpy() - A @ Bh) <= 1e-5 * (abs(A) @ np.abs(Bh)) + 1e-30).all()


@pytest.mark.parametrize("feat,b_dtype", [(32, "f32"), (128, "f32"), (320, "f32"), (1024, "f32"), (64, "bf16"), (512, "bf16")])
def test_rows_of_several_chunks(fa, torch, monkeypatch, feat, b_dtype):
    """Long rows of one chunk, a few, the most that the last chunk's workgroup adds up and one more;
    several runs of one plan, which has to reset its counters, give the same bits."""
    monkeypatch.setenv("LF_DENSE_ROWS", "0")          # (dense rows would be cut differently where B is large)
    rng = np.random.default_rng(feat)
    nc = 140_000
    lens = [257, 1024, 1025, 2048, 2049, 3 * 1024, 64 * 1024, 64 * 1024 + 1]          # chunks of 1024 at this size
    row = np.repeat(np.arange(len(lens)), lens)
    col = np.concatenate([np.sort(rng.choice(nc, size=n, replace=False)) for n in lens])
    g = MTX.from_coo(row, col, (len(lens), nc), data=rng.uniform(-1, 1, size=len(row)).astype(np.float32))
    B = torch.from_numpy(rng.uniform(-1, 1, size=(nc, feat)).astype(np.float32)).cuda()
    if b_dtype == "bf16":
        B = B.to(torch.bfloat16)
    plan = fa.HybSpMM(fa.build_hyb_format_device(g, [[64, 1024]]), feat, b_dtype)
    assert plan.info["heavy_rows"] == 6 and plan.info["partial_rows"] == 2 + 2 + 3 + 3 + 64 + 65
    runs = [plan.run(B).clone() for _ in range(4)]
    assert all(torch.equal(r, runs[0]) for r in runs)
    indptr, indices, data = g.adj_tensors("csr")
    Bh = B.float().cpu().numpy()
    ref = O.spmm_csr_f64(indptr, indices, data, (len(lens), nc), Bh)
    assert (np.abs(runs[0].cpu().numpy() - ref) <= 1e-5 * O.spmm_abs_bound(indptr, indices, data, (len(lens), nc), Bh)).all()


@pytest.mark.parametrize("feat,b_dtype", [(32, "f32"), (256, "f32"), (512, "f32"), (128, "bf16")])
@pytest.mark.parametrize("n_long", [0, 1024, 1025, 3000])
def test_rows_around_the_cooperative_length(fa, torch, feat, b_dtype, n_long):
    """Whole workgroups take rows of more than 64, 128 or 256 slots, by how many rows there are of
    more than 64 and of more than 128: rows on either side of every length, at every choice."""
    rng = np.random.default_rng(n_long + feat)
    nc = 900
    lens = np.concatenate([[1, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513],
                           rng.integers(65, 129, size=n_long), rng.integers(129, 257, size=n_long // 2)]).astype(np.int64)
    if n_long == 0:
        lens = lens[:4]
    row = np.repeat(np.arange(len(lens)), lens)
    pos = np.arange(len(row)) - np.repeat(np.cumsum(lens) - lens, lens)
    g = MTX.from_coo(row, (row * 17 + pos * 7) % nc, (len(lens), nc), data=rng.uniform(-1, 1, size=len(row)).astype(np.float32))
    B = torch.from_numpy(rng.uniform(-1, 1, size=(nc, feat)).astype(np.float32)).cuda().to(torch.bfloat16 if b_dtype == "bf16" else torch.float32)
    got = fa.HybSpMM(fa.build_hyb_format_device(g, [[1, 64, 128, 256, 512]]), feat, b_dtype).run(B).cpu().numpy()
    indptr, indices, data = g.adj_tensors("csr")
    Bh = B.float().cpu().numpy()
    assert (np.abs(got - O.spmm_csr_f64(indptr, indices, data, (len(lens), nc), Bh))
            <= 1e-5 * O.spmm_abs_bound(indptr, indices, data, (len(lens), nc), Bh)).all()


@pytest.mark.parametrize("feat,b_dtype,lanes", [(32, "f32", 8), (128, "f32", 32), (512, "f32", 64), (128, "bf16", 16)])
@pytest.mark.parametrize("n_mid,n_long", [(0, 0), (700, 300), (3000, 0), (3000, 1500), (3000, 2500)])
def test_cooperative_length_of_a_folded_format(fa, torch, feat, b_dtype, lanes, n_mid, n_long):
    """Widest bucket of 32: a row of 65 to 256 entries is several narrow ELL rows, and it is the rows that
    count.  Where a matrix has many of them they are not given a workgroup each."""
    rng = np.random.default_rng(n_mid + n_long + feat)
    nc = 900
    lens = np.concatenate([[1, 2, 3, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129, 255, 256],
                           rng.integers(65, 129, size=n_mid), rng.integers(129, 257, size=n_long)]).astype(np.int64)
    row = np.repeat(np.arange(len(lens)), lens)
    pos = np.arange(len(row)) - np.repeat(np.cumsum(lens) - lens, lens)
    g = MTX.from_coo(row, (row * 17 + pos * 7) % nc, (len(lens), nc), data=rng.uniform(-1, 1, size=len(row)).astype(np.float32))
    B = torch.from_numpy(rng.uniform(-1, 1, size=(nc, feat)).astype(np.float32)).cuda().to(torch.bfloat16 if b_dtype == "bf16" else torch.float32)
    fmt = fa.build_hyb_format_device(g, [[1, 4, 32]])
    plan = fa.HybSpMM(fmt, feat, b_dtype)
    got = plan.run(B).cpu().numpy()
    indptr, indices, data = g.adj_tensors("csr")
    Bh = B.float().cpu().numpy()
    assert (np.abs(got - O.spmm_csr_f64(indptr, indices, data, (len(lens), nc), Bh))
            <= 1e-5 * O.spmm_abs_bound(indptr, indices, data, (len(lens), nc), Bh)).all()
    slots = -(-lens // 32) * 32
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    over64, over128 = int((slots > 64).sum()), int((slots > 128).sum())
    length = 64 if over64 <= 4 * cus else 128 if lanes <= 16 and over128 <= 8 * cus else 256
    chunks = int((slots > length).sum())                    # one each: none is longer than a chunk
    tiles = int(fmt.ell_rows.sum()) // 16 + 4 * cus + 40    # of ELL rows: 16 or more to a tile, or four tiles per CU
    assert chunks <= plan.info["tiles"] <= chunks + tiles, (length, chunks, plan.info)


@pytest.mark.parametrize("feat,b_dtype", [(32, "f32"), (64, "f32"), (96, "f32"), (288, "f32"), (64, "bf16"), (256, "bf16"), (512, "bf16")])
@pytest.mark.parametrize("parts,n_rows", [(1, 700), (2, 17), (3, 8192 + 5)])
def test_parts_of_b_that_the_l2_holds(fa, torch, feat, b_dtype, parts, n_rows):
    """The kernels of launches whose part of B stays in the L2: every staged width, tiles that are
    full and not, rows of several ELL rows, and rows that only some partitions add to."""
    rng = np.random.default_rng(feat + parts)
    nc = 600
    lens = rng.integers(0, 130, size=n_rows) >> rng.integers(0, 7, size=n_rows)
    row = np.repeat(np.arange(n_rows), lens)
    pos = np.arange(len(row)) - np.repeat(np.cumsum(lens) - lens, lens)
    g = MTX.from_coo(row, (row * 17 + pos * 7) % nc, (n_rows, nc), data=rng.uniform(-1, 1, size=len(row)).astype(np.float32))
    B = torch.from_numpy(rng.uniform(-1, 1, size=(nc, feat)).astype(np.float32)).cuda().to(torch.bfloat16 if b_dtype == "bf16" else torch.float32)
    fmt = fa.build_hyb_format_device(g, [[1, 2, 4, 8, 16, 32, 64]] * parts)
    got = fa.HybSpMM(fmt, feat, b_dtype).run(B).cpu().numpy()
    indptr, indices, data = g.adj_tensors("csr")
    Bh = B.float().cpu().numpy()
    assert (np.abs(got - O.spmm_csr_f64(indptr, indices, data, (n_rows, nc), Bh))
            <= 1e-5 * O.spmm_abs_bound(indptr, indices, data, (n_rows, nc), Bh)).all()


@pytest.mark.parametrize("parts,b_dtype", [(16, "f32"), (3, "bf16")])
def test_chunk_tables_of_many_buckets(fa, torch, parts, b_dtype):
    """Plans whose chunked rows lie in more buckets than one launch of the table's kernel takes, and in
    buckets of more ELL rows than one of its workgroups: widths of 8 split every row into many."""
    rng = np.random.default_rng(parts)
    nr, nc = 3000, 60_000
    lens = rng.integers(0, 40, size=nr)
    lens[::97] = rng.integers(2200 * parts, 2400 * parts, size=len(lens[::97]))
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    indices = np.concatenate([np.sort(rng.choice(nc, size=n, replace=False)) for n in lens]).astype(np.int32)
    vals = rng.uniform(-1, 1, size=len(indices)).astype(np.float32)
    g = MTX.from_csr(indptr, indices, (nr, nc), data=vals)
    B = torch.from_numpy(rng.uniform(-1, 1, size=(nc, 64)).astype(np.float32)).cuda()
    B = B.to(torch.bfloat16) if b_dtype == "bf16" else B
    Bh = B.float().cpu().numpy()
    ref = O.spmm_csr_f64(indptr, indices, vals, (nr, nc), Bh)
    bound = 1e-5 * O.spmm_abs_bound(indptr, indices, vals, (nr, nc), Bh)
    for widths in ([[1, 8, 1024]] * parts, [[8]] * parts, [[4, 512, 1024], [8]] + [[2, 1024]] * (parts - 2)):
        plan = fa.HybSpMM(fa.build_hyb_format_device(g, widths), 64, b_dtype)
        out = plan.run(B)
        assert plan.info["heavy_rows"] > 0 or widths[-1] == [2, 1024], widths      # (there chunks of 8192 slots)
        assert (np.abs(out.cpu().numpy() - ref) <= bound).all()
        plan.close()
