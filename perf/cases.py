"""The work that a user of this package has it do, as measurable cases.

``listed()`` names twelve cases over the range of the package: products with a composed hyb
format (the reference's CELL branch), the CSR and BSR products beside it, and the composition
itself, from a matrix on the GPU and from one on the host.  ``draw(rng)`` gives further cases of
the same ranges.  Matrices are synthetic: sizes and row-length laws are those of the package's
benchmark workloads (``liteform_ae_amd.synthetic``) and driver, neighbours are uniform.

Operations (``case["op"]``):
  spmm      C = A_hyb . B with a kept plan: what a graph layer or a solver calls every step
  csr       C = A_csr . B, the row-parallel product without a composed format
  bsr       Y = A_bsr . X, fp16 blocks on the matrix cores
  compose   width search, hyb composition and kernel plan for a matrix on the GPU: paid once per
            matrix and feature size
  host      width search and ``build_hyb_format`` with its numpy result, the reference's own call
  oneshot   COO triplets on the host to one finished product: everything a matrix that is used
            once pays for
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from liteform_ae_amd import format_algos as fa
from liteform_ae_amd.format_matrix_market import MTX

# ---------------------------------------------------------------------------- the cases


def listed():
    return [
        # a small matrix with few features: the cost of a call
        {"name": "spmm_4k_n32", "op": "spmm", "law": "poisson", "rows": 4096, "cols": 4096, "degree": 16.0,
         "feat": 32, "b": "f32"},
        # a citation graph: power-law rows, an operand somewhat larger than an L2
        {"name": "spmm_170k_n128", "op": "spmm", "law": "zipf", "rows": 170_000, "cols": 170_000, "degree": 13_000.0,
         "feat": 128, "b": "f32"},
        # the headline matrix: a graph whose dense operand is far larger than any cache
        {"name": "spmm_2450k_n128", "op": "spmm", "law": "lognormal", "rows": 2_450_000, "cols": 2_450_000,
         "degree": 33.0, "sigma": 1.1, "feat": 128, "b": "f32"},
        # a graph with hundreds of entries per row and an odd feature size
        {"name": "spmm_132k_dense_n96", "op": "spmm", "law": "lognormal", "rows": 132_000, "cols": 132_000,
         "degree": 300.0, "sigma": 0.6, "feat": 96, "b": "f32"},
        # a finite-element-like stencil: neighbouring rows share their columns
        {"name": "spmm_stencil_n256", "op": "spmm", "law": "stencil", "nx": 100, "ny": 100, "nz": 100, "points": 27,
         "feat": 256, "b": "f32"},
        # a rectangular matrix of short rows and a few dense ones, 16-bit operand
        {"name": "spmm_skewed_bf16_n512", "op": "spmm", "law": "pareto", "rows": 500_000, "cols": 2_000_000,
         "degree": 2.0, "dense_rows": 50, "dense_len": 100_000, "feat": 512, "b": "bf16"},
        # the CSR product on a protein-interaction-sized graph
        {"name": "csr_57k_n64", "op": "csr", "law": "lognormal", "rows": 57_000, "cols": 57_000, "degree": 28.0,
         "sigma": 0.9, "feat": 64, "b": "f32"},
        # the block-sparse product at the driver's block size
        {"name": "bsr32_1m_n128", "op": "bsr", "block": 32, "block_rows": 32_768, "block_cols": 32_768, "per_row": 8,
         "feat": 128},
        # ... and a small one with ragged features
        {"name": "bsr16_40k_n200", "op": "bsr", "block": 16, "block_rows": 2_501, "block_cols": 2_501, "per_row": 8,
         "feat": 200},
        # composition of the headline matrix
        {"name": "compose_2450k", "op": "compose", "law": "lognormal", "rows": 2_450_000, "cols": 2_450_000,
         "degree": 33.0, "sigma": 1.1, "feat": 128, "b": "f32"},
        # the reference's composition call, with host arrays out
        {"name": "host_57k", "op": "host", "law": "lognormal", "rows": 57_000, "cols": 57_000, "degree": 28.0,
         "sigma": 0.9, "feat": 128, "b": "f32"},
        # a matrix that arrives as triplets and is multiplied once
        {"name": "oneshot_170k_n64", "op": "oneshot", "law": "zipf", "rows": 170_000, "cols": 170_000,
         "degree": 13_000.0, "feat": 64, "b": "f32"},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _feat(rng, cols, entries, b):
    """A feature size from 32 to 512 for which operand and product stay within the listed ones."""
    step = 64 if b == "bf16" else 32
    most = min(512, int(1.25e9 / (cols * (2 if b == "bf16" else 4))), int(9e9 / max(entries, 1.0)))
    top = max(1, most // step)
    return step * max(1, min(top, round(_log(rng, 1, 512 // step))))


def draw(rng):
    op = rng.choice(("spmm", "spmm", "spmm", "csr", "bsr", "compose", "host", "oneshot"))
    if op == "bsr":
        block = rng.choice((16, 32, 64))
        block_rows = round(_log(rng, 2_000, 800_000) / block)
        return {"op": op, "block": block, "block_rows": block_rows,
                "block_cols": max(16, round(block_rows * _log(rng, 0.5, 1.2))), "per_row": rng.randint(2, 10),
                "feat": 8 * round(_log(rng, 2, 16))}
    b = "bf16" if op == "spmm" and rng.random() < 0.25 else "f32"
    if op == "spmm" and rng.random() < 0.3:
        nx, ny, nz = (round(_log(rng, 16, 100)) for _ in range(3))
        points = rng.choice((7, 27))
        return {"op": op, "law": "stencil", "nx": nx, "ny": ny, "nz": nz, "points": points,
                "feat": _feat(rng, nx * ny * nz, nx * ny * nz * points, b), "b": b}
    if op == "host":
        rows, degree = round(_log(rng, 2_000, 100_000)), _log(rng, 4, 30)
    elif op == "oneshot":
        rows, degree = round(_log(rng, 2_000, 200_000)), _log(rng, 3, 40)
    elif op == "compose":
        rows, degree = round(_log(rng, 4_000, 2_000_000)), _log(rng, 4, 35)
    else:
        rows = round(_log(rng, 2_000, 2_000_000))
        degree = _log(rng, 4, min(400.0, 4e7 / rows))
    cols = round(rows * _log(rng, 0.6, 2.0)) if op in ("spmm", "csr") else rows
    if op != "host" and rng.random() < 0.3:
        case = {"op": op, "law": "zipf", "rows": rows, "cols": cols, "degree": float(round(_log(rng, 200, 13_000)))}
    elif op == "spmm" and rng.random() < 0.2:
        dense = max(1, round(_log(rng, 1, 40)))
        case = {"op": op, "law": "pareto", "rows": rows, "cols": cols, "degree": 2.0, "dense_rows": dense,
                "dense_len": max(16, cols // 20)}
    else:
        case = {"op": op, "law": "lognormal", "rows": rows, "cols": cols, "degree": round(degree, 2),
                "sigma": round(rng.uniform(0.4, 1.1), 2)}
    case["b"] = b
    case["feat"] = _feat(rng, max(rows, cols), _expected_entries(case), b)
    return case


# ---------------------------------------------------------------------------- matrices


@functools.lru_cache(maxsize=64)
def _zipf_mean(cap):
    k = np.arange(1, cap + 1, dtype=np.float64)
    pmf = k ** -2.1
    head = float(pmf.sum())
    tail = (cap + 0.5) ** -1.1 / 1.1                  # rows above the cap are clipped to it
    return float((k * pmf).sum() + cap * tail) / (head + tail)


def _expected_entries(case):
    """Entries of the matrix a case describes (the law's mean)."""
    law = case["law"]
    if law == "stencil":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        if case["points"] == 7:
            n = nx * ny * nz
            return 7.0 * n - 2.0 * (ny * nz + nx * nz + nx * ny)
        return float((3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2))
    if law == "zipf":
        return case["rows"] * _zipf_mean(int(min(case["degree"], case["cols"])))
    if law == "pareto":
        return case["rows"] * 5.5 + case["dense_rows"] * case["dense_len"]
    return case["rows"] * min(case["degree"], case["cols"])


def _degrees(case, seed):
    """Row lengths: the same ones for every seed of a case (so that its format has the same
    shape), in another order."""
    rows, cols, law = case["rows"], case["cols"], case["law"]
    rng = np.random.default_rng(rows)
    if law == "poisson":
        deg = rng.poisson(case["degree"], size=rows)
    elif law == "zipf":
        deg = np.clip(rng.zipf(2.1, size=rows), 1, int(case["degree"]))
    elif law == "pareto":
        deg = np.floor(case["degree"] * (1.0 + rng.pareto(1.5, size=rows)))
        deg[rng.choice(rows, size=min(rows, case["dense_rows"]), replace=False)] = case["dense_len"]
    else:
        mu = math.log(case["degree"]) - 0.5 * case["sigma"] ** 2
        deg = np.clip(np.rint(rng.lognormal(mu, case["sigma"], size=rows)), 1, 17_000)
    return np.random.default_rng(seed).permutation(np.minimum(deg, cols).astype(np.int64))


def _stencil(case):
    """(rows, columns) of the 7- or 27-point stencil on an nx x ny x nz grid, row by row."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    d = torch.tensor([(dx, dy, dz) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)
                      if case["points"] == 27 or abs(dx) + abs(dy) + abs(dz) <= 1], device="cuda")
    i = torch.arange(nx * ny * nz, device="cuda")
    x, y, z = (i % nx)[:, None] + d[:, 0], (i // nx % ny)[:, None] + d[:, 1], (i // (nx * ny))[:, None] + d[:, 2]
    ok = (x >= 0) & (x < nx) & (y >= 0) & (y < ny) & (z >= 0) & (z < nz)
    return i[:, None].expand_as(x)[ok], (x + nx * (y + ny * z))[ok]


def _matrix(case, seed, gen):
    """Canonical CSR arrays on the GPU: (row of every entry, row pointer, columns, values, shape)."""
    if case["law"] == "stencil":
        rows = cols = case["nx"] * case["ny"] * case["nz"]
        row, col = _stencil(case)
    else:
        rows, cols = case["rows"], case["cols"]
        deg = torch.from_numpy(_degrees(case, seed)).cuda()
        row = torch.repeat_interleave(torch.arange(rows, device="cuda"), deg)
        # `deg` distinct columns of a row: ascending draws from the first cols - deg + 1, the i-th moved up by i
        draws = torch.rand(row.shape, device="cuda", generator=gen, dtype=torch.float64) * (cols - deg + 1)[row]
        key = (row * cols + draws.long()).sort().values
        col = key - row * cols + torch.arange(len(row), device="cuda") - (deg.cumsum(0) - deg)[row]
    indptr = torch.searchsorted(row, torch.arange(rows + 1, device="cuda")).to(torch.int32)
    values = torch.rand(len(col), device="cuda", generator=gen)
    if case["law"] in ("stencil", "pareto", "poisson"):
        values = 2.0 * values - 1.0
    return row.to(torch.int32), indptr, col.to(torch.int32), values, (rows, cols)


def _dense(rows, feat, dtype, gen):
    """The dense operand: U(-1, 1)."""
    return torch.rand((rows, feat), device="cuda", generator=gen).mul_(2.0).sub_(1.0).to(dtype)


# ---------------------------------------------------------------------------- measured calls


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    op, feat = case["op"], case["feat"]
    if op == "bsr":
        return _prepare_bsr(case, gen)
    row, indptr, col, values, shape = _matrix(case, seed, gen)
    state = {"case": case}
    if op == "oneshot":
        # a MatrixMarket file lists a matrix column by column
        order = torch.argsort(col, stable=True)
        state.update(row=row[order].cpu().numpy(), col=col[order].cpu().numpy(), data=values[order].cpu().numpy(), shape=shape)
        state["B"] = _dense(shape[1], feat, torch.float32, gen)
        return state
    data = None if op == "host" else values.cpu().numpy()      # the reference's matrices hold ones
    g = MTX.from_csr(indptr.cpu().numpy(), col.cpu().numpy(), shape, data=data)
    del row, indptr, col, values
    if op in ("csr", "compose", "host"):
        fa.matrix_features_device(g)                            # the matrix goes to the GPU
        state["g"] = g
        if op == "csr":
            state["B"] = _dense(shape[1], feat, torch.float32, gen)
        return state
    parts, windows = fa.predict_launch_shape(g, feat, case["b"])
    widths = fa.search_bucket_config(g, parts, fa.CostModelSettings(feat, parts, cost_model="gfx950"))
    state["plan"] = fa.HybSpMM(fa.build_hyb_format_device(g, widths), feat, case["b"], windows=windows)
    state["B"] = _dense(shape[1], feat, torch.bfloat16 if case["b"] == "bf16" else torch.float32, gen)
    return state


def _prepare_bsr(case, gen):
    block, mb, nb = case["block"], case["block_rows"], case["block_cols"]
    key = torch.arange(mb, device="cuda")[:, None] * nb + torch.randint(0, nb, (mb, case["per_row"]), device="cuda", generator=gen)
    key = torch.unique(key)
    bsr = fa._DeviceBSR.__new__(fa._DeviceBSR)                  # block arrays that are on the GPU already
    bsr.block_size, bsr.mb, bsr.nb, bsr.nnzb = block, mb, nb, len(key)
    bsr.indptr = torch.searchsorted(key // nb, torch.arange(mb + 1, device="cuda")).to(torch.int32)
    bsr.indices = (key % nb).to(torch.int32)
    bsr.data = _dense(len(key) * block, block, torch.float16, gen).reshape(-1)
    bsr.checked = False
    return {"case": case, "bsr": bsr, "x": _dense(nb * block, case["feat"], torch.float16, gen)}


def run(state):
    case = state["case"]
    op, feat = case["op"], case["feat"]
    if op == "spmm":
        return state["plan"].run(state["B"])
    if op == "csr":
        return fa.spmm_csr(state["g"], state["B"])
    if op == "bsr":
        return fa.spmm_bsr(state["bsr"], state["x"], case["block"])
    if op == "compose":
        g = state["g"]
        widths = fa.search_bucket_config(g, 1, fa.CostModelSettings(feat, 1))
        fmt = fa.build_hyb_format_device(g, widths)
        plan = fa.HybSpMM(fmt, feat, case["b"])
        plan.close()
        return widths, [fmt.slab(k)[:3] for k in range(fmt.num_buckets)]
    if op == "host":
        g = state["g"]
        return fa.build_hyb_format(g, fa.search_bucket_config(g, 1, fa.CostModelSettings(feat, 1)))
    g = MTX.from_coo(state["row"], state["col"], state["shape"], data=state["data"])
    parts = fa.guess_num_partitions(g, feat)
    widths = fa.search_bucket_config(g, parts, fa.CostModelSettings(feat, parts, cost_model="gfx950"))
    return fa.spmm_hyb(fa.build_hyb_format_device(g, widths), state["B"])


def work(case):
    """Every input read once and every output written once; 2 flops per entry and feature."""
    op, feat = case["op"], case["feat"]
    if op == "bsr":
        block, mb, nb = case["block"], case["block_rows"], case["block_cols"]
        blocks = mb * nb * -math.expm1(case["per_row"] * math.log1p(-1.0 / nb))
        return {"bytes": blocks * (2 * block * block + 4) + 4 * (mb + 1) + 2 * feat * block * (nb + mb),
                "flops": 2.0 * blocks * block * block * feat}
    entries = _expected_entries(case)
    rows = case["rows"] if "rows" in case else case["nx"] * case["ny"] * case["nz"]
    cols = case["cols"] if "cols" in case else rows
    matrix = 8 * entries + 4 * (rows + 1)
    product = cols * feat * (2 if case["b"] == "bf16" else 4) + rows * feat * 4
    if op == "compose":                                         # column and value of every entry, row ids
        return {"bytes": matrix + 8 * entries + 4 * rows, "flops": 0.0}
    if op == "host":                                            # 64-bit columns and mask on the host
        return {"bytes": matrix - 4 * entries + 16 * entries + 8 * rows, "flops": 0.0}
    if op == "oneshot":                                         # triplets in, product out
        return {"bytes": 12 * entries + product, "flops": 2.0 * entries * feat}
    return {"bytes": matrix + product, "flops": 2.0 * entries * feat}


def tolerance(case):
    if case["op"] in ("compose", "host"):
        return "exact"
    if case["op"] == "bsr":                                     # fp32 sums rounded to fp16
        return {"rel": 5e-4, "max": 2e-3}
    return {"rel": 1e-5, "max": 1e-4}                           # fp32 sums of exactly held operands
