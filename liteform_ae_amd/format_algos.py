"""CELL/hyb format selection, composition and SpMM on MI355X.

Same public names and call signatures as the reference module
``playground_pipline/format_algos.py`` (its ``__all__``, format_algos.py:26-31), so the
driver flow of ``proc05.spmm.end-to-end.py:153-176`` runs unchanged:

    cfg   = CostModelSettings(feat_size=N, num_parts=P)
    conf  = search_bucket_config(g, P, cfg)                 # List[P] of ascending widths
    hyb   = build_hyb_format(g, conf)                       # (rows, cols, mask) numpy lists
    ms    = bench_hyb_with_config(g, x, y, feat_size=N, bucket_widths=conf,
                                  bucketing_format=hyb, num_col_parts=P)

All computation happens in liblfhip.so (HIP, gfx950) reached through ctypes; torch-ROCm is
only used to hold device memory and to name the current stream.  There is no CPU path:
without the library or without a GPU these functions raise.

Additions that the reference does not have:
  * ``build_hyb_format_device`` keeps the composed format on the GPU (``HybFormat``) and
    carries A's real values; ``bench_hyb_with_config`` accepts it as ``bucketing_format``;
  * ``HybSpMM`` is the reusable kernel plan (run / time), ``spmm_hyb`` a one-shot product;
  * ``CostModelSettings(..., cost_model="gfx950")`` selects the MI355X traffic model.
"""
from __future__ import annotations

import ctypes as C
import os
import threading
import time
from typing import List, Sequence

import numpy as np

from . import _lib
from .format_matrix_market import MTX, Bucket  # noqa: F401  (re-exported like the reference)

__all__ = ["build_hyb_format", "bench_hyb_with_config", "search_bucket_config",
           "CostModelSettings", "bench_bsrmm", "bench_naive", "spmm_bsr",
           "build_hyb_format_device", "HybFormat", "HybSpMM", "spmm_hyb", "spmm_csr",
           "guess_num_partitions", "choose_num_partitions", "choose_launch_shape", "matrix_features_device",
           "predict_launch_shape", "model_spmm_ms", "row_overlap_device", "pick_launch_shape"]

WIDTH_LIMIT = 1024   # format_algos.py:821


class CostModelSettings:
    """format_algos.py:39-51.  ``cost_model`` is an extension: "reference" (default) or
    "gfx950"."""

    def __init__(self, feat_size: int, num_parts: int, cost_model: str = "reference"):
        self.feat_size = feat_size
        self.num_parts = num_parts
        self.cost_model = cost_model

    def __str__(self) -> str:
        return f"(feat_size={self.feat_size}, num_parts={self.num_parts})"


# --------------------------------------------------------------------------- device plumbing
_gpu_torch = None                # the torch module, once a GPU has been seen


def _torch():
    global _gpu_torch
    if _gpu_torch is None:
        import torch
        if not torch.cuda.is_available():
            raise RuntimeError("liteform_ae_amd needs a ROCm GPU (torch.cuda.is_available() is False); "
                               "there is no CPU fallback")
        torch.cuda.init()
        _gpu_torch = torch
    return _gpu_torch


def _stream():
    """hipStream_t of the current stream of the current device, as an integer."""
    cuda = _torch()._C
    return cuda._cuda_getCurrentRawStream(cuda._cuda_getDevice())


# Page-locked staging buffers: (bytes of one, how many), for arrays below and from _STAGE_LARGE on.
# Large arrays want large pieces (a 326 MB index array 48 GB/s, 27 as a plain copy from pageable
# memory); small ones want the first piece to leave early (three 3 MB arrays 360 us as plain
# copies).  The buffers belong to the process, one set per device, are made on first use and are shared
# under a lock.
_STAGE_LARGE = 64 << 20
_STAGE_SHAPES = {False: (2 << 20, 6), True: (16 << 20, 3)}
_stages = {}
_stage_lock = threading.Lock()
_long_rows_lock = threading.Lock()
_TORCH_TYPES = ("bool", "uint8", "int8", "int16", "int32", "int64", "float16", "float32", "float64")


def _staging(nbytes):
    """(buffers, their events, [the one used last]) for an array of that size on the current device."""
    torch = _torch()
    key = (nbytes >= _STAGE_LARGE, torch.cuda.current_device())      # an event belongs to a device
    if key not in _stages:
        stage_bytes, count = _STAGE_SHAPES[key[0]]
        _stages[key] = ([torch.empty(stage_bytes, dtype=torch.uint8, pin_memory=True) for _ in range(count)],
                        [torch.cuda.Event() for _ in range(count)], [0])
    return _stages[key]


def _upload(array, dtype):
    """A host array as a device tensor of `dtype` (int32 or float32), enqueued on the current stream.
    It goes through page-locked staging buffers: the copy into one runs on the host's threads, the
    conversion to `dtype` with it, while the piece before crosses PCIe."""
    torch = _torch()
    array = np.ascontiguousarray(array)
    if array.dtype.name not in _TORCH_TYPES or not array.dtype.isnative:
        array = np.ascontiguousarray(array, dtype=dtype)
    src = torch.from_numpy(array).reshape(-1)
    n = src.numel()
    out = torch.empty(n, dtype=torch.int32 if dtype is np.int32 else torch.float32, device="cuda")
    with _stage_lock:
        bufs, events, turn = _staging(4 * n)
        chunk = bufs[0].numel() // 4
        for off in range(0, n, chunk):
            m = min(chunk, n - off)
            b = turn[0] = (turn[0] + 1) % len(bufs)
            piece = bufs[b].view(out.dtype)[:m]
            events[b].synchronize()                      # the buffer's previous piece has left
            piece.copy_(src[off:off + m])
            out[off:off + m].copy_(piece, non_blocking=True)
            events[b].record()
    return out


class _Downloads:
    """32-bit tensors of one device as host tensors of given types, through that device's staging
    buffers and behind the work on its current stream: as many pieces as there are buffers are under
    way from the start, and ``get(i)`` converts (on the host's threads) what has arrived until tensor
    i is complete.  To be used as a context, tensors in order.  The tensors' device is the current one
    in it: a copy runs on a stream of the tensor's device, an event is recorded on one of the current
    device's."""

    def __init__(self, wanted):
        torch = _torch()
        self._out = [torch.empty(t.numel(), dtype=dtype) for t, dtype in wanted]
        self._wanted = wanted

    def __enter__(self):
        self._outer = _torch().cuda.current_device()
        self._device = self._wanted[0][0].device.index
        _stage_lock.acquire()
        try:
            self._switch(self._outer, self._device)
            self._bufs, self._events, self._turn = _staging(max(4 * t.numel() for t, _ in self._wanted))
            chunk = self._bufs[0].numel() // 4
            self._todo = [(i, off, min(chunk, t.numel() - off)) for i, (t, _) in enumerate(self._wanted)
                          for off in range(0, t.numel(), chunk)][::-1]
            self._ahead = []
            self._request()
        except BaseException:
            self.__exit__()
            raise
        return self

    @staticmethod
    def _switch(current, wanted):
        if current != wanted:
            _torch().cuda.set_device(wanted)

    def _request(self):
        while self._todo and len(self._ahead) < len(self._bufs):
            i, off, m = self._todo.pop()
            b = self._turn[0] = (self._turn[0] + 1) % len(self._bufs)
            self._events[b].synchronize()                # (an upload's piece may be leaving it)
            src = self._wanted[i][0]
            piece = self._bufs[b].view(src.dtype)[:m]
            piece.copy_(src[off:off + m], non_blocking=True)
            self._events[b].record()
            self._ahead.append((i, off, b, piece))

    def get(self, i):
        while self._ahead and self._ahead[0][0] <= i:
            j, off, b, piece = self._ahead.pop(0)
            self._events[b].synchronize()
            self._out[j][off:off + len(piece)].copy_(piece)
            self._request()
        return self._out[i]

    def __exit__(self, *exc):
        try:
            self._switch(self._device, self._outer)
        finally:
            _stage_lock.release()


def _all_ones(data) -> bool:
    """Whether a host array holds nothing but 1 (the first entries settle it for most that do not)."""
    return bool(np.all(data[:1024] == 1)) and bool(np.all(data == 1))


class _DeviceCSR:
    """CSR arrays of a matrix on the GPU (int32 indices, float32 values): sorted columns,
    duplicates summed - the GPU counterpart of the scipy conversion behind
    adj_tensors("csr") (format_matrix_market.py:74-76).

    Two ways in.  A container made from CSR arrays (``MTX.from_csr``) is uploaded as it is and
    checked on the GPU (lf_csr_check): if the arrays are canonical already they are the
    result - no COO triplets on the host, no sort.  Anything else, and a CSR input that turns
    out unsorted or with duplicates, goes up as COO triplets and is sorted and merged by
    lf_coo_to_csr.  ``self.path`` says which one was taken ("csr" or "coo")."""

    def __init__(self, g):
        torch = _torch()
        self.num_rows = int(g.num_src_nodes())
        self.num_cols = int(g.num_dst_nodes())
        # The reference counts degrees from raw COO triplets (format_algos.py:250, 846); they
        # differ from the CSR row lengths only when the COO holds duplicates.
        self.coo_nnz = int(g.num_edges())
        if self.coo_nnz >= 2**31:
            raise NotImplementedError("matrices with 2^31 or more stored entries are not supported")
        self._g = g
        self._seg_deg = {}
        self._stats_ws = {}          # num_parts -> statistics workspace holding the row bounds
        self._span = None
        self._longest = 0            # entries of the longest row, or more (lf_coo_to_csr_rows)
        self._long_rows = None       # list of long rows and its counts, see csr_work
        self._csr_work = {}
        src = getattr(g, "_csr_source", None)
        if src is not None and self._from_csr(src, bool(getattr(g, "_unit_values", False))):
            self.path = "csr"
        else:
            self._from_coo(*self._triplets())
            self.path = "coo"
        torch.cuda.current_stream().synchronize()

    def _triplets(self):
        triplets = getattr(self._g, "_triplets", None)
        if triplets is None:
            coo = self._g.coo_mtx
            triplets = (coo.row, coo.col, coo.data)
        return triplets[:3]

    @property
    def span(self) -> int:
        """Columns that four neighbouring rows span, on average over a sample (0: not known): measured by the check of
        CSR arrays; of triplets, in whatever order, twice the distance from the diagonal that one in ten exceeds."""
        if self._span is None:
            row, col, _ = self._triplets()
            self._span = 0
            if len(row):
                at = np.linspace(0, len(row) - 1, 512).astype(np.int64)
                away = np.abs(np.asarray(col)[at] - np.asarray(row)[at] * (self.num_cols / self.num_rows))
                self._span = int(2 * np.partition(away, 460)[460])
        return self._span

    def _from_csr(self, csr, unit_values: bool) -> bool:
        """Uploads the CSR arrays; False (nothing kept) when they are not canonical.  Raises
        ValueError for arrays that are not a CSR structure at all."""
        torch = _torch()
        lib = _lib.load()
        nnz = int(csr.nnz)
        indptr = _upload(csr.indptr, np.int32)
        indices = _upload(csr.indices, np.int32)
        values = None if unit_values else _upload(csr.data, np.float32)
        scratch = torch.empty(8, dtype=torch.int32, device="cuda")
        flags, span, longest = C.c_int32(0), C.c_int64(0), C.c_int64(0)
        _lib.check(lib.lf_csr_check_rows(_lib.ptr(indptr), _lib.ptr(indices), _lib.ptr(values), self.num_rows, self.num_cols,
                                         nnz, _lib.ptr(scratch), C.byref(flags), C.byref(span), C.byref(longest), _stream()))
        if not flags.value & _lib.LF_CSR_CANONICAL:
            return False
        self._span, self._longest = int(span.value), int(longest.value)
        self.indptr, self.indices, self.nnz = indptr, indices, nnz
        self.all_ones = unit_values or bool(flags.value & _lib.LF_CSR_UNIT_VALUES)
        self._values = values
        return True

    @property
    def values(self):
        """A's values on the device (ones are made on first use when none were uploaded)."""
        if self._values is None:
            self._values = _torch().ones(self.nnz, dtype=_torch().float32, device="cuda")
        return self._values

    def _from_coo(self, row, col, data):
        torch = _torch()
        lib = _lib.load()
        row = _upload(row, np.int32)
        col = _upload(col, np.int32)
        data = np.asarray(data)
        ones = _all_ones(data)
        val = None if ones else _upload(data, np.float32)
        n = max(self.coo_nnz, 1)
        self.indptr = torch.empty(self.num_rows + 1, dtype=torch.int32, device="cuda")
        indices = torch.empty(n, dtype=torch.int32, device="cuda")
        values = torch.empty(n, dtype=torch.float32, device="cuda")
        nbytes = lib.lf_coo_to_csr_workspace_bytes(self.coo_nnz, self.num_rows, self.num_cols)
        ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device="cuda")
        out, longest = C.c_int64(0), C.c_int64(0)
        _lib.check(lib.lf_coo_to_csr_rows(_lib.ptr(row), _lib.ptr(col), _lib.ptr(val), self.coo_nnz, self.num_rows,
                                          self.num_cols, _lib.ptr(ws), nbytes, _lib.ptr(self.indptr),
                                          _lib.ptr(indices), _lib.ptr(values), C.byref(out), C.byref(longest), _stream()))
        self.nnz, self._longest = int(out.value), int(longest.value)
        self.indices = indices[:self.nnz]
        self._values = values[:self.nnz]
        # duplicates of unit entries add up to 2, 3, ...: only a duplicate-free unit matrix is "all ones"
        self.all_ones = ones and self.nnz == self.coo_nnz

    def csr_work(self, feat: int, dtype: int):
        """What the C call of a CSR product takes: ((rows, columns, entries, span), list of long rows, its counts, bytes of work
        space).  The list (lf_csr_long_rows) is made for the first product that wants it and kept with the matrix; a product
        that is recorded into a graph before there is one does without.  (Tensor and array, no addresses: the matrix may be
        copied with what it holds.)"""
        work = self._csr_work.get((feat, dtype))
        if work is None:
            lib = _lib.load()
            sizes = (self.num_rows, self.num_cols, self.nnz, self.span)
            rows = counts = None
            nbytes = -1
            if self._long_rows is None:
                nbytes = lib.lf_csr_spmm_work_bytes(*sizes, None, self._longest, feat, dtype)
            keep = nbytes >= 0
            if not keep:
                rows, counts = self._long_row_list()
                keep = self._long_rows is not None
                nbytes = lib.lf_csr_spmm_work_bytes(*sizes, _lib.ptr(counts), 0, feat, dtype)
            work = (sizes, rows, counts, nbytes)
            if keep:
                self._csr_work[(feat, dtype)] = work
        return work

    def _long_row_list(self):
        """The list of long rows and its counts; None where there are no such rows, or no list yet and the stream is being
        recorded."""
        with _long_rows_lock:
            if self._long_rows is None and not _torch().cuda.is_current_stream_capturing():
                lib = _lib.load()
                rows = _gpu_torch.empty(lib.lf_csr_long_rows_bytes(self.nnz), dtype=_gpu_torch.uint8, device="cuda")
                counts = np.zeros(3, dtype=np.int64)
                _lib.check(lib.lf_csr_long_rows(self.indptr.data_ptr(), self.num_rows, self.nnz, rows.data_ptr(), rows.numel(),
                                                _lib.np_ptr(counts, C.c_int64), _stream()))
                self._long_rows = (rows, counts) if counts[0] else (None, None)
            return self._long_rows or (None, None)

    def seg_deg(self, num_parts: int):
        """Per-(partition,row) COO degrees on the device, or None when CSR lengths are the same."""
        if self.coo_nnz == self.nnz:
            return None
        if num_parts not in self._seg_deg:
            torch = _torch()
            lib = _lib.load()
            row = torch.from_numpy(np.ascontiguousarray(self._g.coo_mtx.row, dtype=np.int32)).cuda()
            col = torch.from_numpy(np.ascontiguousarray(self._g.coo_mtx.col, dtype=np.int32)).cuda()
            deg = torch.empty((num_parts, max(self.num_rows, 1)), dtype=torch.int32, device="cuda")
            _lib.check(lib.lf_coo_degrees(_lib.ptr(row), _lib.ptr(col), self.coo_nnz, self.num_rows,
                                          self.num_cols, num_parts, _lib.ptr(deg), _stream()))
            torch.cuda.current_stream().synchronize()
            self._seg_deg[num_parts] = deg
        return self._seg_deg[num_parts]


def _matrix_identity(g):
    """The object whose replacement means "another matrix": the container's own token, or the COO
    matrix of a container that has none."""
    token = getattr(g, "_identity", None)
    return g.coo_mtx if token is None else token


def _device_csr(g) -> _DeviceCSR:
    cached = getattr(g, "_lf_device_csr", None)
    if cached is not None and cached[0] is _matrix_identity(g):
        return cached[1]
    dev = _DeviceCSR(g)
    try:
        object.__setattr__(g, "_lf_device_csr", (_matrix_identity(g), dev))
    except Exception:
        pass
    return dev


def _cost_model_id(cfg) -> int:
    name = getattr(cfg, "cost_model", "reference")
    if name == "reference":
        return _lib.LF_COST_REFERENCE
    if name == "gfx950":
        return _lib.LF_COST_GFX950
    raise ValueError(f"unknown cost model {name!r}")


# --------------------------------------------------------------------------- search
def bucket_statistics(g, num_parts: int, width_limit: int = WIDTH_LIMIT, with_columns: bool = True):
    """Per-partition, per-width-class statistics of the initial bucketing
    (what get_init_buckets, format_algos.py:819-900, collects), computed on the GPU.

    Returns (stats, colhist): stats[p][k] = (cost-model rows, nnz, distinct rows, 0) for
    width 2**k; colhist[p][m] = number of columns whose set of touching classes is mask m
    (None with ``with_columns=False``: the gfx950 cost model does not use column sets)."""
    torch = _torch()
    lib = _lib.load()
    dev = _device_csr(g)
    stats = np.zeros((num_parts, _lib.LF_MAX_CLASSES, _lib.LF_STATS_FIELDS), dtype=np.int64)
    hist = np.zeros((num_parts, 1 << _lib.LF_MAX_CLASSES), dtype=np.int64) if with_columns else None
    nbytes = lib.lf_stats_workspace_bytes(dev.num_rows, dev.num_cols, num_parts)
    ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device="cuda")
    _lib.check(lib.lf_bucket_stats(_lib.ptr(dev.indptr), _lib.ptr(dev.indices), _lib.ptr(dev.seg_deg(num_parts)),
                                   dev.num_rows, dev.num_cols, num_parts, width_limit,
                                   _lib.ptr(ws), nbytes, _lib.np_ptr(stats, C.c_int64),
                                   _lib.np_ptr(hist, C.c_int64) if with_columns else None, _stream()))
    if num_parts > 1:
        # the pass left the per-partition row bounds in its workspace; the slab builder takes
        # them over instead of searching the column indices again
        dev._stats_ws[num_parts] = ws
    return stats, hist


def search_from_statistics(stats, hist, cost_model_config, width_limit: int = WIDTH_LIMIT,
                           return_trace: bool = False):
    """Host part of the search (format_algos.py:928-954, 709-816, 1035-1166)."""
    lib = _lib.load()
    num_parts = stats.shape[0]
    stats = np.ascontiguousarray(stats, dtype=np.int64)
    hist = np.ascontiguousarray(hist, dtype=np.int64) if hist is not None else None
    widths = np.zeros((num_parts, _lib.LF_MAX_CLASSES), dtype=np.int32)
    nwidths = np.zeros(num_parts, dtype=np.int32)
    trace = np.zeros((num_parts, _lib.LF_MAX_CLASSES + 1), dtype=np.float64)
    trace_len = np.zeros(num_parts, dtype=np.int32)
    _lib.check(lib.lf_search_bucket_config(
        _lib.np_ptr(stats, C.c_int64), _lib.np_ptr(hist, C.c_int64) if hist is not None else None,
        num_parts, width_limit, int(cost_model_config.feat_size), int(cost_model_config.num_parts), _cost_model_id(cost_model_config),
        _lib.np_ptr(widths, C.c_int32), _lib.np_ptr(nwidths, C.c_int32),
        _lib.np_ptr(trace, C.c_double), _lib.np_ptr(trace_len, C.c_int32)))
    config = [[int(w) for w in widths[p, :nwidths[p]]] for p in range(num_parts)]
    if return_trace:
        return config, [trace[p, :trace_len[p]].tolist() for p in range(num_parts)]
    return config


def search_bucket_config(g, num_parts: int, cost_model_config) -> List[List[int]]:
    """Bucket widths per column partition (format_algos.py:988-1032)."""
    num_parts = int(num_parts)
    needs_columns = _cost_model_id(cost_model_config) == _lib.LF_COST_REFERENCE
    stats, hist = bucket_statistics(g, num_parts, with_columns=needs_columns)
    return search_from_statistics(stats, hist, cost_model_config)


# --------------------------------------------------------------------------- composition
class HybFormat:
    """The composed hyb format resident on the GPU.

    Flat device arrays with one slab per bucket k = (partition, width index):
      rows/meta : ELL rows  [row_off[k], row_off[k] + ell_rows[k])
      cols/vals : slots     [slot_off[k], slot_off[k] + ell_rows[k] * width[k])   (row-major (R, W))
    """

    def __init__(self, widths, num_rows, num_cols):
        self.bucket_widths = [list(map(int, ws)) for ws in widths]
        self.num_parts = len(self.bucket_widths)
        self.num_rows = int(num_rows)
        self.num_cols = int(num_cols)
        self.flat_widths = [w for ws in self.bucket_widths for w in ws]
        self.part_of = [p for p, ws in enumerate(self.bucket_widths) for _ in ws]
        self.ell_rows = None
        self.row_off = None
        self.slot_off = None
        self.rows = self.meta = self.cols = self.vals = self.mask = None
        self.compose_ms = None

    @property
    def num_buckets(self):
        return len(self.flat_widths)

    def slab(self, k):
        """(rows, cols, vals, meta[, mask]) device views of bucket k."""
        r0, s0 = int(self.row_off[k]), int(self.slot_off[k])
        R, W = int(self.ell_rows[k]), self.flat_widths[k]
        out = [self.rows[r0:r0 + R], self.cols[s0:s0 + R * W], self.vals[s0:s0 + R * W], self.meta[r0:r0 + R]]
        if self.mask is not None:
            out.append(self.mask[s0:s0 + R * W])
        return out

    def total_slots(self):
        return int(sum(int(r) * w for r, w in zip(self.ell_rows, self.flat_widths)))

    def to_numpy(self, with_values: bool = False):
        """The reference's return value of build_hyb_format (format_algos.py:361-385):
        per partition and bucket rows (R,), cols (R, W), mask (R, W) as int64 arrays."""
        torch = _torch()
        wanted = [(self.meta, torch.int64), (self.rows, torch.int64), (self.cols, torch.int64)]
        if with_values:
            wanted.append((self.vals, torch.float32))
        rows_nd, cols_nd, mask_nd, vals_nd = [], [], [], []
        mask = torch.empty(self.cols.numel(), dtype=torch.int64)
        place = torch.arange(WIDTH_LIMIT)
        buckets = [(k, w, int(self.ell_rows[k]), int(self.row_off[k]), int(self.slot_off[k]))
                   for k, w in enumerate(self.flat_widths)]
        with _Downloads(wanted) as down:
            # the mask follows from the valid slots of every ELL row, in the low bits of its meta
            # word; it is made while the columns arrive
            lens = down.get(0).bitwise_and_(0x7FF)
            for _, w, R, r0, s0 in buckets:
                torch.lt(place[:w], lens[r0:r0 + R].view(R, 1), out=mask[s0:s0 + R * w].view(R, w))
            rows, cols = down.get(1), down.get(2)
            vals = down.get(3) if with_values else None
        of_bucket = lambda flat, k, w, R, r0, s0: flat[s0:s0 + R * w].view(R, w).numpy()          # noqa: E731
        at = iter(buckets)
        for ws in self.bucket_widths:
            mine = [next(at) for _ in ws]
            rows_nd.append([rows[r0:r0 + R].numpy() for _, _, R, r0, _ in mine])
            cols_nd.append([of_bucket(cols, *b) for b in mine])
            mask_nd.append([of_bucket(mask, *b) for b in mine])
            if with_values:
                vals_nd.append([of_bucket(vals, *b) for b in mine])
        if with_values:
            return rows_nd, cols_nd, mask_nd, vals_nd
        return rows_nd, cols_nd, mask_nd


def _check_widths(bucket_widths):
    for p, ws in enumerate(bucket_widths):
        for b, w in enumerate(ws):
            w = int(w)
            # the reference trips over a non power of two in its padding assertion (format_algos.py:303)
            assert w > 0 and w & (w - 1) == 0, \
                f"invalid padding for col_indices[{p}][{b}] and bucket_width={w}"


def build_hyb_format_device(g, bucket_widths, with_values: bool = True, with_mask: bool = False) -> HybFormat:
    """Compose the hyb format on the GPU and leave it there.

    ``with_values=False`` fills the value slab with ones exactly like the reference's mask
    (format_algos.py:311, 568-570); ``with_mask=True`` additionally writes the 0/1 mask."""
    torch = _torch()
    lib = _lib.load()
    _check_widths(bucket_widths)
    dev = _device_csr(g)
    fmt = HybFormat(bucket_widths, dev.num_rows, dev.num_cols)
    P, nb = fmt.num_parts, fmt.num_buckets
    flat = np.asarray(fmt.flat_widths, dtype=np.int32)
    off = np.zeros(P + 1, dtype=np.int32)
    off[1:] = np.cumsum([len(ws) for ws in fmt.bucket_widths])
    ell_rows = np.zeros(max(nb, 1), dtype=np.int64)
    seg_deg = dev.seg_deg(P)
    nbytes = lib.lf_hyb_workspace_bytes(dev.num_rows, P, nb)
    ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device="cuda")
    stream = _stream()
    t0 = time.perf_counter()
    stats_ws = dev._stats_ws.get(P)
    bounds = lib.lf_stats_seg_bounds(_lib.ptr(stats_ws), dev.num_rows, P) if stats_ws is not None else None
    _lib.check(lib.lf_hyb_plan(_lib.ptr(dev.indptr), _lib.ptr(dev.indices), _lib.ptr(seg_deg), bounds,
                               dev.num_rows, dev.num_cols, P, _lib.np_ptr(flat, C.c_int32),
                               _lib.np_ptr(off, C.c_int32), _lib.ptr(ws), nbytes,
                               _lib.np_ptr(ell_rows, C.c_int64), stream))
    row_off = np.zeros(max(nb, 1), dtype=np.int64)
    slot_off = np.zeros(max(nb, 1), dtype=np.int64)
    tot_rows = C.c_int64(0)
    tot_slots = C.c_int64(0)
    _lib.check(lib.lf_hyb_layout(_lib.np_ptr(ell_rows, C.c_int64), _lib.np_ptr(flat, C.c_int32), nb,
                                 _lib.np_ptr(row_off, C.c_int64), _lib.np_ptr(slot_off, C.c_int64),
                                 C.byref(tot_rows), C.byref(tot_slots)))
    fmt.ell_rows, fmt.row_off, fmt.slot_off = ell_rows[:nb], row_off[:nb], slot_off[:nb]
    nr, ns = max(tot_rows.value, 1), max(tot_slots.value, 1)
    fmt.rows = torch.empty(nr, dtype=torch.int32, device="cuda")
    fmt.meta = torch.empty(nr, dtype=torch.int32, device="cuda")
    fmt.cols = torch.empty(ns, dtype=torch.int32, device="cuda")
    fmt.vals = torch.empty(ns, dtype=torch.float32, device="cuda")
    fmt.mask = torch.empty(ns, dtype=torch.float32, device="cuda") if with_mask else None
    values = dev.values if (with_values and not dev.all_ones) else None
    _lib.check(lib.lf_hyb_build(_lib.ptr(dev.indptr), _lib.ptr(dev.indices), _lib.ptr(values), _lib.ptr(seg_deg),
                                dev.num_rows, dev.num_cols, P, _lib.np_ptr(flat, C.c_int32),
                                _lib.np_ptr(off, C.c_int32), _lib.np_ptr(ell_rows, C.c_int64),
                                _lib.ptr(ws), nbytes, _lib.ptr(fmt.rows), _lib.ptr(fmt.meta),
                                _lib.ptr(fmt.cols), _lib.ptr(fmt.vals), _lib.ptr(fmt.mask), stream))
    torch.cuda.current_stream().synchronize()
    fmt.compose_ms = (time.perf_counter() - t0) * 1e3
    return fmt


def build_hyb_format(g, bucket_widths):
    """format_algos.py:226-385: (row_indices_nd, col_indices_nd, mask_nd), each a list over
    partitions of lists over buckets of numpy arrays with shapes (R,), (R, W), (R, W)."""
    return build_hyb_format_device(g, bucket_widths, with_values=False).to_numpy()


# --------------------------------------------------------------------------- SpMM
class HybSpMM:
    """Kernel plan for C = A_hyb . B on the current device (wraps lf_spmm_plan).

    ``windows`` > 1 computes the product in that many passes over ``feat_size // windows``
    features each (lf_spmm_set_windows): same result up to the summation order of the
    cooperatively reduced rows, and faster when B is much larger than the memory-side cache.

    Runs may be made on any stream and thread.  The runs of a plan with long rows (``info["heavy_rows"]``) share
    scratch memory: one on another stream than the run before waits for it on the GPU.  A run that is
    recorded into a HIP graph has no such guard: the graph must not be launched while another run of
    the plan is under way."""

    def __init__(self, fmt_or_slabs, feat_size: int, b_dtype: str = "f32", num_rows=None, num_cols=None,
                 bucket_widths=None, windows: int = 1):
        torch = _torch()
        if windows < 1 or feat_size % windows:
            raise ValueError(f"feat_size {feat_size} is not a multiple of windows {windows}")
        lib = _lib.load()
        self._lib = lib
        self._keep = []
        self.handle = C.c_void_p(None)
        if isinstance(fmt_or_slabs, HybFormat):
            fmt = fmt_or_slabs
            self._keep.append(fmt)
            descs = (_lib.BucketDesc * max(fmt.num_buckets, 1))()
            rows, cols, vals, meta = (t.data_ptr() for t in (fmt.rows, fmt.cols, fmt.vals, fmt.meta))
            for k, (w, p, n, r0, s0) in enumerate(zip(fmt.flat_widths, fmt.part_of, fmt.ell_rows.tolist(),
                                                      fmt.row_off.tolist(), fmt.slot_off.tolist())):
                descs[k] = _lib.BucketDesc(w, p, n, rows + 4 * r0, cols + 4 * s0, vals + 4 * s0, meta + 4 * r0)
            nb, P = fmt.num_buckets, fmt.num_parts
            num_rows, num_cols = fmt.num_rows, fmt.num_cols
        else:
            # reference-style tuple (rows, cols, mask-or-values) of numpy arrays per (partition, bucket)
            rows_nd, cols_nd, vals_nd = fmt_or_slabs[:3]
            P = len(bucket_widths)
            nb = sum(len(ws) for ws in bucket_widths)
            descs = (_lib.BucketDesc * max(nb, 1))()
            k = 0
            for p, ws in enumerate(bucket_widths):
                for b, w in enumerate(ws):
                    r = torch.from_numpy(np.ascontiguousarray(rows_nd[p][b], dtype=np.int32)).cuda()
                    c = torch.from_numpy(np.ascontiguousarray(cols_nd[p][b], dtype=np.int32).reshape(-1)).cuda()
                    v = torch.from_numpy(np.ascontiguousarray(vals_nd[p][b], dtype=np.float32).reshape(-1)).cuda()
                    self._keep += [r, c, v]
                    descs[k] = _lib.BucketDesc(int(w), p, int(r.numel()), r.data_ptr(), c.data_ptr(),
                                               v.data_ptr(), None)
                    k += 1
        self.feat_size = int(feat_size)
        self.b_dtype = b_dtype
        self.num_rows, self.num_cols = int(num_rows), int(num_cols)
        dt = {"f32": _lib.LF_DTYPE_F32, "bf16": _lib.LF_DTYPE_BF16}[b_dtype]
        self.windows = int(windows)
        self._b_type = torch.float32 if b_dtype == "f32" else torch.bfloat16
        self._b_shape, self._c_shape = (self.num_cols, self.feat_size), (self.num_rows, self.feat_size)
        _lib.check(lib.lf_spmm_create(C.byref(self.handle), descs, nb, P, self.num_rows, self.num_cols,
                                      self.feat_size // self.windows, dt, _stream()))
        if self.windows > 1:
            _lib.check(lib.lf_spmm_set_windows(self.handle, self.windows))
        info = np.zeros(_lib.LF_SPMM_INFO_FIELDS, dtype=np.int64)
        _lib.check(lib.lf_spmm_info(self.handle, _lib.np_ptr(info, C.c_int64)))
        self.info = dict(zip(["tiles", "grid", "launches", "lds_bytes", "heavy_rows", "partial_rows",
                              "cleared_rows", "row_group_buckets", "cell_buckets"], info.tolist()))
        self.info["launches"] *= self.windows
        self.info["windows"] = self.windows

    def _check_operands(self, B, Cout):
        if B.dtype is not self._b_type or not B.is_cuda or not B.is_contiguous() or B.shape != self._b_shape:
            raise ValueError(f"B must be a contiguous CUDA tensor of shape {self._b_shape} and dtype {self._b_type}")
        if Cout is not None and (Cout.dtype is not _gpu_torch.float32 or not Cout.is_cuda or not Cout.is_contiguous()
                                 or Cout.shape != self._c_shape):
            raise ValueError(f"C must be a contiguous float32 CUDA tensor of shape {self._c_shape}")

    def run(self, B, Cout=None):
        self._check_operands(B, Cout)
        if Cout is None:
            Cout = B.new_empty(self._c_shape, dtype=_gpu_torch.float32)
        rc = self._lib.lf_spmm_run(self.handle, B.data_ptr(), Cout.data_ptr(), _stream())
        if rc:
            _lib.check(rc)
        return Cout

    def time_ms(self, B, Cout, warmup: int = 10, repeat: int = 100, flush=None):
        """Kernel time per run in ms (HIP events on the current stream), `repeat` samples."""
        self._check_operands(B, Cout)
        ms = np.zeros(repeat, dtype=np.float32)
        fptr = flush.data_ptr() if flush is not None else None
        fbytes = flush.numel() * flush.element_size() if flush is not None else 0
        _lib.check(self._lib.lf_spmm_time_ms(self.handle, B.data_ptr(), Cout.data_ptr(), warmup, repeat,
                                             fptr, fbytes, _lib.np_ptr(ms, C.c_float), _stream()))
        return ms

    def close(self):
        if self.handle:
            self._lib.lf_spmm_destroy(self.handle)
            self.handle = C.c_void_p(None)

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def spmm_hyb(fmt: HybFormat, B, b_dtype: str = "f32"):
    """One-shot C = A_hyb . B; B is a CUDA tensor (cols, N); returns a CUDA float32 tensor."""
    plan = HybSpMM(fmt, B.shape[1], b_dtype)
    try:
        out = plan.run(B)
        _torch().cuda.current_stream().synchronize()
    finally:
        plan.close()
    return out


_B_DTYPES = {"f32": _lib.LF_DTYPE_F32, "bf16": _lib.LF_DTYPE_BF16}


def spmm_csr(g, B, b_dtype: str = "f32", use_values: bool = True):
    """Row-parallel CSR product on the GPU (kernel of bench_naive, format_algos.py:1689-1755)."""
    torch = _torch()
    lib = _lib.load()
    dev = _device_csr(g)
    feat, dtype = int(B.shape[1]), _B_DTYPES[b_dtype]
    out = dev.indptr.new_empty((dev.num_rows, feat), dtype=torch.float32)
    vals = dev.values if use_values else None
    work = dev._csr_work.get((feat, dtype))
    # the device arrays were made by lf_coo_to_csr or have passed lf_csr_check: no second check
    if work is None:
        rc = lib.lf_csr_spmm_trusted_rows(dev.indptr.data_ptr(), dev.indices.data_ptr(), None if vals is None else vals.data_ptr(),
                                          dev.num_rows, dev.num_cols, dev.nnz, dev.span if dev._span is None else dev._span, dev._longest,
                                          feat, dtype, B.data_ptr(), out.data_ptr(), _stream())
        if rc == 0:
            return out
        if rc != _lib.LF_WANTS_WORK:
            _lib.check(rc)
    sizes, rows, counts, nbytes = work or dev.csr_work(feat, dtype)
    work = torch.empty(nbytes, dtype=torch.uint8, device="cuda") if nbytes else None
    rc = lib.lf_csr_spmm_trusted_work(dev.indptr.data_ptr(), dev.indices.data_ptr(), None if vals is None else vals.data_ptr(), *sizes,
                                      _lib.ptr(rows), _lib.ptr(counts), _lib.ptr(work), nbytes, feat, dtype, B.data_ptr(),
                                      out.data_ptr(), _stream())
    if rc:
        _lib.check(rc)
    return out


def _flush_buffer():
    """Cache-eviction buffer used between timed runs when FLUSH_L2=ON, as the reference's
    driver script sets it (drive05.spmm.end-to-end.sh:1; format_algos.py:171, 187).  512 MB:
    larger than L2 plus the 256 MB memory-side cache."""
    if os.getenv("FLUSH_L2", "OFF") != "ON":
        return None
    return _torch().empty(int(512e6), dtype=_torch().int8, device="cuda")


def _timing_params():
    return int(os.getenv("LF_WARMUP", "10")), int(os.getenv("LF_REPEAT", "100"))


def bench_hyb_with_config(g, x, y_ndarray, feat_size=128, bucket_widths=[], bucketing_format=[],
                          coarsening_factor=2, num_col_parts=1, use_implicit_unroll=False,
                          check_correctness=False, feature_windows=1):
    """Build and time the fused hyb SpMM kernel; returns the mean kernel time in ms
    (format_algos.py:388-605).  ``feature_windows`` (not in the reference) computes the
    product in that many passes over the features, see ``HybSpMM``.

    ``bucketing_format`` is what build_hyb_format returned - then, as in the reference, the
    mask is used as A's values (format_algos.py:568-570) - or a ``HybFormat`` from
    build_hyb_format_device, which carries A's real values.  ``coarsening_factor`` and
    ``use_implicit_unroll`` steer the reference's CUDA schedule and have no effect here."""
    torch = _torch()
    t_start = time.perf_counter()
    num_rows = g.num_src_nodes()
    num_cols = g.num_dst_nodes()
    if isinstance(bucketing_format, HybFormat):
        plan = HybSpMM(bucketing_format, feat_size, "f32", windows=feature_windows)
    else:
        plan = HybSpMM(bucketing_format, feat_size, "f32", num_rows=num_rows, num_cols=num_cols,
                       bucket_widths=[list(ws) for ws in bucket_widths][:num_col_parts], windows=feature_windows)
    try:
        xb = x.numpy() if hasattr(x, "numpy") else np.asarray(x)
        B = torch.from_numpy(np.ascontiguousarray(xb.reshape(num_cols, feat_size), dtype=np.float32)).cuda()
        Cout = torch.empty((num_rows, feat_size), dtype=torch.float32, device="cuda")
        print(f"plan_build_time(s): {time.perf_counter() - t_start:.6}")
        plan.run(B, Cout)
        torch.cuda.current_stream().synchronize()
        if check_correctness:
            np.testing.assert_allclose(Cout.cpu().numpy().reshape(-1, feat_size), y_ndarray, rtol=1e-4)
        warmup, repeat = _timing_params()
        ms = plan.time_ms(B, Cout, warmup, repeat, _flush_buffer())
        dur = float(ms.mean())
        bench_hyb_with_config.last_output = Cout
    finally:
        plan.close()
    print("cell exe time: {:.6f} ms".format(dur))
    return dur


class _DeviceBSR:
    """scipy BSR arrays on the GPU: int32 index arrays, fp16 blocks."""

    checked = False                   # the first product checks the block index arrays on the GPU

    def __init__(self, bsr_mat, block_size: int):
        torch = _torch()
        if tuple(bsr_mat.blocksize) != (block_size, block_size):
            raise ValueError(f"matrix has blocks {bsr_mat.blocksize}, expected {(block_size, block_size)}")
        if not bsr_mat.has_sorted_indices:
            bsr_mat = bsr_mat.copy()
            bsr_mat.sort_indices()
        self.block_size = block_size
        self.mb = bsr_mat.shape[0] // block_size
        self.nb = bsr_mat.shape[1] // block_size
        self.nnzb = int(len(bsr_mat.indices))
        self.indptr = torch.from_numpy(np.ascontiguousarray(bsr_mat.indptr, dtype=np.int32)).cuda()
        self.indices = torch.from_numpy(np.ascontiguousarray(bsr_mat.indices, dtype=np.int32)).cuda()
        self.data = torch.from_numpy(np.ascontiguousarray(bsr_mat.data, dtype=np.float16).reshape(-1)).cuda()


def spmm_bsr(bsr, x, block_size: int = 32):
    """Y = A_bsr . X on the matrix cores.  ``bsr`` is a scipy BSR matrix or a ``_DeviceBSR``;
    ``x`` a CUDA fp16 tensor (cols, N).  Returns a CUDA fp16 tensor (rows, N)."""
    torch = _torch()
    lib = _lib.load()
    dev = bsr if isinstance(bsr, _DeviceBSR) else _DeviceBSR(bsr, block_size)
    feat = x.shape[1]
    if x.dtype != torch.float16 or not x.is_cuda or not x.is_contiguous() or x.shape[0] != dev.nb * dev.block_size:
        raise ValueError(f"x must be a contiguous CUDA fp16 tensor with {dev.nb * dev.block_size} rows")
    y = x.new_empty((dev.mb * dev.block_size, feat))
    if not dev.checked:
        scratch = torch.empty(4, dtype=torch.int32, device="cuda")
        _lib.check(lib.lf_bsr_spmm(_lib.ptr(dev.indptr), _lib.ptr(dev.indices), _lib.ptr(dev.data), dev.mb, dev.nb,
                                   dev.nnzb, dev.block_size, feat, x.data_ptr(), y.data_ptr(), _lib.ptr(scratch),
                                   _stream()))
        dev.checked = True
    else:
        rc = lib.lf_bsr_spmm_trusted_nnz(dev.indptr.data_ptr(), dev.indices.data_ptr(), dev.data.data_ptr(), dev.mb,
                                         dev.nb, dev.nnzb, dev.block_size, feat, x.data_ptr(), y.data_ptr(), _stream())
        if rc:
            _lib.check(rc)
    return y


def bench_bsrmm(bsr_mat, x, block_size: int):
    """Time the block-sparse fp16 kernel; returns the mean kernel time in ms
    (format_algos.py:1562-1643).  ``x`` is a (cols, N) fp16 torch tensor on the host, as the
    driver makes it (proc05.spmm.end-to-end.py:221)."""
    torch = _torch()
    dev = _DeviceBSR(bsr_mat, block_size)
    xd = x.to(torch.float16).contiguous().cuda()
    bench_bsrmm.last_output = spmm_bsr(dev, xd)
    warmup, repeat = _timing_params()
    flush = _flush_buffer()
    for _ in range(warmup):
        spmm_bsr(dev, xd)
    starts = [torch.cuda.Event(enable_timing=True) for _ in range(repeat)]
    ends = [torch.cuda.Event(enable_timing=True) for _ in range(repeat)]
    for i in range(repeat):
        if flush is not None:
            flush.zero_()
        starts[i].record()
        spmm_bsr(dev, xd)
        ends[i].record()
    torch.cuda.synchronize()
    avg_time = float(np.mean([s.elapsed_time(e) for s, e in zip(starts, ends)]))
    print("bsrmm time: \t{:.5f}ms".format(avg_time))
    return avg_time


def bench_naive(g, x, y_ndarray, feat_size=128, coarsening_factor=2, check_correctness=False):
    """Time the row-parallel CSR kernel (format_algos.py:1689-1755).  Like the reference,
    A's stored values are taken as ones (format_algos.py:1746)."""
    torch = _torch()
    num_cols = g.num_dst_nodes()
    xb = x.numpy() if hasattr(x, "numpy") else np.asarray(x)
    B = torch.from_numpy(np.ascontiguousarray(xb.reshape(num_cols, feat_size), dtype=np.float32)).cuda()
    out = spmm_csr(g, B, use_values=False)
    torch.cuda.current_stream().synchronize()
    if check_correctness:
        np.testing.assert_allclose(out.cpu().numpy().reshape(-1, feat_size), y_ndarray, rtol=1e-4)
    warmup, repeat = _timing_params()
    flush = _flush_buffer()
    for _ in range(warmup):
        spmm_csr(g, B, use_values=False)
    starts = [torch.cuda.Event(enable_timing=True) for _ in range(repeat)]
    ends = [torch.cuda.Event(enable_timing=True) for _ in range(repeat)]
    for i in range(repeat):
        if flush is not None:
            flush.zero_()
        starts[i].record()
        spmm_csr(g, B, use_values=False)
        ends[i].record()
    torch.cuda.synchronize()
    dur = float(np.mean([s.elapsed_time(e) for s, e in zip(starts, ends)]))
    print("csr naive time: {:.5f} ms".format(dur))
    return dur


# --------------------------------------------------------------------------- partition count
def matrix_features_device(g) -> dict:
    """``MTX.matrix_features`` (format_matrix_market.py:153-202) with the pass over the
    row pointer done on the GPU: the kernel returns min, max, sum and sum of squares of the
    row lengths as exact integers; mean, standard deviation and the densities follow from
    them in float64 (the standard deviation as sqrt(E[d^2] - E[d]^2), which agrees with
    numpy's two-pass value to ~1e-12 relative for these integer inputs)."""
    torch = _torch()
    lib = _lib.load()
    dev = _device_csr(g)
    out = np.zeros(4, dtype=np.int64)
    scratch = torch.empty(4, dtype=torch.int64, device="cuda")
    _lib.check(lib.lf_row_features(_lib.ptr(dev.indptr), dev.num_rows, _lib.ptr(scratch),
                                   _lib.np_ptr(out, C.c_int64), _stream()))
    rows, cols = dev.num_rows, dev.num_cols
    lo, hi, total, squares = (int(x) for x in out)
    mean = total / rows if rows else 0.0
    var = max(0.0, squares / rows - mean * mean) if rows else 0.0
    std = float(np.sqrt(var))
    return {
        "name": getattr(g, "name", None),
        "num_rows": rows,
        "num_cols": cols,
        "nnz": dev.coo_nnz,                      # stored COO entries, as the reference reports
        "avg_nnz_per_row": mean,
        "min_nnz_per_row": lo,
        "max_nnz_per_row": hi,
        "std_dev_nnz_per_row": std,
        "avg_nnz_density_per_row": mean / cols,
        "min_nnz_density_per_row": lo / cols,
        "max_nnz_density_per_row": hi / cols,
        "std_dev_nnz_density_per_row": std / cols,
    }


ROW_OVERLAP_STRUCTURED = 0.3      # rows sharing this share of their columns with the row before: structured


def row_overlap_device(g, max_samples: int = 8192) -> float:
    """Share of a row's columns that also occur in the row before it, from a sample of rows
    (lf_row_overlap).  Near 0 for graphs with scattered neighbours, 0.67 for a 27-point
    stencil: one of the matrix features behind the launch-shape choice, next to
    ``matrix_features_device``."""
    torch = _torch()
    lib = _lib.load()
    dev = _device_csr(g)
    if dev.nnz == 0 or dev.num_rows < 2:
        return 0.0
    out = np.zeros(2, dtype=np.int64)
    scratch = torch.empty(2, dtype=torch.int64, device="cuda")
    stride = max(1, dev.num_rows // max_samples)
    _lib.check(lib.lf_row_overlap(_lib.ptr(dev.indptr), _lib.ptr(dev.indices), dev.num_rows, stride,
                                  _lib.ptr(scratch), _lib.np_ptr(out, C.c_int64), _stream()))
    return float(out[0]) / float(out[1]) if out[1] else 0.0


def model_spmm_ms(stats, windows: int, num_rows: int, num_cols: int, feat_size: int, b_dtype: str = "f32") -> float:
    """Predicted milliseconds of one product for the partitions described by ``stats``
    (``bucket_statistics``) and ``windows`` feature windows (lf_model_spmm_ms; host only)."""
    return _modelled_ms("lf_model_spmm_ms", stats, windows, num_rows, num_cols, feat_size, b_dtype)


def _modelled_ms(model: str, stats, windows: int, num_rows: int, num_cols: int, feat_size: int, b_dtype: str) -> float:
    lib = _lib.load()
    stats = np.ascontiguousarray(stats, dtype=np.int64)
    out = C.c_double(0.0)
    dt = {"f32": _lib.LF_DTYPE_F32, "bf16": _lib.LF_DTYPE_BF16}[b_dtype]
    _lib.check(getattr(lib, model)(_lib.np_ptr(stats, C.c_int64), int(stats.shape[0]), int(windows), int(num_rows),
                                   int(num_cols), int(feat_size), dt, C.byref(out)))
    return float(out.value)


def pick_launch_shape(predicted: dict):
    """The (partitions, windows) pair with the fewest launches among those predicted (or
    measured) within 2 % of the fastest: fewer partitions mean less memory and fewer passes
    over C, and differences below that are noise."""
    fastest = min(predicted.values())
    return min((k for k, t in predicted.items() if t <= 1.02 * fastest), key=lambda k: (k[0] * k[1], k[0]))


# Partition counts the launch-shape model prices.  The reference's predictor and its driver go up
# to 32 (proc05.spmm.end-to-end.py:145-148: 16 for ppi, 32 for proteins).
PARTITION_CANDIDATES = (1, 2, 3, 4, 8, 16, 32)
# More than four partitions pay only where the part of B that one launch reads fits an L2, and
# each of the eight L2s has to fetch that part itself: a row of B must be used more than eight
# times for anything to be left to hit.
DENSE_USES_PER_B_ROW = 8


def predict_launch_shape(g, feat_size: int, b_dtype: str = "f32", candidates: Sequence[int] = PARTITION_CANDIDATES,
                         windows: Sequence[int] = None, return_predictions: bool = False):
    """Column-partition count and feature-window count from a model of the MI355X memory
    system, without composing a format or running a kernel.  Takes the place of the
    reference's partition predictor, a RandomForest on eight matrix features
    (proc05.spmm.end-to-end.py:82-97, 142) whose model file is not distributed.

    Inputs: the bucket statistics of every candidate partition count (one pass over the row
    pointer each, on the GPU) and the share of columns consecutive rows have in common.  A
    structured matrix (stencil, band) reads B through the L2 whatever the shape: one
    partition, one window.  Otherwise lf_model_shape_ms prices every candidate and
    ``pick_launch_shape`` takes the cheapest; candidates above four partitions are priced only
    for matrices that use a row of B more than eight times on average.  Costs a few
    milliseconds of GPU time at most where ``choose_launch_shape`` spends hundreds composing and
    timing."""
    if windows is None:
        windows = _window_candidates(feat_size, b_dtype)
    rows, cols = int(g.num_src_nodes()), int(g.num_dst_nodes())
    dense = int(g.num_edges()) > DENSE_USES_PER_B_ROW * cols
    few = [p for p in candidates if p <= 4] or [min(candidates)]
    priced = [p for p in candidates if p in few or dense]
    at_once = _shape_statistics(g, priced)
    predicted = {}
    overlap = at_once[1] if at_once is not None else row_overlap_device(g)
    if overlap >= ROW_OVERLAP_STRUCTURED:
        best = (min(candidates), _structured_windows(feat_size, b_dtype, windows))
    else:
        for i, p in enumerate(priced):
            if at_once is not None:
                stats = at_once[0][i]
            else:
                try:
                    stats, _ = bucket_statistics(g, p, with_columns=False)
                except ValueError:
                    continue
            for w in windows:
                predicted[(p, w)] = _modelled_ms("lf_model_shape_ms", stats, w, rows, cols, feat_size, b_dtype)
        best = pick_launch_shape(predicted)
        # a statistics pass leaves its per-partition row bounds behind for the slab builder
        # ((P + 1) x rows words each); only those of the chosen partition count are of use
        kept = _device_csr(g)._stats_ws
        for p in [p for p in kept if p != best[0]]:
            del kept[p]
    return (best, predicted) if return_predictions else best


def _shape_statistics(g, parts: Sequence[int], max_samples: int = 8192):
    """(statistics of every partition count in ``parts``, row overlap) from one pass on the GPU
    (lf_shape_stats), or None where its limits do not allow it: degrees that are not the CSR's
    (duplicates in the COO), more than 16 counts or 128 partitions together."""
    dev = _device_csr(g)
    total = sum(parts)
    if dev.coo_nnz != dev.nnz or dev.nnz == 0 or dev.num_rows < 2 or len(parts) > 16 or total > 128 or min(parts) < 1:
        return None
    torch = _torch()
    lib = _lib.load()
    stats = np.empty((total, _lib.LF_MAX_CLASSES, _lib.LF_STATS_FIELDS), dtype=np.int64)
    shared = np.empty(2, dtype=np.int64)
    counts = np.asarray(parts, dtype=np.int32)
    nbytes = lib.lf_shape_stats_workspace_bytes(total)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    _lib.check(lib.lf_shape_stats(dev.indptr.data_ptr(), dev.indices.data_ptr(), dev.num_rows, dev.num_cols,
                                  _lib.np_ptr(counts, C.c_int32), len(parts), WIDTH_LIMIT, max(1, dev.num_rows // max_samples),
                                  ws.data_ptr(), nbytes, _lib.np_ptr(stats, C.c_int64), _lib.np_ptr(shared, C.c_int64),
                                  _stream()))
    ends = np.cumsum(counts)
    overlap = float(shared[0]) / float(shared[1]) if shared[1] else 0.0
    return [stats[e - p:e] for p, e in zip(parts, ends.tolist())], overlap


def _structured_windows(feat_size: int, b_dtype: str, windows: Sequence[int]) -> int:
    """Feature windows for a structured matrix.  Its kernels hold one accumulator per output row
    and feature slice in registers, so they want a row of B to be one 16-byte load per lane:
    256 fp32 features per pass for the 16-row cells (27-point stencil on 100^3, N = 512: one
    pass of four-row groups 3.29 ms, two passes of 256 with cells 1.19 ms), 128 where 256 does not divide N."""
    want = 1
    if b_dtype == "f32":
        if feat_size % 256 == 0:
            want = feat_size // 256
        elif feat_size % 128 == 0:
            want = feat_size // 128
    return want if want in windows else min(windows)


def guess_num_partitions(g, feat_size: int, b_dtype: str = "f32") -> int:
    """Column-partition count for a single pass over the features, from the model
    (``predict_launch_shape`` with one window)."""
    return predict_launch_shape(g, feat_size, b_dtype, windows=(1,))[0]


def _window_candidates(feat_size: int, b_dtype: str) -> List[int]:
    """Feature-window counts worth timing: windows of at least 64 features (32-feature
    passes lost on every matrix measured) that the kernels support."""
    step = 64 if b_dtype == "bf16" else 32
    return [w for w in (1, 2, 4, 8) if feat_size % w == 0 and feat_size // w >= 64 and (feat_size // w) % step == 0] or [1]


def choose_launch_shape(g, feat_size: int, b_dtype: str = "f32", candidates: Sequence[int] = PARTITION_CANDIDATES,
                        windows: Sequence[int] = None, cost_model: str = "gfx950", runs: int = 5,
                        return_timings: bool = False):
    """Column-partition count and feature-window count by measurement: composes the format
    for every candidate partition count, times the fused kernel for every window count (a
    few runs each) and returns the pair (partitions, windows) with the fewest launches among
    those within 2 % of the fastest.  The fallback (and the yardstick) of
    ``predict_launch_shape``, which decides from a model in a fraction of the time."""
    torch = _torch()
    want = torch.float32 if b_dtype == "f32" else torch.bfloat16
    if windows is None:
        windows = _window_candidates(feat_size, b_dtype)
    # random operand: constant data lets the GPU clock higher and flatters every candidate
    B = (torch.rand((g.num_dst_nodes(), feat_size), dtype=torch.float32, device="cuda") - 0.5).to(want)
    Cout = torch.empty((g.num_src_nodes(), feat_size), dtype=torch.float32, device="cuda")
    timings = {}
    for p in candidates:
        try:
            cfg = search_bucket_config(g, p, CostModelSettings(feat_size, p, cost_model=cost_model))
        except ValueError:
            continue                      # a partition with a single nonzero: not a usable split
        fmt = build_hyb_format_device(g, cfg)
        for w in windows:
            plan = HybSpMM(fmt, feat_size, b_dtype, windows=w)
            try:
                timings[(p, w)] = float(np.median(plan.time_ms(B, Cout, warmup=2, repeat=runs)))
            finally:
                plan.close()
        del fmt
    if not timings:
        raise ValueError("no candidate partition count is usable for this matrix")
    best = pick_launch_shape(timings)
    return (best, timings) if return_timings else best


def choose_num_partitions(g, feat_size: int, b_dtype: str = "f32", candidates: Sequence[int] = PARTITION_CANDIDATES,
                          cost_model: str = "gfx950", runs: int = 5, return_timings: bool = False):
    """Column-partition count by measurement for a single pass over the features
    (choose_launch_shape with one window)."""
    best, timings = choose_launch_shape(g, feat_size, b_dtype, candidates, windows=(1,), cost_model=cost_model,
                                        runs=runs, return_timings=True)
    flat = {p: t for (p, _), t in timings.items()}
    return (best[0], flat) if return_timings else best[0]
