"""Matrix container for the CELL/hyb SpMM path.

Mirrors the interface of the reference's ``format_matrix_market`` module
(playground_pipline/format_matrix_market.py:12-205): ``Bucket`` is the cost-model
record, ``MTX`` wraps a ``scipy.sparse.coo_matrix`` and hands out CSR/CSC/COO views.
Anything that accepted a reference ``MTX`` accepts this one (same attribute and
method names, same return types).

Differences, all additive:
  * ``MTX.from_coo`` / ``MTX.from_csr`` build a matrix from arrays without a file and
    may keep real values (the reference forces every stored value to 1.0,
    format_matrix_market.py:54, 63-64);
  * the graph-dataset names of the reference need the ``dgl``/``ogb`` packages and a
    network connection; they raise ``RuntimeError`` here.
"""
from __future__ import annotations

import os
import sys
from os.path import basename, splitext

import numpy as np
from scipy import sparse as sp

__all__ = ["MTX", "Bucket"]

_GRAPH_DATASETS = ("cora", "citeseer", "pubmed", "ppi", "arxiv", "proteins", "reddit")


def _are_plain_triplets(row, col, data, shape):
    """Whether scipy would keep the arrays as they are: int32 indices inside the shape, one real value
    each.  (Anything else is left to scipy, which converts it or raises.)  One pass over either
    index array - a negative index is a large unsigned one - where scipy's constructor makes four."""
    if not (row.dtype == col.dtype == np.int32 and data.dtype in (np.float32, np.float64)):
        return False
    if not (row.ndim == col.ndim == data.ndim == 1 and 0 < len(row) == len(col) == len(data)):
        return False
    if not (isinstance(shape, tuple) and len(shape) == 2 and all(isinstance(n, (int, np.integer)) and 0 < n < 2**31 for n in shape)):
        return False
    return all(_inside(i, n) for i, n in zip((row, col), shape))


# Entries from which torch's threads are faster than one (us, one -> all, two arrays of as many entries: 100K 9 -> 17, 192K 15 -> 18,
# 400K 30 -> 19, 3M 223 -> 41).
_BY_THREADS = 1 << 18
_forked = {}                 # process id -> whether it is a fork that runs its parent's program


def _is_forked() -> bool:
    """Whether this process is a fork that has not started a program of its own.  The threads that its parent had are gone in
    it, and torch, which does not know, would wait for them for ever.  (The kernel's flag PF_FORKNOEXEC; unknown counts as one.)"""
    pid = os.getpid()
    if pid not in _forked:
        try:
            with open("/proc/self/stat") as stat:
                _forked[pid] = bool(int(stat.read().rpartition(")")[2].split()[6]) & 0x40)
        except (OSError, ValueError, IndexError):
            _forked[pid] = True
    return _forked[pid]


def _inside(index, n) -> bool:
    """Whether every entry of an int32 array is in [0, n); by torch's threads where the array is long and the process has
    them (a process that works with host arrays only does not load torch for this)."""
    if len(index) >= _BY_THREADS and index.flags.c_contiguous and index.flags.writeable and "torch" in sys.modules and not _is_forked():
        torch = sys.modules["torch"]
        lo, hi = torch.aminmax(torch.from_numpy(index))
        return 0 <= int(lo) and int(hi) < n
    return int(index.view(np.uint32).max()) < n


class Bucket:
    """One (partition, width) bucket as the cost model sees it
    (format_matrix_market.py:12-37)."""

    def __init__(self, bucket_width: int, num_rows: int, nnz: int,
                 row_indices: list, col_indices: set):
        self.bucket_width = bucket_width
        self.num_rows = num_rows
        self.nnz = nnz
        self.row_indices = row_indices
        self.col_indices = col_indices

    def __str__(self):
        head = (f"Bucket(bucket_width={self.bucket_width}, num_rows={self.num_rows}, "
                f"nnz={self.nnz}, len(row_indices)={len(self.row_indices)}, ")
        if len(self.row_indices) < 11 and len(self.col_indices) < 11:
            return (head + f"row_indices={self.row_indices}, "
                    f"len(col_indices)={len(self.col_indices)}, col_indices={self.col_indices})")
        return head + f"len(col_indices)={len(self.col_indices)})"


class MTX:
    """Sparse matrix held as scipy COO (format_matrix_market.py:40-205).

    ``MTX(None)`` gives an empty shell whose ``coo_mtx`` the caller assigns;
    ``MTX(path)`` reads a MatrixMarket file and sets every stored value to 1.
    """

    def __init__(self, filename):
        self._coo = None
        self._csr = None
        self._csr_source = None       # the CSR matrix this container was made from (from_csr), as given
        self._triplets = None         # (row, col, data, shape) this container was made from (from_coo)
        self._unit_values = False     # from_csr without data: every stored value is 1
        self._identity = object()     # replaced with the matrix: what a copy on the GPU is kept under
        if filename is None:
            self.name = None
        elif filename in _GRAPH_DATASETS:
            raise RuntimeError(
                f"dataset '{filename}' is downloaded through dgl/ogb in the reference; "
                "those loaders are not part of this library - build the matrix with "
                "MTX.from_coo / MTX.from_csr or pass a MatrixMarket path")
        else:
            from scipy.io import mmread
            self.name = splitext(basename(filename))[0]
            coo = sp.coo_matrix(mmread(filename))
            coo.data = np.ones(len(coo.data))          # format_matrix_market.py:63-64
            self.coo_mtx = coo

    # ``coo_mtx`` is the reference's one data attribute (format_matrix_market.py:44-46).  A
    # container made from CSR arrays or checked triplets keeps them and builds the COO view only
    # when it is asked for, so that they can go to the GPU as they are.  Whoever holds the view may
    # change it in place (sum_duplicates, eliminate_zeros, ``.data = ...``): once it has been handed
    # out it is the matrix, and the arrays it was built from are let go.
    @property
    def coo_mtx(self):
        coo = self._coo_view()
        self._forget_sources()
        return coo

    def _forget_sources(self):
        if self._csr is not None and self._csr is self._csr_source:
            self._csr = None
        self._csr_source = None
        self._triplets = None
        self._unit_values = False

    def _coo_view(self):
        """The COO view for use inside this class, where nothing is changed through it."""
        if self._coo is None:
            if self._csr_source is not None:
                self._coo = self._csr_source.tocoo()
            elif self._triplets is not None:
                row, col, data, shape = self._triplets
                self._coo = sp.coo_matrix((data, (row, col)), shape=shape)
        return self._coo

    @coo_mtx.setter
    def coo_mtx(self, value):
        self._coo = value
        self._csr = None                               # cached views follow the COO
        self._forget_sources()
        self._identity = object()

    # ---- constructors without a file -------------------------------------------------
    @classmethod
    def from_coo(cls, row, col, shape, data=None, name=None):
        m = cls(None)
        m.name = name
        row = np.asarray(row)
        col = np.asarray(col)
        if data is None:
            data = np.ones(len(row))
        data = np.asarray(data)
        if _are_plain_triplets(row, col, data, shape):
            m._triplets = (row, col, data, (int(shape[0]), int(shape[1])))
        else:
            m.coo_mtx = sp.coo_matrix((data, (row, col)), shape=shape)
        return m

    @classmethod
    def from_csr(cls, indptr, indices, shape, data=None, name=None):
        """Container around CSR arrays, kept as they are (no copy for int32 / float32 input).
        ``data=None`` stores ones, like every matrix of the reference."""
        indptr = np.asarray(indptr)
        indices = np.asarray(indices)
        unit = data is None
        if unit:
            data = np.ones(len(indices), dtype=np.float32)
        m = cls(None)
        m.name = name
        m._csr_source = sp.csr_matrix((np.asarray(data), indices, indptr), shape=shape)
        m._unit_values = unit
        return m

    # ---- the reference's accessors ----------------------------------------------------
    def _csr_view(self):
        """Canonical CSR (sorted columns, duplicates summed): what coo.tocsr() gives
        (format_matrix_market.py:74-76)."""
        if self._csr is None:
            src = self._csr_source
            if src is not None and src.has_canonical_format:
                self._csr = src
            else:
                self._csr = self._coo_view().tocsr()
        return self._csr

    def _shape(self):
        if self._coo is None and self._triplets is not None:
            return self._triplets[3]
        return (self._csr_source if self._coo is None and self._csr_source is not None else self._coo_view()).shape

    def adj_tensors(self, format: str):
        if format == "coo":
            return self.coo_mtx.row, self.coo_mtx.col
        elif format == "csc":
            csc = self._coo_view().tocsc()
            return csc.indptr, csc.indices, csc.data
        elif format == "csr":
            csr = self._csr_view()
            return csr.indptr, csr.indices, csr.data
        raise TypeError(f"Format {format} is not suppoted.")

    def num_src_nodes(self):
        return self._shape()[0]

    def num_dst_nodes(self):
        return self._shape()[1]

    def num_edges(self):
        # stored entries: the COO view of a CSR matrix holds exactly its stored entries
        if self._coo is None and self._csr_source is not None:
            return self._csr_source.nnz
        if self._coo is None and self._triplets is not None:
            return len(self._triplets[2])
        return self._coo_view().nnz

    def dot(self, B):
        """A @ B through scipy (format_matrix_market.py:89-99)."""
        return self._coo_view().tocsc().dot(B)

    def tobsr(self, blocksize=None, copy=False):
        """scipy BSR view (format_matrix_market.py:101-112)."""
        return self._coo_view().tobsr(blocksize=blocksize, copy=copy)

    def tobsr_with_padding(self, shape, blocksize=None):
        """BSR matrix of the given (padded) shape with fp16-valued entries, shape % blocksize == 0
        (format_matrix_market.py:115-136).  The reference stores the values as float16; scipy
        1.15 no longer accepts that dtype in sparse containers, so the values are rounded to
        fp16 and held as float32 (every value is exactly representable in fp16)."""
        data = np.array(self._coo_view().data, dtype=np.float16).astype(np.float32)
        ij = [self._coo_view().row, self._coo_view().col]
        return sp.bsr_matrix((data, ij), blocksize=blocksize, shape=shape)

    def tocsr(self, copy=False):
        return self._coo_view().tocsr(copy=copy)

    def matrix_features(self):
        """Row-length statistics used by the format selector
        (format_matrix_market.py:153-202)."""
        num_rows, num_cols = self._shape()
        indptr = self._csr_view().indptr
        per_row = np.diff(indptr)
        avg = np.mean(per_row)
        lo = per_row.min()
        hi = per_row.max()
        return {
            "name": self.name,
            "num_rows": num_rows,
            "num_cols": num_cols,
            "nnz": self.num_edges(),
            "avg_nnz_per_row": avg,
            "min_nnz_per_row": lo,
            "max_nnz_per_row": hi,
            "std_dev_nnz_per_row": np.std(per_row),
            "avg_nnz_density_per_row": avg / num_cols,
            "min_nnz_density_per_row": lo / num_cols,
            "max_nnz_density_per_row": hi / num_cols,
            "std_dev_nnz_density_per_row": np.std(per_row / num_cols),
        }

    def __str__(self):
        return str(self._coo_view())
