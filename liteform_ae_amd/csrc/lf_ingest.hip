// COO -> canonical CSR on the GPU: sort by (row, column), add up duplicate entries, build
// the row pointer.  This is what the reference's matrix container does on the host every
// time a CSR view is asked for (playground_pipline/format_matrix_market.py:74-76:
// scipy's coo.tocsr(), which sorts columns and sums duplicates); it is the step that feeds
// lf_bucket_stats / lf_hyb_build.  Up to 8.4 million entries go through bins of rows that are sorted in LDS, a kernel each
// for counting, offsets, distribution and sorting, and three more that add up duplicates; more of them, bins that do not
// fit and entries outside the matrix through plain library
// primitives (rocPRIM radix sort and reduce-by-key on a 64-bit key row * cols + col), with kernels
// that pack / unpack keys and locate the row boundaries.
//
// Also here: the structural check of CSR arrays that come from a caller (lf_csr_check), which
// every entry point that gathers through caller-supplied CSR or BSR index arrays runs first,
// and which tells an already canonical CSR (the fast path: no sort) from one that has to go
// through the COO route.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_reduce_by_key.hpp>
#include <rocprim/functional.hpp>

#include "lf_internal.h"
#include "lf_spmm_device.h"

namespace {

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

__global__ void pack_keys_kernel(const int32_t* __restrict__ row, const int32_t* __restrict__ col,
                                 const float* __restrict__ val, long long nnz, long long cols,
                                 unsigned long long* __restrict__ keys, float* __restrict__ vals, int* __restrict__ longest) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *longest = 0;     // for row_pointer_kernel
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < nnz;
         i += (long long)gridDim.x * blockDim.x) {
        keys[i] = (unsigned long long)row[i] * (unsigned long long)cols + (unsigned long long)col[i];
        vals[i] = val ? val[i] : 1.0f;
    }
}

__global__ void unpack_cols_kernel(const unsigned long long* __restrict__ keys, const int* __restrict__ n_unique,
                                   long long cols, int32_t* __restrict__ indices) {
    const long long n = *n_unique;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        indices[i] = (int32_t)(keys[i] % (unsigned long long)cols);
}

// indptr[r] = number of unique keys below r * cols (keys are sorted).  A workgroup's last row is the next one's first, so that it
// knows the lengths of all but that one.
constexpr int kPointerThreads = 256, kPointerRows = kPointerThreads - 1;
__global__ void __launch_bounds__(kPointerThreads)
row_pointer_kernel(const unsigned long long* __restrict__ keys, const int* __restrict__ n_unique,
                   long long rows, long long cols, int32_t* __restrict__ indptr, int* __restrict__ longest) {
    __shared__ int s_first[kPointerThreads];
    const long long r = (long long)blockIdx.x * kPointerRows + threadIdx.x;
    long long lo = 0, hi = *n_unique;
    const unsigned long long bound = (unsigned long long)min(r, rows) * (unsigned long long)cols;
    while (lo < hi) {
        const long long mid = (lo + hi) >> 1;
        if (keys[mid] < bound) lo = mid + 1; else hi = mid;
    }
    if (r <= rows) indptr[r] = (int32_t)lo;
    s_first[threadIdx.x] = (int)lo;
    __syncthreads();
    int most = threadIdx.x < kPointerRows ? s_first[threadIdx.x + 1] - (int)lo : 0;
    for (int d = 32; d > 0; d >>= 1) most = max(most, __shfl_xor(most, d));
    if ((threadIdx.x & 63) == 0 && most > __hip_atomic_load(longest, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(longest, most);
}

// ---- bins of rows sorted in LDS
// A bin is 2^lg_rows consecutive rows, an entry in it one word - row in the bin, column - and its value.  Entries are
// distributed to their bins (unordered within one), a workgroup then sorts a bin in LDS and writes its part of the
// arrays and of the row pointer.  Bound by launches and by the latency of each kernel's two or three dependent passes.
// With the wait for the flags, us, the library's sort with the kernels around it -> this: 6K entries 65 -> 42, 64K 79 -> 45,
// 300K 165 -> 55, 860K of a power-law graph (a row of 41,000) 234 -> 134, 1.6M 201 -> 79, 4M 350 -> 180, 7.8M 571 -> 340;
// with a duplicate 61 -> 68, 80 -> 72, 165 -> 86, 228 -> 214, 202 -> 130, 349 -> 266, 578 -> 535.  Rows in the order of their
// lengths, so that the first bins are large: 1.6M 204 -> 104, 4M 349 -> 213, 7.8M 573 -> 443.  Where the sort has to be
// taken after all, counting and the wait are lost: 600K 208 -> 239, 2.4M 293 -> 338, 5M 472 -> 566, 7.6M 565 -> 666.
// Beyond 8.4M entries bins outgrow the LDS, and the sort's few passes over memory are what counts.
// flags: [kNotHere] an entry outside the matrix or bins of too many, known before anything is distributed, and
// [kCrowded] a long row with too many of its columns beside each other: the other way has to be taken; [kReads] windows
// that large bins' parts will read; [kLargeParts] parts left to bin_sort_large_kernel; [kTwice] entries that are to be
// added to another one of their place.  From [kLongest] on: entries of the longest row of every bin, of which bin_report_kernel takes the
// largest (an atomic of every bin on one word was 7 - 13 us).
constexpr int kNotHere = 0, kReads = 1, kCrowded = 2, kLargeParts = 3, kTwice = 4, kFlags = 5, kLongest = kFlags;
constexpr int kBinThreads = 512;
constexpr int kBinChunk = 4096;            // entries that a workgroup distributes at least
constexpr int kBinMaxChunks = 1024;
constexpr int kBinRowMost = 4096;          // entries in a row on average: a few long rows are a few bins' work (3 rows of
                                           // 16,000: 109 us, the other way 75)
constexpr int kBinMost = 4096;             // bins: counters and bases in LDS
constexpr int kBinLgRows = 9;              // rows of a bin: the same
constexpr int kBinFew = 128, kBinUsual = 1024;     // entries in a bin on average: the first up to kBinUsual bins, then the
constexpr int kBinTargetMost = 2048;               // second, and this at most
constexpr int kBinSmall = 4096;            // entries sorted in 48 KB of LDS
constexpr int kBinLarge = 8192;            // ... in 96 KB, a part of a larger bin at a time
constexpr int kBinWindow = kBinLarge / 2;  // parts of a large bin: every kBinWindow entries
// Each part reads all of its bin: windows of a bin at most, and windows read in all for every kBinWindow entries of the
// matrix, beyond one bin of the most.  Us, the library's sort -> with such bins: 520K entries, 120K of them in
// one bin 190 -> 203; 7.8M, 1.2 windows read for each 570 -> 442; 7.6M in 60 bins of 120K, 29 for each 562 -> 1393.
constexpr int kBinMostWindows = 32, kBinReadsMost = 6;
constexpr int kBinLargeBytes = 3 * 4 * kBinLarge;
constexpr int kBinLargeGrid = 256;

struct BinShape {
    int lg_rows, lg_cols, bins, chunks, per_chunk, most_reads;     // bins == 0: too large, or more than 32 bits to an entry
    size_t counts, totals, bases, list, flags, records, twice, before, partial, total;
};

BinShape bin_shape(long long nnz, long long rows, long long cols) {
    BinShape b{};
    if (nnz <= 0 || rows <= 0 || cols <= 0 || nnz > (long long)kBinMost * kBinTargetMost || nnz / rows > kBinRowMost) return b;
    while ((1ll << b.lg_cols) < cols) ++b.lg_cols;
    const long long by_entries = std::max<long long>(nnz / kBinUsual, std::min<long long>(nnz / kBinFew, kBinUsual));
    const long long want = std::min<long long>(kBinMost, std::max<long long>(by_entries, (rows >> kBinLgRows) + 1));
    while ((rows + (1ll << b.lg_rows) - 1) >> b.lg_rows > want) ++b.lg_rows;
    if (b.lg_rows + b.lg_cols > 31 || b.lg_rows > kBinLgRows) return b;      // (the largest key fills up a sort)
    b.bins = (int)((rows + (1ll << b.lg_rows) - 1) >> b.lg_rows);
    b.per_chunk = (int)align_up((size_t)std::max<long long>(kBinChunk, (nnz + kBinMaxChunks - 1) / kBinMaxChunks), kBinThreads);
    b.chunks = (int)((nnz + b.per_chunk - 1) / b.per_chunk);
    b.most_reads = kBinMostWindows * kBinMostWindows + kBinReadsMost * (int)(nnz / kBinWindow);
    size_t off = 0;
    b.records = off; off += align_up((size_t)nnz * 8, 256);
    b.counts = off; off += align_up((size_t)b.bins * b.chunks * 4, 256);
    b.totals = off; off += align_up((size_t)b.bins * 4, 256);
    b.bases = off; off += align_up((size_t)b.bins * 4, 256);
    b.list = off; off += align_up((size_t)(nnz / kBinWindow + b.bins) * 4, 256);
    b.flags = off; off += align_up((size_t)(kLongest + b.bins) * 4, 256);
    b.twice = off; off += align_up((size_t)nnz * 4, 256);
    b.before = off; off += align_up((size_t)(nnz + 1) * 4, 256);
    b.partial = off; off += align_up((size_t)(nnz / 1024 + 2) * 4, 256);
    b.total = off;
    return b;
}

__device__ __forceinline__ bool in_matrix(int row, int col, long long rows, long long cols) {
    return (unsigned long long)(unsigned)row < (unsigned long long)rows && (unsigned long long)(unsigned)col < (unsigned long long)cols;
}

// counter[i] += 1 for every active lane; what it held before, the lanes in their order.  To be called by whole wavefronts.
// Lanes of one counter are taken one after the other by the LDS, and a power-law graph's longest row is most of its bin:
// the first lanes' counters are served with one atomic for all that share them (760K entries with a row of 13,000,
// sorting 79 -> 22 us together with the buckets).
__device__ __forceinline__ int count_up(int* counter, int i, bool active) {
    const int lane = threadIdx.x & 63;
    int before = 0;
#pragma unroll
    for (int round = 0; round < 2; ++round) {
        const unsigned long long left = __ballot(active);
        if (left == 0) return before;
        const int leader = __builtin_ctzll(left);
        const bool same = active && i == __builtin_amdgcn_readlane(i, leader);
        const unsigned long long shared = __ballot(same);
        int first = 0;
        if (lane == leader) first = atomicAdd(&counter[i], __popcll(shared));
        first = __builtin_amdgcn_readlane(first, leader);
        if (same) {
            before = first + __popcll(shared & ((1ull << lane) - 1ull));
            active = false;
        }
    }
    if (active) before = atomicAdd(&counter[i], 1);
    return before;
}

// counts[bin][chunk]: entries of a chunk (blockIdx.x) in a bin
__global__ void __launch_bounds__(kBinThreads)
bin_count_kernel(const int32_t* __restrict__ row, const int32_t* __restrict__ col, long long nnz, long long rows, long long cols,
                 int lg_rows, int bins, int per_chunk, int* __restrict__ counts, int* __restrict__ flags) {
    __shared__ int s_count[kBinMost];
    for (int i = threadIdx.x; i < bins; i += kBinThreads) s_count[i] = 0;
    __syncthreads();
    const long long lo = (long long)blockIdx.x * per_chunk, hi = min(lo + per_chunk, nnz);
    bool bad = false;
    for (long long i0 = lo; i0 < hi; i0 += kBinThreads) {
        const long long i = i0 + threadIdx.x;
        const int r = i < hi ? row[i] : -1;
        const bool ok = i < hi && in_matrix(r, col[i], rows, cols);
        bad |= i < hi && !ok;
        count_up(s_count, r >> lg_rows, ok);
    }
    if (__ballot(bad) != 0 && (threadIdx.x & 63) == 0) flags[kNotHere] = 1;
    __syncthreads();
    for (int i = threadIdx.x; i < bins; i += kBinThreads) counts[(size_t)i * gridDim.x + blockIdx.x] = s_count[i];
}

// A wavefront to a bin: its counts become the chunks' offsets in it, totals[bin] their sum.
__global__ void __launch_bounds__(256)
bin_offsets_kernel(int* __restrict__ counts, int bins, int chunks, int* __restrict__ totals, int most_reads, int* __restrict__ flags) {
    const int bin = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (bin >= bins) return;
    int* mine = counts + (size_t)bin * chunks;
    int before = 0;
    for (int c0 = 0; c0 < chunks; c0 += 64) {
        const int x = c0 + lane < chunks ? mine[c0 + lane] : 0;
        int incl = x;
        for (int d = 1; d < 64; d <<= 1) {
            const int y = __shfl_up(incl, d);
            if (lane >= d) incl += y;
        }
        if (c0 + lane < chunks) mine[c0 + lane] = before + incl - x;
        before += __shfl(incl, 63);
    }
    if (lane == 0) totals[bin] = before;
    if (lane == 0 && before > kBinSmall) {
        const int windows = (before + kBinWindow - 1) / kBinWindow, reads = windows * windows;
        if (windows > kBinMostWindows || atomicAdd(&flags[kReads], reads) + reads > most_reads) flags[kNotHere] = 1;
    }
}

// Distributes a chunk's entries.  Every workgroup scans the bins' totals for itself; the first leaves the bases.
__global__ void __launch_bounds__(kBinThreads)
bin_distribute_kernel(const int32_t* __restrict__ row, const int32_t* __restrict__ col, const float* __restrict__ val, long long nnz,
                      long long rows, long long cols, int lg_rows, int lg_cols, int bins, int per_chunk,
                      const int* __restrict__ counts, const int* __restrict__ totals, int* __restrict__ bases,
                      uint2* __restrict__ records, const int* __restrict__ flags) {
    __shared__ int s_at[kBinMost];
    __shared__ int s_wave[kBinThreads / 64];
    constexpr int kPer = kBinMost / kBinThreads;           // consecutive bins of a thread
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, b0 = threadIdx.x * kPer;
    const int not_here = flags[kNotHere];
    int sum = 0;
    for (int i = b0; i < min(b0 + kPer, bins); ++i) sum += totals[i];
    int incl = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(incl, d);
        if (lane >= d) incl += y;
    }
    if (not_here) return;
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    int base = incl - sum;
    for (int w = 0; w < wave; ++w) base += s_wave[w];
    for (int i = b0; i < min(b0 + kPer, bins); ++i) {
        s_at[i] = base + counts[(size_t)i * gridDim.x + blockIdx.x];
        if (blockIdx.x == 0) bases[i] = base;
        base += totals[i];
    }
    __syncthreads();
    const long long lo = (long long)blockIdx.x * per_chunk, hi = min(lo + per_chunk, nnz);
    const int row_mask = (1 << lg_rows) - 1;
    for (long long i0 = lo; i0 < hi; i0 += kBinThreads) {
        const long long i = i0 + threadIdx.x;
        const int r = i < hi ? row[i] : -1, c = i < hi ? col[i] : -1;
        const float v = i < hi && val ? val[i] : 1.0f;
        const bool ok = in_matrix(r, c, rows, cols);       // (others are flagged, and none of this runs)
        const int at = count_up(s_at, r >> lg_rows, ok);
        if (ok) records[at] = make_uint2(((unsigned)(r & row_mask) << lg_cols) | (unsigned)c, __float_as_uint(v));
    }
}

// Inclusive scan of a workgroup's values; s_wave: a word per wavefront.
template <int THREADS> __device__ __forceinline__ int scan_workgroup(int x, int* s_wave) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    for (int w = 0; w < wave; ++w) x += s_wave[w];
    __syncthreads();
    return x;
}

struct BinSort {
    const uint2* records;
    const int *bases, *totals;
    long long rows;
    int lg_rows, lg_cols;
    unsigned inverse;                          // 2^32 / columns: a column's place among them as a 32-bit fraction
    int32_t *indptr, *indices;
    float* values;
    int *list, *flags;
};

// One bin.  The rows are counted, which gives the row pointer.  A row of len entries then has len buckets, the i-th for
// the i-th part of the columns: counting puts its entries together bucket by bucket (s_key, s_val), and an entry's
// place follows from the few of its bucket, equal keys by value.  Where the columns of rows crowd into few buckets
// (more than kBucketReads reads an entry) the part is sorted bitonically.
// (Comparing an entry with its whole row: 57K rows of 28 entries 72 us for this kernel, 760K entries of a power-law
// graph 79; so 25 and 22.)
// LARGE: a part of a bin, the `window`-th kBinWindow of its sorted entries.  The rows that start in it and have no more than
// that are at most 2 * kBinWindow - 1 entries.  A longer row is cut into as many ranges of columns as windows start inside
// it, a window to a range.
constexpr int kBinRows = 1 << kBinLgRows;
constexpr int kBucketReads = 64;
template <int THREADS, int CAPACITY, bool LARGE>
__device__ __forceinline__ void sort_bin(const BinSort& a, int bin, int window, unsigned* s_key, unsigned* s_val, int* s_bucket, int* s_wave) {
    __shared__ int s_first[kBinRows];          // of a row in the bin; not sorted here: -1
    __shared__ int s_count[kBinRows];
    __shared__ int s_from, s_long, s_long_at, s_before, s_sorted, s_most;
    __shared__ float s_squares;
    constexpr int kOwn = LARGE ? 16 : CAPACITY / THREADS;  // records in registers: usually all, loaded once
    const int base = a.bases[bin], n = a.totals[bin];
    const long long r0 = (long long)bin << a.lg_rows;
    const int n_rows = (int)min(1ll << a.lg_rows, a.rows - r0);
    const unsigned col_mask = (unsigned)((1ull << a.lg_cols) - 1);
    const uint2* records = a.records + base;
    uint2 own[kOwn];
    auto load = [&](int from) {
#pragma unroll
        for (int k = 0; k < kOwn; ++k) {
            const int i = from + k * THREADS + (int)threadIdx.x;
            own[k] = i < n ? records[i] : make_uint2(0, 0);
        }
    };
    const bool once = !LARGE || n <= kOwn * THREADS;
    if (once) load(0);
    auto each = [&](auto use) {                            // use(record, is there one), by whole wavefronts
        for (int from = 0; from < (once ? 1 : n); from += kOwn * THREADS) {
            if (!once) load(from);
#pragma unroll
            for (int k = 0; k < kOwn; ++k)
                if (from + k * THREADS < n) use(own[k], from + k * THREADS + (int)threadIdx.x < n);
        }
    };
    auto fraction = [&](unsigned key) { return (key & col_mask) * a.inverse; };      // (below 2^32: column < columns)
    int repeats = 0;                                       // entries behind another one of their place
    bool crowded = false;
    // The records that `selected` takes: by bucket(key), which ascends with the key, and then in full; out(key, place)
    // is where the place-th goes.  More than CAPACITY are too many.
    auto sort_part = [&](auto selected, auto bucket, auto out) {
        constexpr int kPer = CAPACITY / THREADS;
        for (int i = threadIdx.x; i < CAPACITY; i += THREADS) s_bucket[i] = 0;
        if (threadIdx.x == 0) s_squares = 0.f;
        __syncthreads();
        each([&](const uint2& x, bool in) {
            if (in && selected(x.x)) atomicAdd(&s_bucket[bucket(x.x)], 1);
        });
        __syncthreads();
        int sum = 0;
        float squares = 0.f;
        for (int k = 0; k < kPer; ++k) {
            const int x = s_bucket[threadIdx.x * kPer + k];
            sum += x;
            squares += (float)x * (float)x;
        }
        const int upto = scan_workgroup<THREADS>(sum, s_wave);
        int before = upto - sum;
        for (int k = 0; k < kPer; ++k) {
            const int x = s_bucket[threadIdx.x * kPer + k];
            s_bucket[threadIdx.x * kPer + k] = before;
            before += x;
        }
        if (squares > 0.f) atomicAdd(&s_squares, squares);
        if (threadIdx.x == THREADS - 1) s_sorted = upto;
        __syncthreads();
        const int sorted = s_sorted;
        if (sorted > CAPACITY) {
            crowded = true;
            return;
        }
        each([&](const uint2& x, bool in) {
            if (!in || !selected(x.x)) return;
            const int to = atomicAdd(&s_bucket[bucket(x.x)], 1);   // (and becomes the bucket's end)
            s_key[to] = x.x;
            s_val[to] = x.y;
        });
        __syncthreads();
        if (s_squares <= (float)sorted * kBucketReads) {
            for (int i = threadIdx.x; i < sorted; i += THREADS) {
                const unsigned key = s_key[i], val = s_val[i];
                const int q = bucket(key), first = q > 0 ? s_bucket[q - 1] : 0, end = s_bucket[q];
                int place = first, ahead = 0;
                for (int j = first; j < end; ++j) {
                    const unsigned other = s_key[j];
                    place += other < key;
                    if (other == key && j != i) ahead += s_val[j] < val || (s_val[j] == val && j < i);    // by value, then as they lie here
                }
                place += ahead;
                repeats += ahead > 0;
                const int to = out(key, place);
                a.indices[to] = (int32_t)(key & col_mask);
                a.values[to] = __uint_as_float(val);
            }
        } else {
            int padded = 64;
            while (padded < sorted) padded <<= 1;
            for (int i = sorted + threadIdx.x; i < padded; i += THREADS) s_key[i] = s_val[i] = ~0u;
            __syncthreads();
            for (int size = 2; size <= padded; size <<= 1)
                for (int stride = size >> 1; stride > 0; stride >>= 1) {
                    for (int p = threadIdx.x; p < padded >> 1; p += THREADS) {
                        const int i = ((p & ~(stride - 1)) << 1) | (p & (stride - 1)), j = i + stride;
                        const unsigned ki = s_key[i], kj = s_key[j], vi = s_val[i], vj = s_val[j];
                        if ((ki > kj || (ki == kj && vi > vj)) == ((i & size) == 0)) {
                            s_key[i] = kj;
                            s_key[j] = ki;
                            s_val[i] = vj;
                            s_val[j] = vi;
                        }
                    }
                    __syncthreads();
                }
            for (int i = threadIdx.x; i < sorted; i += THREADS) {
                const unsigned key = s_key[i];
                const int to = out(key, i);
                a.indices[to] = (int32_t)(key & col_mask);
                a.values[to] = __uint_as_float(s_val[i]);
                repeats += i > 0 && s_key[i - 1] == key;
            }
        }
    };

    for (int r = threadIdx.x; r < n_rows; r += THREADS) s_count[r] = 0;
    if (threadIdx.x == 0) s_most = 0;
    if (LARGE && threadIdx.x == 0) {
        s_from = n;
        s_long = -1;
        s_before = 0;
    }
    __syncthreads();
    each([&](const uint2& x, bool in) { count_up(s_count, (int)(x.x >> a.lg_cols), in); });
    __syncthreads();
    // a thread's consecutive rows
    const int per = (n_rows + THREADS - 1) / THREADS, lo = min((int)threadIdx.x * per, n_rows), hi = min(lo + per, n_rows);
    int sum = 0, most = 0;
    for (int r = lo; r < hi; ++r) {
        sum += s_count[r];
        most = max(most, s_count[r]);
    }
    int at = scan_workgroup<THREADS>(sum, s_wave) - sum;
    for (int r = lo; r < hi; ++r) {
        const int len = s_count[r];
        const bool starts = !LARGE || min(at, n - 1) / kBinWindow == window;       // (empty rows behind the last entry: with it)
        if (starts) a.indptr[r0 + r] = base + at;
        const bool mine = starts && (!LARGE || len <= kBinWindow);
        s_first[r] = mine ? at : -1;
        if (LARGE && mine && len > 0) atomicMin(&s_from, at);
        if (LARGE && len > kBinWindow && at < window * kBinWindow && at + len > window * kBinWindow) {       // one at most
            s_long = r;
            s_long_at = at;
        }
        at += len;
    }
    if (r0 + n_rows == a.rows && threadIdx.x == THREADS - 1) a.indptr[a.rows] = base + n;
    if (__ballot(most > 0) != 0) {                         // (an atomic of every lane on one word is 64 rounds)
        for (int d = 32; d > 0; d >>= 1) most = max(most, __shfl_xor(most, d));
        if ((threadIdx.x & 63) == 0) atomicMax(&s_most, most);
    }
    __syncthreads();
    if (threadIdx.x == 0) a.flags[kLongest + bin] = s_most;        // (every window of a large bin the same)
    const int first = LARGE ? s_from : 0;                  // in the bin, of what is sorted together
    sort_part([&](unsigned key) { return !LARGE || s_first[key >> a.lg_cols] >= 0; },
              [&](unsigned key) {
                  const int r = (int)(key >> a.lg_cols);
                  return s_first[r] - first + (int)__umulhi(fraction(key), (unsigned)s_count[r]);
              },
              [&](unsigned, int place) { return base + first + place; });
    if (LARGE && s_long >= 0) {
        const unsigned row = (unsigned)s_long;
        const int row_at = s_long_at;
        __syncthreads();                                   // the rows have been read out
        const unsigned before = (unsigned)(row_at / kBinWindow) + 1, k = (unsigned)window - before;
        const unsigned ranges = (unsigned)((row_at + s_count[row] - 1) / kBinWindow) + 1 - before;
        auto scaled = [&](unsigned key) { return (unsigned long long)fraction(key) * ranges; };
        int lower = 0;
        each([&](const uint2& x, bool in) { lower += in && x.x >> a.lg_cols == row && scaled(x.x) >> 32 < k; });
        if (lower > 0) atomicAdd(&s_before, lower);
        sort_part([&](unsigned key) { return key >> a.lg_cols == row && scaled(key) >> 32 == k; },
                  [&](unsigned key) { return (int)__umulhi((unsigned)scaled(key), CAPACITY); },
                  [&](unsigned, int place) { return base + row_at + s_before + place; });
    }
    if (__ballot(repeats > 0) != 0) {
        for (int d = 32; d > 0; d >>= 1) repeats += __shfl_xor(repeats, d);
        if ((threadIdx.x & 63) == 0) atomicAdd(&a.flags[kTwice], repeats);
    }
    if (__ballot(crowded) != 0 && (threadIdx.x & 63) == 0) a.flags[kCrowded] = 1;
}

__global__ void __launch_bounds__(kBinThreads)
bin_sort_kernel(BinSort a) {
    __shared__ unsigned s_key[kBinSmall], s_val[kBinSmall];
    __shared__ int s_bucket[kBinSmall];
    __shared__ int s_wave[kBinThreads / 64];
    const int n = a.totals[blockIdx.x];
    if (a.flags[kNotHere]) return;
    if (n > kBinSmall) {
        const int windows = (n + kBinWindow - 1) / kBinWindow;
        if (threadIdx.x < 64) {
            int at = 0;
            if (threadIdx.x == 0) at = atomicAdd(&a.flags[kLargeParts], windows);
            at = __builtin_amdgcn_readfirstlane(at);
            for (int i = threadIdx.x; i < windows; i += 64) a.list[at + i] = (int)blockIdx.x | i * kBinMost;
        }
        return;
    }
    sort_bin<kBinThreads, kBinSmall, false>(a, blockIdx.x, 0, s_key, s_val, s_bucket, s_wave);
}

__global__ void __launch_bounds__(1024)
bin_sort_large_kernel(BinSort a) {
    extern __shared__ unsigned s_large[];                  // [3][kBinLarge]: keys, values, buckets
    __shared__ int s_wave[16];
    const int n = a.flags[kLargeParts];
    for (int i = blockIdx.x; i < n; i += gridDim.x) {
        const int item = a.list[i];
        __syncthreads();                                   // the part before has been read out
        sort_bin<1024, kBinLarge, true>(a, item % kBinMost, item / kBinMost, s_large, s_large + kBinLarge, (int*)(s_large + 2 * kBinLarge), s_wave);
    }
}

// The flags, and in [kLongest] the entries of the longest row of all bins: to `out`, which may be the host's.
__global__ void __launch_bounds__(256)
bin_report_kernel(const int* __restrict__ flags, int bins, int* out) {
    __shared__ int s_most[4];
    int most = 0;
    for (int i = threadIdx.x; i < bins; i += 256) most = max(most, flags[kLongest + i]);
    for (int d = 32; d > 0; d >>= 1) most = max(most, __shfl_xor(most, d));
    if ((threadIdx.x & 63) == 0) s_most[threadIdx.x >> 6] = most;
    __syncthreads();
    if (threadIdx.x < kFlags) out[threadIdx.x] = flags[threadIdx.x];
    if (threadIdx.x == kFlags) out[kLongest] = max(max(s_most[0], s_most[1]), max(s_most[2], s_most[3]));
}

// ---- duplicates in the sorted arrays: marked, counted up to every entry, and added up into its first.  They lie in the
// order of the sort, by value, in which a float sum is the worst there is (300 values of U(-1, 1): 2.2e-5 off, in any
// order some 3e-6): the sums are taken in 64 bits and rounded once.  A run of more than kSerialTwice is a wavefront's, 64 at a
// time: a thread's chain of loads over 8000 entries of one place is longer than everything else here.
__global__ void __launch_bounds__(256)
mark_twice_kernel(const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices, long long nnz, long long rows, int32_t* __restrict__ twice) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= nnz) return;
    bool same = i > 0 && indices[i - 1] == indices[i];
    if (same) {                                            // or the first of its row?
        long long lo = 0, hi = rows;
        while (lo < hi) {
            const long long mid = (lo + hi) >> 1;
            if (indptr[mid] < i) lo = mid + 1; else hi = mid;
        }
        same = indptr[lo] != i;
    }
    twice[i] = same;
}

constexpr int kSerialTwice = 16;
__global__ void __launch_bounds__(256)
add_up_kernel(const int32_t* __restrict__ indices, const float* __restrict__ values, const int32_t* __restrict__ twice,
              const int32_t* __restrict__ before, long long nnz, int32_t* __restrict__ out_indices, float* __restrict__ out_values) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const bool first = i < nnz && !twice[i];
    double sum = first ? values[i] : 0.0;
    long long j = i + 1;
    bool more = first && j < nnz && twice[j];
    for (int k = 0; k < kSerialTwice && more; ++k) {
        sum += values[j];
        ++j;
        more = j < nnz && twice[j];
    }
    for (unsigned long long left = __ballot(more); left != 0; left &= left - 1) {
        const int leader = __builtin_ctzll(left);
        long long at = __shfl(j, leader);
        double part = 0.0;
        for (int n = 64; n == 64; at += n) {
            const long long mine = at + lane;
            const unsigned long long ends = __ballot(mine >= nnz || !twice[mine]);
            n = ends != 0 ? __builtin_ctzll(ends) : 64;
            if (lane < n) part += values[mine];
        }
        for (int d = 32; d > 0; d >>= 1) part += __shfl_xor(part, d);
        if (lane == leader) sum += part;
    }
    if (!first) return;
    const long long to = i - before[i];
    out_indices[to] = indices[i];
    out_values[to] = (float)sum;
}

// The rows' starts, and the entries back into the caller's arrays (one launch where two copies of the runtime's were 12 us).
__global__ void __launch_bounds__(256)
close_up_kernel(int32_t* __restrict__ indptr, const int32_t* __restrict__ before, long long rows, long long nnz, const int32_t* __restrict__ from_indices,
                const float* __restrict__ from_values, int32_t* __restrict__ indices, float* __restrict__ values) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i <= rows) indptr[i] -= before[indptr[i]];
    if (i < nnz - before[nnz]) {
        indices[i] = from_indices[i];
        values[i] = from_values[i];
    }
}

__global__ void clear_words_kernel(int* __restrict__ p, int n) {
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0;
}

// One pass over the row pointer and one over the column indices.  out[0] is raised for
// anything a gather must not meet: a row pointer that does not start at 0, decreases, or
// does not end at nnz, or a column outside [0, num_cols).  out[1] counts the positions i > 0
// with indices[i] <= indices[i - 1] ("descents"), out[2] the non-empty rows whose first
// entry is such a position: the columns of every row ascend strictly (sorted, no
// duplicates) exactly when the two counts are equal.  out[3] is raised when a value differs
// from 1 (values == nullptr: not looked at).  That is bit 0 of out[0] and out[3]; above it are sums over every
// `sample_stride`-th row with entries in it or the three rows behind it: of the columns between the least first and the
// largest last one, in kSpanUnits of all, and of ones.  *longest (optional): the entries of the longest row.
// Bound by the two streams (8 bytes an entry).  81M entries with values: 2.25 ms with one atomic
// per wavefront and counter (65K updates of one cache line), 0.29 ms with one per workgroup of a
// grid that is resident at once, and 16-byte loads.
constexpr int kCheckGrid = 2048;       // 8 workgroups on each of 256 CUs
constexpr int kSpanUnits = 4096, kSpanSamples = 1024;      // (twice the samples at most: sums below 2^24)
// four consecutive 32-bit values at a 4-byte aligned address (one 16-byte load)
struct __attribute__((packed, aligned(4))) Packed4i { int x, y, z, w; };
struct __attribute__((packed, aligned(4))) Packed4f { float x, y, z, w; };
__global__ void __launch_bounds__(256)
csr_check_kernel(const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices,
                 const float* __restrict__ values, long long rows, long long cols, long long nnz, int sample_stride,
                 unsigned int* __restrict__ out, int* __restrict__ longest) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    const long long t0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    int most = 0;
    bool bad = false, not_one = false;
    unsigned int descents = 0, boundary = 0, span = 0, samples = 0;
    for (long long r = t0; r < rows; r += stride) {
        const long long lo = indptr[r], hi = indptr[r + 1];
        bad |= lo < 0 || hi < lo || hi > nnz;
        most = max(most, (int)(hi - lo));
        if (r == 0) bad |= lo != 0;
        if (r == rows - 1) bad |= hi != nnz;
        if (hi > lo && lo > 0 && lo < nnz && indices[lo] <= indices[lo - 1]) ++boundary;
        if ((unsigned)r % (unsigned)sample_stride == 0) {
            int first = 0x7FFFFFFF, last = -1;
            for (long long q = r; q < min(r + 4, rows); ++q) {
                const long long from = indptr[q], to = indptr[q + 1];
                if (from < 0 || from >= to || to > nnz) continue;
                first = min(first, indices[from]);
                last = max(last, indices[to - 1]);
            }
            if (last >= first) {
                span += (unsigned int)min((long long)kSpanUnits, ((long long)last - first) * kSpanUnits / cols);
                ++samples;
            }
        }
    }
    const unsigned int limit = (unsigned int)cols;                     // cols < 2^31
    for (long long i = 4 * t0; i < nnz; i += 4 * stride) {
        int prev = i > 0 ? indices[i - 1] : -1;
        if (i + 4 <= nnz) {
            const Packed4i c = *reinterpret_cast<const Packed4i*>(indices + i);
            bad |= (unsigned int)c.x >= limit || (unsigned int)c.y >= limit || (unsigned int)c.z >= limit ||
                   (unsigned int)c.w >= limit;
            descents += (i > 0 && c.x <= prev) + (c.y <= c.x) + (c.z <= c.y) + (c.w <= c.z);
            if (values) {
                const Packed4f v = *reinterpret_cast<const Packed4f*>(values + i);
                not_one |= v.x != 1.0f || v.y != 1.0f || v.z != 1.0f || v.w != 1.0f;
            }
        } else {
            for (long long k = i; k < nnz; ++k) {
                const int c = indices[k];
                bad |= (unsigned int)c >= limit;
                if (k > 0 && c <= prev) ++descents;
                if (values) not_one |= values[k] != 1.0f;
                prev = c;
            }
        }
    }
    for (int d = 32; d > 0; d >>= 1) {
        descents += __shfl_xor(descents, d);
        boundary += __shfl_xor(boundary, d);
        span += __shfl_xor(span, d);
        samples += __shfl_xor(samples, d);
        most = max(most, __shfl_xor(most, d));
    }
    __shared__ unsigned int s_sum[4][4];
    __shared__ int s_most[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) { s_sum[0][wave] = descents; s_sum[1][wave] = boundary; s_sum[2][wave] = span; s_sum[3][wave] = samples; s_most[wave] = most; }
    const bool any_bad = __syncthreads_or(bad) != 0;
    const bool any_not_one = __syncthreads_or(not_one) != 0;
    if (threadIdx.x == 0) {
        descents = s_sum[0][0] + s_sum[0][1] + s_sum[0][2] + s_sum[0][3];
        boundary = s_sum[1][0] + s_sum[1][1] + s_sum[1][2] + s_sum[1][3];
        span = s_sum[2][0] + s_sum[2][1] + s_sum[2][2] + s_sum[2][3];
        samples = s_sum[3][0] + s_sum[3][1] + s_sum[3][2] + s_sum[3][3];
        if (any_bad) atomicOr(&out[0], 1u);
        if (any_not_one) atomicOr(&out[3], 1u);
        if (span) atomicAdd(&out[0], span << 1);
        if (samples) atomicAdd(&out[3], samples << 1);
        if (descents) atomicAdd(&out[1], descents);
        if (boundary) atomicAdd(&out[2], boundary);
        if (longest) {
            most = max(max(s_most[0], s_most[1]), max(s_most[2], s_most[3]));
            if (most > __hip_atomic_load(longest, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(longest, most);
        }
    }
}

struct IngestLayout {
    size_t keys_a, keys_b, vals_a, count, temp, temp_bytes, total;
};

hipError_t ingest_layout(long long nnz, int key_bits, IngestLayout* L) {
    size_t sort_bytes = 0, reduce_bytes = 0;
    unsigned long long* k = nullptr;
    float* v = nullptr;
    int* c = nullptr;
    hipError_t e = rocprim::radix_sort_pairs(nullptr, sort_bytes, k, k, v, v, (size_t)nnz, 0u, (unsigned)key_bits);
    if (e != hipSuccess) return e;
    e = rocprim::reduce_by_key(nullptr, reduce_bytes, k, v, (size_t)nnz, k, v, c, rocprim::plus<float>(),
                               rocprim::equal_to<unsigned long long>());
    if (e != hipSuccess) return e;
    size_t off = 0;
    L->keys_a = off; off += align_up((size_t)nnz * 8, 256);
    L->keys_b = off; off += align_up((size_t)nnz * 8, 256);
    L->vals_a = off; off += align_up((size_t)nnz * 4, 256);
    L->count = off;  off += 256;
    L->temp = off;
    L->temp_bytes = std::max(sort_bytes, reduce_bytes);
    off += align_up(L->temp_bytes, 256);
    L->total = off;
    return hipSuccess;
}

bool overlap(const void* a, size_t a_bytes, const void* b, size_t b_bytes) {
    return a && b && (uintptr_t)a < (uintptr_t)b + b_bytes && (uintptr_t)b < (uintptr_t)a + a_bytes;
}

int key_bits_for(long long rows, long long cols) {
    const unsigned long long top = (unsigned long long)rows * (unsigned long long)cols;
    int bits = 1;
    while (bits < 64 && (top >> bits) != 0) ++bits;
    return bits;
}

}  // namespace

namespace lf {

int csr_check(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values, int64_t num_rows,
              int64_t num_cols, int64_t nnz, void* d_scratch, int32_t* h_flags, int64_t* h_span, int64_t* h_longest, const char* what, hipStream_t s) {
    LF_REQUIRE(num_rows >= 0 && num_rows < (1ll << 31) && num_cols >= 1 && num_cols < (1ll << 31), LF_ERR_INVALID,
               "bad shape %lld x %lld", (long long)num_rows, (long long)num_cols);
    LF_REQUIRE(nnz >= 0 && nnz < (1ll << 31), LF_ERR_UNSUPPORTED, "nnz must be below 2^31");
    if (h_flags) *h_flags = LF_CSR_CANONICAL | (d_values ? LF_CSR_UNIT_VALUES : 0);
    if (h_span) *h_span = 0;
    if (h_longest) *h_longest = 0;
    if (num_rows == 0) {
        LF_REQUIRE(nnz == 0, LF_ERR_INVALID, "%s: a matrix without rows holds %lld entries", what, (long long)nnz);
        return LF_OK;
    }
    LF_REQUIRE(d_indptr && (nnz == 0 || d_indices), LF_ERR_INVALID, "%s: null index array", what);
    LF_REQUIRE(d_scratch && (uintptr_t)d_scratch % 4 == 0, LF_ERR_INVALID, "%s: the check needs 16 bytes of device scratch", what);
    unsigned int* out = (unsigned int*)d_scratch;
    const size_t bytes = h_longest ? 20 : 16;
    LF_HIP(hipMemsetAsync(out, 0, bytes, s));
    const long long units = std::max<long long>(num_rows, (nnz + 3) / 4);
    const int grid = (int)std::min<long long>((units + 255) / 256, kCheckGrid);
    csr_check_kernel<<<grid, 256, 0, s>>>(d_indptr, d_indices, d_values, num_rows, num_cols, nnz,
                                     (int)std::max<long long>(1, num_rows / kSpanSamples), out, h_longest ? (int*)out + 4 : nullptr);
    LF_HIP(hipGetLastError());
    unsigned int h[5] = {0, 0, 0, 0, 0};
    LF_HIP(lf::read_back(h, out, bytes, s));
    LF_REQUIRE((h[0] & 1) == 0, LF_ERR_INVALID,
               "%s: the row pointer is not a non-decreasing sequence from 0 to nnz = %lld, or an index lies outside [0, %lld)",
               what, (long long)nnz, (long long)num_cols);
    if (h_flags) *h_flags = (h[1] == h[2] ? LF_CSR_CANONICAL : 0) | (d_values && (h[3] & 1) == 0 ? LF_CSR_UNIT_VALUES : 0);
    if (h_longest) *h_longest = h[4];
    if (h_span && h[1] == h[2] && h[3] >> 1 > 0)
        *h_span = (int64_t)((double)(h[0] >> 1) / (h[3] >> 1) * (double)num_cols / kSpanUnits);
    return LF_OK;
}

}  // namespace lf

extern "C" {

int lf_csr_check(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values, int64_t num_rows,
                 int64_t num_cols, int64_t nnz, void* d_scratch, int32_t* h_flags, lf_stream_t stream) {
    return lf::csr_check(d_indptr, d_indices, d_values, num_rows, num_cols, nnz, d_scratch, h_flags, nullptr, nullptr, "CSR arrays",
                         (hipStream_t)stream);
}

int lf_csr_check_span(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values, int64_t num_rows,
                      int64_t num_cols, int64_t nnz, void* d_scratch, int32_t* h_flags, int64_t* h_span, lf_stream_t stream) {
    return lf::csr_check(d_indptr, d_indices, d_values, num_rows, num_cols, nnz, d_scratch, h_flags, h_span, nullptr, "CSR arrays",
                         (hipStream_t)stream);
}

int lf_csr_check_rows(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values, int64_t num_rows,
                      int64_t num_cols, int64_t nnz, void* d_scratch, int32_t* h_flags, int64_t* h_span, int64_t* h_longest, lf_stream_t stream) {
    return lf::csr_check(d_indptr, d_indices, d_values, num_rows, num_cols, nnz, d_scratch, h_flags, h_span, h_longest, "CSR arrays",
                         (hipStream_t)stream);
}

size_t lf_coo_to_csr_workspace_bytes(int64_t nnz, int64_t num_rows, int64_t num_cols) {
    if (nnz <= 0 || num_rows <= 0 || num_cols <= 0) return 256;
    IngestLayout L{};
    if (ingest_layout(nnz, key_bits_for(num_rows, num_cols), &L) != hipSuccess) return 0;
    return std::max(L.total, bin_shape(nnz, num_rows, num_cols).total);
}

int lf_coo_to_csr(const int32_t* d_coo_row, const int32_t* d_coo_col, const float* d_coo_val, int64_t nnz,
                  int64_t num_rows, int64_t num_cols, void* d_workspace, size_t workspace_bytes,
                  int32_t* d_indptr, int32_t* d_indices, float* d_values, int64_t* h_nnz_out,
                  lf_stream_t stream) {
    int64_t longest = 0;
    return lf_coo_to_csr_rows(d_coo_row, d_coo_col, d_coo_val, nnz, num_rows, num_cols, d_workspace, workspace_bytes, d_indptr, d_indices, d_values,
                              h_nnz_out, &longest, stream);
}

int lf_coo_to_csr_rows(const int32_t* d_coo_row, const int32_t* d_coo_col, const float* d_coo_val, int64_t nnz,
                       int64_t num_rows, int64_t num_cols, void* d_workspace, size_t workspace_bytes,
                       int32_t* d_indptr, int32_t* d_indices, float* d_values, int64_t* h_nnz_out, int64_t* h_longest,
                       lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(num_rows >= 0 && num_rows < (1ll << 31) && num_cols >= 1 && num_cols < (1ll << 31), LF_ERR_INVALID,
               "bad shape %lld x %lld", (long long)num_rows, (long long)num_cols);
    LF_REQUIRE(nnz >= 0 && nnz < (1ll << 31), LF_ERR_UNSUPPORTED, "nnz must be below 2^31");
    LF_REQUIRE(d_indptr && h_nnz_out && h_longest, LF_ERR_INVALID, "null output");
    if (nnz == 0) {
        *h_longest = 0;
        LF_HIP(hipMemsetAsync(d_indptr, 0, (size_t)(num_rows + 1) * 4, s));
        LF_HIP(hipStreamSynchronize(s));
        *h_nnz_out = 0;
        return LF_OK;
    }
    LF_REQUIRE(d_coo_row && d_coo_col && d_indices && d_values, LF_ERR_INVALID, "null argument");
    const int key_bits = key_bits_for(num_rows, num_cols);
    IngestLayout L{};
    LF_HIP(ingest_layout(nnz, key_bits, &L));
    LF_REQUIRE(d_workspace && workspace_bytes >= L.total, LF_ERR_WORKSPACE, "workspace has %zu bytes, %zu needed",
               workspace_bytes, L.total);
    char* ws = (char*)d_workspace;
    const BinShape b = bin_shape(nnz, num_rows, num_cols);
    // The bins write the results before it is known whether the triplets have to be read again; the sort does not.
    bool in_place = false;
    for (const void* in : {(const void*)d_coo_row, (const void*)d_coo_col, (const void*)d_coo_val})
        in_place = in_place || overlap(in, (size_t)nnz * 4, d_indices, (size_t)nnz * 4) || overlap(in, (size_t)nnz * 4, d_values, (size_t)nnz * 4) ||
                   overlap(in, (size_t)nnz * 4, d_indptr, (size_t)(num_rows + 1) * 4);
    if (b.bins > 0 && workspace_bytes >= b.total && !in_place) {
        int *counts = (int*)(ws + b.counts), *totals = (int*)(ws + b.totals), *bases = (int*)(ws + b.bases);
        int *list = (int*)(ws + b.list), *flags = (int*)(ws + b.flags);
        uint2* records = (uint2*)(ws + b.records);
        const unsigned inverse = (unsigned)std::min<unsigned long long>((1ull << 32) / (unsigned long long)num_cols, 0xFFFFFFFFull);
        const BinSort sort{records, bases, totals, num_rows, b.lg_rows, b.lg_cols, inverse, d_indptr, d_indices, d_values, list, flags};
        LF_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(bin_sort_large_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kBinLargeBytes));
        clear_words_kernel<<<1, 64, 0, s>>>(flags, kFlags);
        bin_count_kernel<<<b.chunks, kBinThreads, 0, s>>>(d_coo_row, d_coo_col, nnz, num_rows, num_cols, b.lg_rows, b.bins, b.per_chunk, counts, flags);
        bin_offsets_kernel<<<(b.bins + 3) / 4, 256, 0, s>>>(counts, b.bins, b.chunks, totals, b.most_reads, flags);
        bin_distribute_kernel<<<b.chunks, kBinThreads, 0, s>>>(d_coo_row, d_coo_col, d_coo_val, nnz, num_rows, num_cols, b.lg_rows, b.lg_cols, b.bins,
                                                               b.per_chunk, counts, totals, bases, records, flags);
        bin_sort_kernel<<<b.bins, kBinThreads, 0, s>>>(sort);
        if (nnz > kBinSmall) {
            const unsigned grid = (unsigned)std::min<long long>(nnz / kBinWindow + b.bins, kBinLargeGrid);
            bin_sort_large_kernel<<<grid, 1024, kBinLargeBytes, s>>>(sort);
        }
        LF_HIP(hipGetLastError());
        // The loan goes back when this returns: every way out from here on has waited for the stream.
        lf::PinnedLoan back((kLongest + 1) * 4);
        LF_REQUIRE(back.ok(), LF_ERR_HIP, "out of host memory");
        int* report = back.pinned() ? back.as<int>() : (int*)(ws + b.totals);
        bin_report_kernel<<<1, 256, 0, s>>>(flags, b.bins, report);
        hipError_t reported = hipGetLastError();
        if (reported == hipSuccess && !back.pinned())
            reported = hipMemcpyAsync(back.as<char>(), report, (kLongest + 1) * 4, hipMemcpyDeviceToHost, s);
        const hipError_t waited = hipStreamSynchronize(s);
        LF_HIP(reported);
        LF_HIP(waited);
        const int* h_flags = back.as<int>();
        const bool sorted = h_flags[kNotHere] == 0 && h_flags[kCrowded] == 0;
        if (sorted) *h_longest = h_flags[kLongest];
        if (sorted && h_flags[kTwice] == 0) {
            *h_nnz_out = nnz;
            return LF_OK;
        }
        if (sorted) {
            int32_t *twice = (int32_t*)(ws + b.twice), *before = (int32_t*)(ws + b.before), *partial = (int32_t*)(ws + b.partial);
            int32_t* out_indices = (int32_t*)records;
            float* out_values = (float*)(out_indices + nnz);
            const unsigned blocks = (unsigned)((nnz + 255) / 256);
            mark_twice_kernel<<<blocks, 256, 0, s>>>(d_indptr, d_indices, nnz, num_rows, twice);
            LF_HIP(exclusive_scan_i32(twice, nnz, partial, before, s));
            add_up_kernel<<<blocks, 256, 0, s>>>(d_indices, d_values, twice, before, nnz, out_indices, out_values);
            close_up_kernel<<<(unsigned)(std::max<long long>(num_rows + 1, nnz) + 255) / 256, 256, 0, s>>>(
                d_indptr, before, num_rows, nnz, out_indices, out_values, d_indices, d_values);
            LF_HIP(hipGetLastError());
            LF_HIP(hipStreamSynchronize(s));
            *h_nnz_out = nnz - h_flags[kTwice];
            return LF_OK;
        }
    }
    unsigned long long* keys_a = (unsigned long long*)(ws + L.keys_a);
    unsigned long long* keys_b = (unsigned long long*)(ws + L.keys_b);
    float* vals_a = (float*)(ws + L.vals_a);
    int* count = (int*)(ws + L.count);
    void* temp = ws + L.temp;
    size_t temp_bytes = L.temp_bytes;

    const int grid = (int)std::min<long long>((nnz + 255) / 256, 65535);
    pack_keys_kernel<<<grid, 256, 0, s>>>(d_coo_row, d_coo_col, d_coo_val, nnz, num_cols, keys_a, d_values, count + 1);
    LF_HIP(hipGetLastError());
    // sorted keys -> keys_b, values in the same order -> vals_a
    LF_HIP(rocprim::radix_sort_pairs(temp, temp_bytes, keys_a, keys_b, d_values, vals_a, (size_t)nnz, 0u,
                                     (unsigned)key_bits, s));
    // unique keys -> keys_a, summed values -> d_values, count
    temp_bytes = L.temp_bytes;
    LF_HIP(rocprim::reduce_by_key(temp, temp_bytes, keys_b, vals_a, (size_t)nnz, keys_a, d_values, count,
                                  rocprim::plus<float>(), rocprim::equal_to<unsigned long long>(), s));
    unpack_cols_kernel<<<grid, 256, 0, s>>>(keys_a, count, num_cols, d_indices);
    LF_HIP(hipGetLastError());
    row_pointer_kernel<<<(unsigned)std::max<int64_t>(1, (num_rows + kPointerRows - 1) / kPointerRows), kPointerThreads, 0, s>>>(
        keys_a, count, num_rows, num_cols, d_indptr, count + 1);
    LF_HIP(hipGetLastError());
    int h_count[2] = {0, 0};                                   // entries, those of the longest row
    LF_HIP(lf::read_back(h_count, count, sizeof(h_count), s));
    *h_nnz_out = h_count[0];
    *h_longest = h_count[1];
    return LF_OK;
}

}  // extern "C"
