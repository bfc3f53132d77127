// Device side of format composition for gfx950: bucket statistics for the width search
// and the hyb (column partition x power-of-two ELL bucket) builder.
//
// Reference behaviour reproduced here:
//   get_init_buckets   playground_pipline/format_algos.py:819-900   (lf_bucket_stats)
//   build_hyb_format   playground_pipline/format_algos.py:226-385   (lf_hyb_plan / lf_hyb_build)
//
// The reference walks nonzeros one at a time on the host.  On the GPU the same result is
// obtained from per-(row, partition) segments: CSR is row-major with ascending columns,
// so the nonzeros of one segment are contiguous, every bucket receives whole segments in
// ascending row order, and a segment of `fill` entries occupies ceil(fill / W) consecutive
// ELL rows that carry the same row id, with (0, 0) padding only after its last entry.
// ELL-row offsets are therefore an exclusive scan, in row order, of per-segment ELL-row
// counts, taken separately for each bucket.  All counting uses integer arithmetic, so the
// output does not depend on scheduling.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "lf_index.h"
#include "lf_internal.h"

// Accumulators of lf_row_features_static: {min, max, sum, sum of squares}.  One copy of the
// array lives on every GPU the library runs on, for the life of the process.  Host code never
// uses the array's name as an address: static_scratch() below asks the runtime where the
// current device keeps it.
static __device__ __align__(256) unsigned long long lf_static_scratch[4];

namespace {

constexpr int kBlock = 256;          // rows per workgroup in the per-segment kernels
constexpr int kStatsGrid = 2048;     // workgroups per partition in the statistics pass at most
// meta word of an ELL row: bits 0..10 valid slots (1..1024); bits 11..30 a count: on the
// first ELL row of a source row's segment the number of ELL rows in the segment, on a
// continuation row its index inside the segment; bit 31 set on continuation rows.
constexpr int kMetaLenBits = 11;
constexpr int kMetaSegMax = (1 << (31 - kMetaLenBits)) - 1;
constexpr uint32_t kMetaCont = 0x80000000u;

__host__ __device__ inline int32_t make_meta(int len, int i, int n_ell) {
    return (int32_t)((uint32_t)len | ((uint32_t)(i == 0 ? n_ell : i) << kMetaLenBits) | (i == 0 ? 0u : kMetaCont));
}

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// ---------------------------------------------------------------------------- device utils
__device__ __forceinline__ int lower_bound_i32(const int32_t* __restrict__ a, int lo, int hi, int64_t key) {
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((int64_t)a[mid] < key) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// Segment (row r, partition p): offset of its first entry in the CSR arrays and its length.
// With one partition the segment is the row; otherwise boundaries were precomputed into
// bnd[(P + 1)][rows] (partition-major so that neighbouring threads read neighbouring words).
struct SegView {
    const int32_t* indptr;
    const int32_t* bnd;
    int64_t rows;
    int parts;
};

__device__ __forceinline__ void seg_range(const SegView& v, int64_t r, int p, int& start, int& fill) {
    if (v.parts == 1) {
        start = v.indptr[r];
        fill = v.indptr[r + 1] - start;
    } else {
        start = v.bnd[(int64_t)p * v.rows + r];
        fill = v.bnd[(int64_t)(p + 1) * v.rows + r] - start;
    }
}

__global__ void fill_u32_kernel(uint32_t* __restrict__ p, int64_t n, uint32_t value) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = value;
}

hipError_t fill_u32(void* p, int64_t n_words, uint32_t value, hipStream_t s) {
    if (n_words <= 0) return hipSuccess;
    const int grid = (int)std::min<int64_t>((n_words + 255) / 256, 4096);
    fill_u32_kernel<<<grid, 256, 0, s>>>((uint32_t*)p, n_words, value);
    return hipGetLastError();
}

// bnd[p][r] = first CSR position of row r whose column is >= p * psize   (p = 0..P)
__global__ void seg_bounds_kernel(const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices,
                                  int64_t rows, int parts, int64_t psize, int32_t* __restrict__ bnd) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const int lo = indptr[r], hi = indptr[r + 1];
    bnd[r] = lo;
    int cur = lo;
    for (int p = 1; p < parts; ++p) {
        cur = lower_bound_i32(indices, cur, hi, (int64_t)p * psize);
        bnd[(int64_t)p * rows + r] = cur;
    }
    bnd[(int64_t)parts * rows + r] = hi;
}

// deg[p][r] += 1 for every COO triplet (format_algos.py:846-849 counts raw triplets)
__global__ void coo_degree_kernel(const int32_t* __restrict__ row, const int32_t* __restrict__ col,
                                  int64_t nnz, int64_t rows, int64_t psize, int32_t* __restrict__ deg) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nnz;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t p = col[i] / psize;
        atomicAdd(&deg[p * rows + row[i]], 1);
    }
}

// out = {min, max, sum, sum of squares} of the row lengths; out[0] starts at ~0, the rest at 0
__global__ void __launch_bounds__(kBlock)
row_features_kernel(const int32_t* __restrict__ indptr, int64_t rows, unsigned long long* __restrict__ out) {
    __shared__ unsigned long long s_red[4][kBlock / 64];
    unsigned long long lo = ~0ull, hi = 0, sum = 0, sq = 0;
    for (int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x; r < rows; r += (int64_t)gridDim.x * kBlock) {
        const unsigned long long d = (unsigned long long)(indptr[r + 1] - indptr[r]);
        lo = d < lo ? d : lo;
        hi = d > hi ? d : hi;
        sum += d;
        sq += d * d;
    }
    for (int d = 32; d > 0; d >>= 1) {
        const unsigned long long l2 = __shfl_xor(lo, d), h2 = __shfl_xor(hi, d);
        lo = l2 < lo ? l2 : lo;
        hi = h2 > hi ? h2 : hi;
        sum += __shfl_xor(sum, d);
        sq += __shfl_xor(sq, d);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) { s_red[0][wave] = lo; s_red[1][wave] = hi; s_red[2][wave] = sum; s_red[3][wave] = sq; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / 64; ++w) {
            lo = s_red[0][w] < lo ? s_red[0][w] : lo;
            hi = s_red[1][w] > hi ? s_red[1][w] : hi;
            sum += s_red[2][w];
            sq += s_red[3][w];
        }
        atomicMin(&out[0], lo);
        atomicMax(&out[1], hi);
        atomicAdd(&out[2], sum);
        atomicAdd(&out[3], sq);
    }
}

// out[0] += entries of row r that also occur in row r - 1, out[1] += entries of row r, for every
// stride-th row r >= 1.  A wavefront takes a pair of rows: lane i holds the i-th entry of either row
// and looks its entry of row r up among those of row r - 1.  Only the first kOverlapEntries = 64
// entries of either row are looked at: a sample that lands on a row of 100,000 entries would
// otherwise take longer than composing the whole format (11 ms against 0.3 ms for a 500k x 2M matrix
// with 50 such rows).  Bound by latency: a thread per pair with a two-pointer walk was a chain of up
// to 128 loads, 15.6 us for 8192 pairs.
constexpr int kOverlapEntries = 64;
constexpr int kOverlapThreads = 1024;      // few, large workgroups: each ends with two atomics on one line
constexpr int kOverlapGrid = 128;
__device__ __forceinline__ void
row_overlap(const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices, int64_t rows,
            int64_t stride, unsigned long long* __restrict__ out, int group, int groups) {
    const int lane = threadIdx.x & 63;
    uint32_t both = 0, seen = 0;
    const int64_t waves = (int64_t)groups * (kOverlapThreads / 64);
    for (int64_t i = (int64_t)group * (kOverlapThreads / 64) + (threadIdx.x >> 6);; i += waves) {
        const int64_t r = 1 + i * stride;
        if (r >= rows) break;
        const int a = indptr[r - 1], b = indptr[r];
        const int na = min(b - a, kOverlapEntries), nb = min(indptr[r + 1] - b, kOverlapEntries);
        const int ca = lane < na ? indices[a + lane] : 0x7FFFFFFF;      // columns are below 2^31 - 1
        const int cb = lane < nb ? indices[b + lane] : -1;
        int lo = 0;                                     // entries of row r - 1 below cb
#pragma unroll
        for (int step = 32; step > 0; step >>= 1) {
            const int x = __shfl(ca, lo + step - 1);
            if (x < cb) lo += step;
        }
        const int hit = __shfl(ca, lo & 63);            // (all lanes take part)
        both += lane < nb && hit == cb;
        seen += lane < nb;
    }
    for (int d = 32; d > 0; d >>= 1) {
        both += __shfl_xor(both, d);
        seen += __shfl_xor(seen, d);
    }
    __shared__ uint32_t s_sum[2][kOverlapThreads / 64];
    if (lane == 0) { s_sum[0][threadIdx.x >> 6] = both; s_sum[1][threadIdx.x >> 6] = seen; }
    __syncthreads();
    if (threadIdx.x < 2) {
        unsigned long long sum = 0;
        for (int w = 0; w < kOverlapThreads / 64; ++w) sum += s_sum[threadIdx.x][w];
        if (sum) atomicAdd(&out[threadIdx.x], sum);
    }
}

__global__ void __launch_bounds__(kOverlapThreads)
row_overlap_kernel(const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices, int64_t rows,
                   int64_t stride, unsigned long long* __restrict__ out) {
    row_overlap(indptr, indices, rows, stride, out, blockIdx.x, gridDim.x);
}

inline int overlap_groups(int64_t rows, int64_t stride) {
    const int64_t samples = (rows - 1 + stride - 1) / stride, per = kOverlapThreads / 64;
    return (int)std::min<int64_t>((samples + per - 1) / per, kOverlapGrid);
}

inline hipError_t launch_row_overlap(const int32_t* indptr, const int32_t* indices, int64_t rows, int64_t stride,
                                     unsigned long long* out, hipStream_t s) {
    row_overlap_kernel<<<overlap_groups(rows, stride), kOverlapThreads, 0, s>>>(indptr, indices, rows, stride, out);
    return hipGetLastError();
}

// Initial width class of a segment of `deg` entries: width = min(next_pow2(deg), limit),
// cost-model rows = max(1, next_pow2(deg) / limit)            (format_algos.py:875-882)
__device__ __forceinline__ void width_class(int deg, int kmax, int& k, int& cost_rows) {
    k = deg <= 1 ? 0 : 32 - __clz(deg - 1);
    cost_rows = 1;
    if (k > kmax) {
        cost_rows = 1 << (k - kmax);
        k = kmax;
    }
}

// Where the counters of partition p and class k lie: field f (0 cost rows, 1 nnz, 2 segments) has a
// 128-byte line of its own, because atomics of all workgroups on one line are taken one after the
// other (all counters of a partition side by side: 25 us of class_count_kernel's time).
constexpr int kStatLine = 16;              // 64-bit words
__host__ __device__ constexpr size_t stat_at(int p, int k, int f) { return (((size_t)p * LF_MAX_CLASSES + k) * 3 + f) * kStatLine; }

// stats(p, k) += {cost rows, nnz, 1} for every segment of partition p = blockIdx.y.
// A workgroup counts a contiguous range of rows in LDS - a 64-bit word {segments, entries} for every class and lane, so that the
// lanes of a wavefront never meet - and adds its sums with one atomic per counter.  (One word per class took 48 us for 2.45M
// rows, counters in registers, 33 selects a row, 22, this takes 12.)
constexpr int kCountGrid = 256, kCountThreads = 1024;      // (atomics of 512 workgroups on a counter's line: 9 us)
constexpr int kRowUnroll = 4;              // rows whose bounds a thread requests together

// Segments of rows r0 < end, r0 + stride, ... and their degrees (0 past `end`).  Every lane loads: behind a condition the loads of a
// row would wait for those of the row before.
__device__ __forceinline__ void seg_degrees(const SegView& v, const int32_t* __restrict__ seg_deg, int p, int64_t r0,
                                            int64_t stride, int64_t end, int (&start)[kRowUnroll], int (&fill)[kRowUnroll], int (&deg)[kRowUnroll]) {
    const int32_t *first = v.parts == 1 ? v.indptr : v.bnd + (int64_t)p * v.rows, *last = v.parts == 1 ? v.indptr + 1 : first + v.rows;
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u) {
        const int64_t r = min(r0 + u * stride, end - 1);
        start[u] = first[r];
        fill[u] = last[r];
    }
    if (seg_deg) {
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) deg[u] = seg_deg[(int64_t)p * v.rows + min(r0 + u * stride, end - 1)];
    }
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u) {
        fill[u] -= start[u];
        if (!seg_deg) deg[u] = fill[u];
        if (r0 + u * stride >= end) deg[u] = 0;
    }
}

// What the workgroups of class_count_kernel counted, for class_list_kernel: segments of class k of partition p in workgroup g;
// kmax + 1: of the last class, those of more than kMarkBigSegment entries.
constexpr int kCountClasses = 16;
__host__ __device__ constexpr size_t count_at(int p, int k, int g) { return ((size_t)p * kCountClasses + k) * kCountGrid + g; }
constexpr int kMarkBigSegment = 8192;      // longer segments are shared by all workgroups of their item, see below

__global__ void __launch_bounds__(kCountThreads)
class_count_kernel(SegView v, const int32_t* __restrict__ seg_deg, int kmax, unsigned long long* __restrict__ stats, int32_t* __restrict__ counts) {
    static_assert(LF_MAX_CLASSES < kCountClasses && kCountThreads == 64 * kCountClasses);
    constexpr int kCntShift = 40;          // entries of a lane's rows stay below 2^31, their number below 2^23
    __shared__ unsigned long long s_sum[LF_MAX_CLASSES * 64];
    __shared__ uint32_t s_more, s_big;     // cost rows beyond one a segment; segments of more than kMarkBigSegment entries
    const int p = blockIdx.y;
    for (int i = threadIdx.x; i < LF_MAX_CLASSES * 64; i += kCountThreads) s_sum[i] = 0;
    if (threadIdx.x == 0) s_more = s_big = 0;
    __syncthreads();
    const int64_t per = (v.rows + gridDim.x - 1) / gridDim.x;
    const int64_t lo = (int64_t)blockIdx.x * per, hi = lo + per < v.rows ? lo + per : v.rows;
    unsigned long long* mine = s_sum + (threadIdx.x & 63);
    for (int64_t r0 = lo + threadIdx.x; r0 < hi; r0 += kRowUnroll * kCountThreads) {
        int start[kRowUnroll], fill[kRowUnroll], deg[kRowUnroll];
        seg_degrees(v, seg_deg, p, r0, kCountThreads, hi, start, fill, deg);
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) {
            if (deg[u] <= 0) continue;
            int k, cost_rows;
            width_class(deg[u], kmax, k, cost_rows);
            atomicAdd(&mine[k * 64], (1ull << kCntShift) | (unsigned long long)deg[u]);
            if (cost_rows > 1) atomicAdd(&s_more, (uint32_t)(cost_rows - 1));
            if (deg[u] > kMarkBigSegment && k == kmax) atomicAdd(&s_big, 1u);
        }
    }
    __syncthreads();
    const int k = threadIdx.x >> 6;                                          // a wavefront to a class
    unsigned long long nnz = 0;
    uint32_t cnt = 0;
    if (k < LF_MAX_CLASSES) {
        const unsigned long long x = s_sum[threadIdx.x];
        nnz = x & ((1ull << kCntShift) - 1);
        cnt = (uint32_t)(x >> kCntShift);
    }
    for (int d = 1; d < 64; d <<= 1) {
        nnz += __shfl_xor(nnz, d);
        cnt += __shfl_xor(cnt, d);
    }
    if ((threadIdx.x & 63) != 0) return;
    const uint32_t big = s_big;
    if (k < LF_MAX_CLASSES && cnt) {
        atomicAdd(&stats[stat_at(p, k, 0)], (unsigned long long)cnt + (k == kmax ? s_more : 0u));
        atomicAdd(&stats[stat_at(p, k, 1)], nnz);
        atomicAdd(&stats[stat_at(p, k, 2)], (unsigned long long)cnt);
        if (k == kmax && big) atomicAdd(&stats[stat_at(p, k, 2) + 2], (unsigned long long)big);      // (a spare word of the counter's line)
    }
    if (counts) counts[count_at(p, k, blockIdx.x)] = (int)(k == kmax + 1 ? big : k == kmax ? cnt - big : k < kmax ? cnt : 0u);
}

// ---- statistics of several partition counts at once
// What the launch-shape choice prices: the counters of class_count_kernel for every partition of
// every candidate count, from one pass over the rows.  A thread finds the partition bounds of its
// row for each candidate in turn (binary search in the row's ascending columns) and adds the
// segments to counters in LDS; a workgroup leaves its counters in the workspace and
// shape_reduce_kernel adds the workgroups up.  Bound by the latency of the searches.  One statistics
// call per candidate - bounds written to memory and read back, a launch of its own for each kernel
// and a synchronisation - took 41 us each for a 170K-row graph (four candidates and the row overlap
// 235 us, now 86 with the Python around it).
constexpr int kShapeCands = 16;
constexpr int kShapeParts = 128;           // partitions of all candidates together
constexpr int kShapeGrid = 1024;
// A lane searches the boundaries of a row one after the other, each search a chain of loads; those of a longer row are searched by the
// lanes of the wavefront side by side (170K rows, the longest of 13,000 entries, 7 partitions: 21.5 -> 17 us; from 8 entries on 21.6, from 16 18.6).
constexpr int kShapeLongRow = 64;
struct ShapeCands {
    int n, total;
    int parts[kShapeCands];
};

// A workgroup's counters: total * LF_MAX_CLASSES words {nnz in the low half, segments in the high half}
// (both sums stay below 2^31), then per partition the cost rows of the last class beyond one per segment.
constexpr int shape_words(int total) { return total * (LF_MAX_CLASSES + 1); }

__global__ void __launch_bounds__(kBlock)
shape_stats_kernel(const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices, int64_t rows, int64_t cols,
                   ShapeCands cands, int kmax, unsigned long long* __restrict__ partial,
                   unsigned long long* __restrict__ out, int n_out) {
    __shared__ unsigned long long s_cnt[shape_words(kShapeParts)];
    __shared__ int64_t s_end[kShapeParts];                     // first column behind a partition; behind a candidate's last: none
    __shared__ uint8_t s_first[kShapeParts];                   // a candidate's first partition
    const int n_words = shape_words(cands.total);
    for (int i = threadIdx.x; i < n_words; i += kBlock) s_cnt[i] = 0;
    for (int c = 0, q = 0; c < cands.n; q += cands.parts[c++]) {
        const int parts = cands.parts[c];
        const int64_t psize = (cols + parts - 1) / parts;
        for (int p = threadIdx.x; p < parts; p += kBlock) {
            s_end[q + p] = p + 1 < parts ? (p + 1) * psize : INT64_MAX;
            s_first[q + p] = p == 0;
        }
    }
    if (blockIdx.x == 0)                                       // for the launch behind this one
        for (int i = threadIdx.x; i < n_out; i += kBlock) out[i] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    auto count = [&](int q, int fill) {
        if (fill <= 0) return;
        int k, cost_rows;
        width_class(fill, kmax, k, cost_rows);
        atomicAdd(&s_cnt[q * LF_MAX_CLASSES + k], (1ull << 32) | (unsigned long long)fill);
        if (cost_rows > 1) atomicAdd(&s_cnt[cands.total * LF_MAX_CLASSES + q], (unsigned long long)(cost_rows - 1));
    };
    for (int64_t r0 = (int64_t)blockIdx.x * kBlock + threadIdx.x - lane; r0 < rows; r0 += (int64_t)gridDim.x * kBlock) {
        const int64_t r = min(r0 + lane, rows - 1);
        const int lo = indptr[r], hi = r0 + lane < rows ? indptr[r + 1] : lo;
        const bool alone = hi - lo <= kShapeLongRow;
        for (int q = 0, cur = lo; q < cands.total && alone; ++q) {
            const int from = s_first[q] ? lo : cur;
            cur = s_end[q] < INT64_MAX ? lower_bound_i32(indices, from, hi, s_end[q]) : hi;
            count(q, cur - from);
        }
        for (unsigned long long pending = __ballot(!alone); pending != 0; pending &= pending - 1) {
            const int src = __builtin_ctzll(pending), first = __shfl(lo, src), last = __shfl(hi, src);
            int before = first;                                // end of the partition before this round's
            for (int q0 = 0; q0 < cands.total; q0 += 64) {
                const int q = min(q0 + lane, cands.total - 1);
                const int end = s_end[q] < INT64_MAX ? lower_bound_i32(indices, first, last, s_end[q]) : last;
                int from = __shfl_up(end, 1);
                if (lane == 0) from = before;
                if (s_first[q]) from = first;
                if (q0 + lane < cands.total) count(q, end - from);
                before = __shfl(end, 63);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n_words; i += kBlock) partial[(size_t)blockIdx.x * n_words + i] = s_cnt[i];
}

// out[q][k] = {cost rows, nnz, segments, 0}: 64 words to a workgroup, 16 threads add up each.  The workgroups behind those sample
// the row overlap, whose two sums follow the statistics.
static_assert(kOverlapThreads == 1024);
__global__ void __launch_bounds__(1024)
shape_reduce_kernel(const unsigned long long* __restrict__ partial, int n_groups, int total, int kmax,
                    unsigned long long* __restrict__ out, const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices,
                    int64_t rows, int64_t stride) {
    __shared__ unsigned long long s_sum[16][64];
    const int reducers = (shape_words(total) + 63) / 64;
    if ((int)blockIdx.x >= reducers) {
        row_overlap(indptr, indices, rows, stride, out + (size_t)total * LF_MAX_CLASSES * LF_STATS_FIELDS, blockIdx.x - reducers, gridDim.x - reducers);
        return;
    }
    const int n_words = shape_words(total);
    const int w = blockIdx.x * 64 + (threadIdx.x & 63), slice = threadIdx.x >> 6;
    unsigned long long sum = 0;
    if (w < n_words) {
        for (int g0 = slice; g0 < n_groups; g0 += 16 * 8) {
            unsigned long long x[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) x[u] = g0 + 16 * u < n_groups ? partial[(size_t)(g0 + 16 * u) * n_words + w] : 0ull;
#pragma unroll
            for (int u = 0; u < 8; ++u) sum += x[u];
        }
    }
    s_sum[slice][threadIdx.x & 63] = sum;
    __syncthreads();
    if (slice != 0 || w >= n_words) return;
    for (int i = 1; i < 16; ++i) sum += s_sum[i][threadIdx.x];
    // the cost rows of the last class come from two words: each adds its part to a cleared field
    if (w < total * LF_MAX_CLASSES) {
        unsigned long long* o = out + (size_t)w * LF_STATS_FIELDS;
        atomicAdd(&o[0], sum >> 32);
        o[1] = sum & 0xFFFFFFFFull;
        o[2] = sum >> 32;
        o[3] = 0;
    } else if (sum) {
        atomicAdd(&out[((size_t)(w - total * LF_MAX_CLASSES) * LF_MAX_CLASSES + kmax) * LF_STATS_FIELDS], sum);
    }
}

// Column sets as byte planes, for matrices that the bitmaps below do not take: plane[k][c] = 1 for
// every column c of a segment of class k; blockIdx.y is the partition.
// Column sets are one byte per (class, column), written with plain stores after an "already
// set?" probe: no atomics, and a stale probe (another XCD's L2 still holds the old line) only
// repeats a store of the same value.  blockIdx.z is the class a workgroup marks: workgroups
// are handed out z last, so the launch works through one class (and partition) at a time.
// The columns of a class are walked by the whole workgroup over the concatenation of its
// segments among 256 rows (element -> segment by a binary search over LDS prefix sums), four
// independent elements per thread, so neither a long row nor the chain "index load -> probe"
// of one row serialises.  Measured for 81.6M nonzeros, 2.45M columns: one thread per row
// with a 32-bit mask per column and atomicOr 2.0 ms; workgroup walk with 16-bit masks and
// atomicOr 1.86 ms, of which the ~13M atomics take 1.2 ms (a mask copy per XCD makes it
// 3.1 ms: more atomics, and they cost the same wherever the line lives); byte planes with
// all classes in flight 1.47 ms; byte planes class by class 1.44 ms (0.38 ms walk, 0.27 ms
// probes, 0.8 ms stores).  The counters show one 64-byte line fetched per probe and one
// written per first-touch store (5.2 GB + 1.1 GB): the pass runs at the rate the fabric
// moves single lines, the planes do not stay in the L2s between probes.
constexpr int kMarkUnroll = 4;

__global__ void __launch_bounds__(kBlock)
mark_planes_kernel(SegView v, const int32_t* __restrict__ indices, const int32_t* __restrict__ seg_deg,
                   int kmax, uint8_t* __restrict__ planes, int64_t cols) {
    __shared__ int s_off[kBlock + 1];      // exclusive prefix of the lengths of this class's segments
    __shared__ int s_start[kBlock];
    __shared__ int s_wave[kBlock / 64];
    const int p = blockIdx.y;
    const int kz = blockIdx.z;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint8_t* plane = planes + (size_t)kz * (size_t)cols;
    for (int64_t base = (int64_t)blockIdx.x * kBlock; base < v.rows; base += (int64_t)gridDim.x * kBlock) {
        const int64_t r = base + threadIdx.x;
        int start = 0, fill = 0, deg = 0;
        if (r < v.rows) {
            seg_range(v, r, p, start, fill);
            deg = seg_deg ? seg_deg[(int64_t)p * v.rows + r] : fill;
        }
        int k = -1;
        if (deg > 0) {
            int cost_rows;
            width_class(deg, kmax, k, cost_rows);
        }
        const int x = k == kz ? fill : 0;
        if (!__syncthreads_or(x)) continue;            // no segment of this class among these rows
        int incl = x;
        for (int d = 1; d < 64; d <<= 1) {
            const int y = __shfl_up(incl, d);
            if (lane >= d) incl += y;
        }
        if (lane == 63) s_wave[wave] = incl;
        __syncthreads();
        int wave_off = 0;
        for (int wv = 0; wv < wave; ++wv) wave_off += s_wave[wv];
        s_off[threadIdx.x] = wave_off + incl - x;
        s_start[threadIdx.x] = start;
        if (threadIdx.x == kBlock - 1) s_off[kBlock] = wave_off + incl;
        __syncthreads();
        const int total = s_off[kBlock];
        for (int j0 = 0; j0 < total; j0 += kBlock * kMarkUnroll) {
            int c[kMarkUnroll];
            uint8_t seen[kMarkUnroll];
#pragma unroll
            for (int u = 0; u < kMarkUnroll; ++u) {
                const int j = j0 + u * kBlock + (int)threadIdx.x;
                c[u] = -1;
                if (j < total) {
                    int lo = 0, hi = kBlock - 1;       // last segment whose offset is <= j
#pragma unroll
                    for (int step = 0; step < 8; ++step) {
                        const int mid = (lo + hi + 1) >> 1;
                        if (s_off[mid] <= j) lo = mid; else hi = mid - 1;
                    }
                    c[u] = indices[s_start[lo] + (j - s_off[lo])];
                }
            }
#pragma unroll
            for (int u = 0; u < kMarkUnroll; ++u) seen[u] = c[u] >= 0 ? plane[c[u]] : (uint8_t)1;
#pragma unroll
            for (int u = 0; u < kMarkUnroll; ++u)
                if (seen[u] == 0) plane[c[u]] = 1;
        }
        __syncthreads();                               // the tables are rewritten by the next block of rows
    }
}

// hist[p][mask] = number of columns of partition p whose set of classes is mask
__global__ void __launch_bounds__(kBlock)
colmask_hist_kernel(const uint8_t* __restrict__ planes, int num_classes, int64_t cols, int64_t psize,
                    unsigned long long* __restrict__ hist) {
    constexpr int kBins = 1 << LF_MAX_CLASSES;
    __shared__ uint32_t s_hist[kBins];
    for (int i = threadIdx.x; i < kBins; i += kBlock) s_hist[i] = 0;
    __syncthreads();
    const int p = blockIdx.y;
    const int64_t lo = (int64_t)p * psize;
    const int64_t hi = lo + psize < cols ? lo + psize : cols;
    for (int64_t c = lo + (int64_t)blockIdx.x * kBlock + threadIdx.x; c < hi;
         c += (int64_t)gridDim.x * kBlock) {
        uint32_t m = 0;
        for (int k = 0; k < num_classes; ++k) m |= planes[(size_t)k * (size_t)cols + c] ? 1u << k : 0u;
        atomicAdd(&s_hist[m], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kBins; i += kBlock)
        if (s_hist[i]) atomicAdd(&hist[(size_t)p * kBins + i], (unsigned long long)s_hist[i]);
}

// ---- column sets through bitmaps in LDS
// The byte planes above cost one line over the fabric per probe and per first-touch store.  Where
// a partition's columns fit a few bitmaps of one LDS each, a workgroup instead owns one (partition,
// slice of columns, class) at a time: it walks its share of the class's segments, ORs their
// columns into a bitmap in LDS and writes the bitmap out once; colbits_hist_kernel ORs the bitmaps
// of the workgroups that shared an item and counts the class masks.  The indices are streamed once
// per slice, everything else stays in the CU.  2.45M columns (two slices), 81M entries: the
// column pass takes 0.16 ms where the planes took 1.38 (marking 0.13, listing 0.01, histogram 0.02).
// Marking is bound by the lines of the class's scattered segments (4.6M past the L2s, 0.6 GB) and by what a CU has under way.  It took
// 202 us with loads behind a condition, one of a wavefront under way at a time, the slices' workgroups wherever they fell (8.8M
// lines past the L2s) and shares by the lanes of a step: the last workgroups ended 50 us after most.
//
// Segments are first listed by class (class_list_kernel), because a class is a scattered subset of
// the rows: finding it again in every workgroup would cost 11 sweeps over the row pointer.
constexpr int kMarkThreads = 1024;
constexpr int kMarkMaxWords = 38912;       // 152 KB of the 160 KB of LDS: 1,245,184 columns
constexpr int kMarkTwoPerCu = 18432;       // bitmaps of up to 72 KB: two workgroups share a CU
constexpr int kMarkItems = 512;            // (partition, slice, class) triples at most
constexpr int kMarkMaxSlices = 8;          // every slice of a partition streams the indices again
// Below this many rows the two launches more cost what the planes' lines do (search statistics, 30
// entries a row: 54 us either way at 30K rows, 89 against 97 at 100K rows and two partitions).
constexpr int64_t kMarkMinRows = 131072;
constexpr int64_t kMarkMaxSegments = 1ll << 26;     // 8 bytes each in the workspace
constexpr int kMarkUnrollB = 8;
constexpr int kMarkFours = 4;              // loads of four entries in flight, of a segment that a wavefront walks alone
constexpr int kMarkEntries = 16384;        // entries that are worth one more workgroup

struct MarkShape {
    int slices;              // slices of a partition; 0: the bitmap path does not apply
    int words;               // bitmap words of a slice
    int64_t slice_cols;      // columns of a slice (a multiple of 32)
    int groups;              // workgroups
};

MarkShape mark_shape(int64_t rows, int64_t cols, int parts) {
    MarkShape m{};
    const int64_t psize = (cols + parts - 1) / parts;
    const int64_t slices = (psize + (int64_t)kMarkMaxWords * 32 - 1) / ((int64_t)kMarkMaxWords * 32);
    if (rows < kMarkMinRows || slices > kMarkMaxSlices || slices * parts * LF_MAX_CLASSES > kMarkItems || rows * parts > kMarkMaxSegments) return m;
    m.slices = (int)slices;
    m.slice_cols = ((psize + slices - 1) / slices + 31) / 32 * 32;
    m.words = (int)(m.slice_cols / 32);
    m.groups = m.words <= kMarkTwoPerCu ? 512 : 256;
    if (m.groups < m.slices * parts * LF_MAX_CLASSES) m.groups = kMarkItems;
    return m;
}

// lists[p * rows + first segment of class k ..) = (start, fill) of the segments of class k of partition
// p; the classes follow one another, a class's segments in the order of the workgroups' row ranges, those
// of more than kMarkBigSegment entries behind the last class.  The ranges are class_count_kernel's, whose counts say where a
// workgroup's segments go (a sweep of its own to count them again and an atomic per class and workgroup: 27 us for 2.45M rows, this 12).
__global__ void __launch_bounds__(kCountThreads)
class_list_kernel(SegView v, const int32_t* __restrict__ seg_deg, int kmax, const int32_t* __restrict__ counts, int2* __restrict__ lists) {
    __shared__ uint32_t s_at[kCountClasses], s_all[kCountClasses];
    const int p = blockIdx.y;
    {
        const int k = threadIdx.x >> 6, part = threadIdx.x & 63;
        uint32_t before = 0, all = 0;
        for (int g = part; g < (int)gridDim.x; g += 64) {
            const uint32_t n = (uint32_t)counts[count_at(p, k, g)];
            all += n;
            before += g < (int)blockIdx.x ? n : 0u;
        }
        for (int d = 1; d < 64; d <<= 1) {
            before += __shfl_xor(before, d);
            all += __shfl_xor(all, d);
        }
        if (part == 0) {
            s_at[k] = before;
            s_all[k] = all;
        }
    }
    __syncthreads();
    if (threadIdx.x < kCountClasses) {
        uint32_t first = s_at[threadIdx.x];
        for (int i = 0; i < (int)threadIdx.x; ++i) first += s_all[i];
        s_at[threadIdx.x] = first;
    }
    __syncthreads();
    const int64_t per = (v.rows + gridDim.x - 1) / gridDim.x;
    const int64_t lo = (int64_t)blockIdx.x * per, hi = lo + per < v.rows ? lo + per : v.rows;
    int2* out = lists + (size_t)p * (size_t)v.rows;
    for (int64_t r0 = lo + threadIdx.x; r0 < hi; r0 += kRowUnroll * kCountThreads) {
        int deg[kRowUnroll], start[kRowUnroll], fill[kRowUnroll];
        seg_degrees(v, seg_deg, p, r0, kCountThreads, hi, start, fill, deg);
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) {
            int k, cost_rows;
            if (deg[u] <= 0) continue;
            width_class(deg[u], kmax, k, cost_rows);
            out[atomicAdd(&s_at[deg[u] > kMarkBigSegment && k == kmax ? kmax + 1 : k], 1u)] = make_int2(start[u], fill[u]);
        }
    }
}

// Four entries of a segment with one load, which need only be aligned as they are; the last lanes of a segment move back to end where
// it ends and mark entries twice.
struct __attribute__((packed, aligned(4))) Four { uint32_t c[4]; };
constexpr int kMarkPiece = 256 * kMarkFours;

// Marks up to kMarkPiece entries of a segment from its entry j on.
template <int N, typename Mark>
__device__ __forceinline__ void mark_fours(const int32_t* __restrict__ first, int j, int fill, Mark mark) {
    const int lane = threadIdx.x & 63;
    Four f[N];
#pragma unroll
    for (int u = 0; u < N; ++u) f[u] = *(const Four*)(first + min(j + u * 256 + lane * 4, fill - 4));
#pragma unroll
    for (int u = 0; u < N; ++u)
        for (int i = 0; i < 4; ++i) mark(f[u].c[i], j + u * 256 + lane * 4 < fill);
}
template <typename Mark>
__device__ __forceinline__ void mark_piece(const int32_t* __restrict__ indices, int start, int j, int fill, Mark mark) {
    const int lane = threadIdx.x & 63;
    if (fill - j > 256)
        mark_fours<kMarkFours>(indices + start, j, fill, mark);
    else if (fill >= 4)
        mark_fours<1>(indices + start, j, fill, mark);
    else if (lane < fill)
        mark((uint32_t)indices[start + lane], true);
}

// The segments of the last class, of any length, one at a time per wavefront.
template <typename Mark>
__device__ __forceinline__ void mark_long(const int32_t* __restrict__ indices, const int2* __restrict__ list, int n_seg,
                                          int first_wave, int waves, Mark mark) {
    int2 seg = first_wave < n_seg ? list[first_wave] : make_int2(0, 0);
    for (int i = first_wave; i < n_seg; i += waves) {
        const int start = __builtin_amdgcn_readfirstlane(seg.x), fill = __builtin_amdgcn_readfirstlane(seg.y);
        if (i + waves < n_seg) seg = list[i + waves];                // a round ahead
        for (int j = 0; j < fill; j += kMarkPiece) mark_piece(indices, start, j, fill, mark);
    }
}

// Lanes that hold no segment of `least` entries or more point to one that another lane holds, with no entries: then every lane can
// load.  (Loads behind a condition are branches, and the compiler waited for each before it used the next one's registers: one load
// of a wavefront under way at a time instead of eight.)  False where no lane holds one.
__device__ __forceinline__ bool spare_lanes(int2& seg, int least) {
    const unsigned long long held = __ballot(seg.y >= least);
    if (held == 0) return false;
    const int start = __builtin_amdgcn_readlane(seg.x, __builtin_ctzll(held));
    if (seg.y < least) seg = make_int2(start, 0);
    return true;
}

// Marks the segments of class k < 3 (at most 2^k entries) that fall to one wavefront.
// The wavefront takes 64 segments at a time, one lane holding each, and walks them in steps of 64 >> K segments side by side, eight
// steps' loads in flight.
template <int K, typename Mark>
__device__ __forceinline__ void mark_short(const int32_t* __restrict__ indices, const int2* __restrict__ list, int n_seg,
                                           int first_wave, int waves, Mark mark) {
    constexpr int kSide = 64 >> K, kSteps = 1 << K, kFlight = kSteps < kMarkUnrollB ? kSteps : kMarkUnrollB;
    const int lane = threadIdx.x & 63;
    const int q = lane & ((1 << K) - 1), sub = lane >> K;
    int64_t i0 = (int64_t)first_wave * 64;
    const int64_t stride = (int64_t)waves * 64;
    int2 seg = make_int2(0, 0);
    if (i0 + lane < n_seg) seg = list[i0 + lane];
    for (; i0 < n_seg; i0 += stride) {
        int2 cur = seg;
        seg = make_int2(0, 0);
        if (i0 + stride + lane < n_seg) seg = list[i0 + stride + lane];      // a round ahead
        if (!spare_lanes(cur, 1)) continue;
#pragma unroll
        for (int t0 = 0; t0 < kSteps; t0 += kFlight) {
            uint32_t c[kFlight];
            bool on[kFlight];
#pragma unroll
            for (int u = 0; u < kFlight; ++u) {
                const int start = __shfl(cur.x, (t0 + u) * kSide + sub), fill = __shfl(cur.y, (t0 + u) * kSide + sub);
                on[u] = q < fill;
                c[u] = (uint32_t)indices[start + max(min(q, fill - 1), 0)];
            }
#pragma unroll
            for (int u = 0; u < kFlight; ++u)
                mark(c[u], on[u]);
        }
    }
}

// Marks the segments of class k >= 3 (at most 2^k entries) that fall to one wavefront; L = min(k - 2, 6).
// A lane takes four entries with one load of 16 bytes, which need only be aligned as the entries are; the last lane of a segment
// moves back to end where it ends and marks up to three entries twice.  So 64 >> L segments are walked side by side, or 256 entries of a
// longer one.
template <int L, typename Mark>
__device__ __forceinline__ void mark_class(const int32_t* __restrict__ indices, const int2* __restrict__ list, int n_seg,
                                           int k, int first_wave, int waves, Mark mark) {
    constexpr int kSide = 64 >> L;                     // segments side by side
    constexpr int kFlight = L < 3 ? 1 << L : 8;        // (never more than a group's steps; 8 against 4: 130 -> 124 us)
    const int lane = threadIdx.x & 63;
    const int q = lane & ((1 << L) - 1), sub = lane >> L;
    const int log_pieces = k - 2 - L;                  // L < 6: 0
    const int group = max(64 >> max(k - 6, 0), 4);     // segments of a group: about as many entries in every class
    const int steps = (group / kSide) << log_pieces;
    int64_t i0 = (int64_t)first_wave * group;
    const int64_t stride = (int64_t)waves * group;
    int2 seg = make_int2(0, 0);
    if (lane < group && i0 + lane < n_seg) seg = list[i0 + lane];
    for (; i0 < n_seg; i0 += stride) {
        int2 cur = seg;
        seg = make_int2(0, 0);
        if (lane < group && i0 + stride + lane < n_seg) seg = list[i0 + stride + lane];      // a round ahead
        // (a segment's class is that of its degree, which may count twice what the structure holds once)
        if (__ballot(cur.y > 0 && cur.y < 4) != 0)
            for (int i = 0; i < cur.y && cur.y < 4; ++i) mark((uint32_t)indices[cur.x + i]);
        if (!spare_lanes(cur, 4)) continue;
        for (int t0 = 0; t0 < steps; t0 += kFlight) {
            Four f[kFlight];
            bool on[kFlight];
#pragma unroll
            for (int u = 0; u < kFlight; ++u) {
                const int t = t0 + u;
                int start, fill, at = q * 4;
                if constexpr (L == 6) {
                    const int src = (t >> log_pieces) & 63;
                    start = __builtin_amdgcn_readlane(cur.x, src);
                    fill = __builtin_amdgcn_readlane(cur.y, src);
                    at += (t & ((1 << log_pieces) - 1)) << 8;
                } else {
                    start = __shfl(cur.x, (t * kSide + sub) & 63);
                    fill = __shfl(cur.y, (t * kSide + sub) & 63);
                }
                on[u] = at < fill;
                f[u] = *(const Four*)(indices + start + max(min(at, fill - 4), 0));
            }
#pragma unroll
            for (int u = 0; u < kFlight; ++u)
                for (int j = 0; j < 4; ++j) mark(f[u].c[j], on[u]);
        }
    }
}

// One workgroup per slice and share of an item (partition p, class k), i = p * classes + k: places for a workgroup of every slice are
// dealt out in proportion to the entries of the item, at least one to an item that has any.  table[i] = first place of item i,
// table[n_items] = places in use; slice s of place j writes bitmap s * (groups / slices) + j.
__global__ void __launch_bounds__(kMarkThreads)
mark_columns_kernel(const int32_t* __restrict__ indices, const int2* __restrict__ lists, int64_t rows, int parts,
                    int num_classes, MarkShape shape, int64_t psize, int64_t cols,
                    const unsigned long long* __restrict__ stats, int32_t* __restrict__ table,
                    uint32_t* __restrict__ bitmaps) {
    extern __shared__ uint32_t s_bits[];
    __shared__ int s_first[kMarkItems + 1];
    __shared__ unsigned long long s_sum[kMarkThreads / 64];
    __shared__ int s_cnt[kMarkThreads / 64];
    __shared__ int s_item;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n_items = parts * num_classes;

    // ---- workgroup -> (slice s, place j): the workgroups of a place are eight apart, on one XCD, and read the same lines
    const int S = shape.slices, places = gridDim.x / S, whole = gridDim.x / (8 * S) * 8;      // whole: places in full rounds of eight
    int s, j;
    if ((int)blockIdx.x < whole * S) {
        s = (int)blockIdx.x / 8 % S;
        j = (int)blockIdx.x / (8 * S) * 8 + (int)blockIdx.x % 8;
    } else {
        const int rest = (int)blockIdx.x - whole * S, left = max(places - whole, 1);
        s = rest / left;
        j = whole + rest % left;
        if (s >= S || j >= places) return;
    }

    // ---- which item, and which share of it
    unsigned long long w = 0;
    if (tid < n_items) {
        const int kk = tid % num_classes, pp = tid / num_classes;
        const unsigned long long entries = stats[stat_at(pp, kk, 1)], segs = stats[stat_at(pp, kk, 2)];
        w = entries + 6 * segs;                        // as their times were; fewer loads are under way
        if (kk < 3) w += w / 2;                        // where a group's steps are few
        if (kk == num_classes - 1) w += w / 8;         // or a wavefront has one segment
    }
    unsigned long long sum = w;
    for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d);
    if (lane == 0) { s_sum[wave] = sum; }
    const int nz_wave = __popcll(__ballot(w > 0));
    if (lane == 0) s_cnt[wave] = nz_wave;
    __syncthreads();
    unsigned long long total = 0;
    int nz = 0;
    for (int i = 0; i < kMarkThreads / 64; ++i) { total += s_sum[i]; nz += s_cnt[i]; }
    const unsigned long long worth = total / kMarkEntries;      // a small matrix is not spread over more bitmaps than it pays for
    const unsigned long long more = worth < (unsigned long long)(places - nz) ? worth : places - nz;
    const int m = w > 0 ? 1 + (int)(more * w / total) : 0;
    int incl = m;
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(incl, d);
        if (lane >= d) incl += y;
    }
    __syncthreads();
    if (lane == 63) s_cnt[wave] = incl;
    if (tid == 0) s_item = -1;
    __syncthreads();
    int before = incl - m;
    for (int i = 0; i < wave; ++i) before += s_cnt[i];
    if (tid < n_items) {
        s_first[tid] = before;
        if (tid == n_items - 1) s_first[n_items] = before + m;
        if (j >= before && j < before + m) s_item = tid;
    }
    for (int i = tid; i < shape.words; i += kMarkThreads) s_bits[i] = 0;
    __syncthreads();
    if (blockIdx.x == 0)
        for (int i = tid; i <= n_items; i += kMarkThreads) table[i] = s_first[i];
    const int item = s_item;
    if (item < 0) return;                              // more places than shares

    const int k = item % num_classes, p = item / num_classes;
    const int share = j - s_first[item], shares = s_first[item + 1] - s_first[item];
    const int64_t c0 = (int64_t)p * psize + (int64_t)s * shape.slice_cols;
    int64_t c1 = c0 + shape.slice_cols;
    if (c1 > (int64_t)(p + 1) * psize) c1 = (int64_t)(p + 1) * psize;
    if (c1 > cols) c1 = cols;
    const uint32_t span = c1 > c0 ? (uint32_t)(c1 - c0) : 0u;
    const uint32_t base_col = (uint32_t)c0;
    uint32_t first = 0;
    for (int i = 0; i < k; ++i) first += (uint32_t)stats[stat_at(p, i, 2)];
    const int n_big = k == num_classes - 1 ? (int)stats[stat_at(p, k, 2) + 2] : 0;
    const int n_seg = (int)stats[stat_at(p, k, 2)] - n_big;
    const int2* list = lists + (size_t)p * (size_t)rows + first;
    auto mark = [&](uint32_t c, bool on = true) {
        const uint32_t x = c - base_col;               // (wraps to a large value below the slice)
        if (x < (on ? span : 0u)) atomicOr(&s_bits[x >> 5], 1u << (x & 31u));
    };

    const int waves = shares * (kMarkThreads / 64);
    const int first_wave = share * (kMarkThreads / 64) + wave;
    switch (k < num_classes - 1 ? k : LF_MAX_CLASSES) {
        case 0: mark_short<0>(indices, list, n_seg, first_wave, waves, mark); break;
        case 1: mark_short<1>(indices, list, n_seg, first_wave, waves, mark); break;
        case 2: mark_short<2>(indices, list, n_seg, first_wave, waves, mark); break;
        case 3: mark_class<1>(indices, list, n_seg, k, first_wave, waves, mark); break;
        case 4: mark_class<2>(indices, list, n_seg, k, first_wave, waves, mark); break;
        case 5: mark_class<3>(indices, list, n_seg, k, first_wave, waves, mark); break;
        case 6: mark_class<4>(indices, list, n_seg, k, first_wave, waves, mark); break;
        case 7: mark_class<5>(indices, list, n_seg, k, first_wave, waves, mark); break;
        default:
            if (k < num_classes - 1) mark_class<6>(indices, list, n_seg, k, first_wave, waves, mark);
            break;
    }
    if (k == num_classes - 1) mark_long(indices, list, n_seg, first_wave, waves, mark);
    for (int i = 0; i < n_big; ++i) {
        const int2 seg = list[n_seg + i];
        const int64_t stride = (int64_t)waves * kMarkPiece;
        for (int64_t at = (int64_t)first_wave * kMarkPiece; at < seg.y; at += stride)
            mark_piece(indices, seg.x, (int)at, seg.y, mark);
    }
    __syncthreads();
    uint32_t* out = bitmaps + ((size_t)s * places + j) * shape.words;
    for (int i = tid; i < shape.words; i += kMarkThreads) out[i] = s_bits[i];
}

// hist[p][mask] from the bitmaps; blockIdx.y = p * slices + s.  A workgroup takes tiles of 64 words:
// thread (class, word) ORs the bitmaps of the workgroups that shared the item, all classes' loads in
// flight together, then every thread builds the masks of two of the tile's 2048 columns.
constexpr int kHistThreads = 1024;
constexpr int kHistGrid = 256;
__global__ void __launch_bounds__(kHistThreads)
colbits_hist_kernel(const uint32_t* __restrict__ bitmaps, const int32_t* __restrict__ table, int num_classes,
                    MarkShape shape, int64_t psize, int64_t cols, unsigned long long* __restrict__ hist) {
    constexpr int kBins = 1 << LF_MAX_CLASSES;
    __shared__ uint32_t s_hist[kBins];
    __shared__ uint32_t s_bits[16][64];
    for (int i = threadIdx.x; i < kBins; i += kHistThreads) s_hist[i] = 0;
    const int p = blockIdx.y / shape.slices, s = blockIdx.y % shape.slices;
    const int64_t c0 = (int64_t)p * psize + (int64_t)s * shape.slice_cols;
    int64_t c1 = c0 + shape.slice_cols;
    if (c1 > (int64_t)(p + 1) * psize) c1 = (int64_t)(p + 1) * psize;
    if (c1 > cols) c1 = cols;
    const int k = threadIdx.x >> 6, word = threadIdx.x & 63;
    int g0 = 0, g1 = 0;
    if (k < num_classes) {
        const int first = s * (shape.groups / shape.slices);
        g0 = first + table[p * num_classes + k];
        g1 = first + table[p * num_classes + k + 1];
    }
    for (int w0 = blockIdx.x * 64; w0 < shape.words && c0 + (int64_t)w0 * 32 < c1; w0 += gridDim.x * 64) {      // uniform
        uint32_t bits = 0;
        if (w0 + word < shape.words) {
            for (int g = g0; g < g1; g += 8) {
                uint32_t x[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) x[u] = bitmaps[(size_t)min(g + u, g1 - 1) * shape.words + w0 + word];
#pragma unroll
                for (int u = 0; u < 8; ++u) bits |= x[u];
            }
        }
        s_bits[k][word] = bits;
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int c = h * kHistThreads + threadIdx.x;        // column of the tile
            if (c0 + (int64_t)w0 * 32 + c < c1) {
                uint32_t mask = 0;
#pragma unroll
                for (int i = 0; i < LF_MAX_CLASSES; ++i) mask |= ((s_bits[i][c >> 5] >> (c & 31)) & 1u) << i;
                atomicAdd(&s_hist[mask], 1u);
            }
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < kBins; i += kHistThreads)
        if (s_hist[i]) atomicAdd(&hist[(size_t)p * kBins + i], (unsigned long long)s_hist[i]);
}

// ---------------------------------------------------------------------------- hyb plan/build
// Width table on the device: wtab[p][0] = count, wtab[p][1 + b] = width, wtab[p][12] = index
// of the partition's first bucket in the flat (p, b) bucket order.
constexpr int kWtabStride = 16;

// Bucket of a segment: first width >= deg, else the widest (format_algos.py:275-279).
__device__ __forceinline__ int pick_bucket(const int32_t* __restrict__ w, int n, int deg) {
    int b = 0;
    while (b < n && w[1 + b] < deg) ++b;
    return b == n ? n - 1 : b;
}

// Per workgroup of kBlock rows and per bucket: number of ELL rows the block contributes.
// blockcnt[(bucket_base[p] + b) * nblk + blk]
__global__ void __launch_bounds__(kBlock)
hyb_count_kernel(SegView v, const int32_t* __restrict__ seg_deg, const int32_t* __restrict__ wtab,
                 int nblk, int32_t* __restrict__ blockcnt, int32_t* __restrict__ flags) {
    __shared__ int s_cnt[LF_MAX_CLASSES];
    if (threadIdx.x < LF_MAX_CLASSES) s_cnt[threadIdx.x] = 0;
    __syncthreads();
    const int p = blockIdx.y;
    const int32_t* w = wtab + p * kWtabStride;
    const int n = w[0];
    const int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (r < v.rows) {
        int start, fill;
        seg_range(v, r, p, start, fill);
        if (fill > 0) {
            if (n == 0) {
                atomicOr(&flags[0], 1);       // nonzeros in a partition without widths
            } else {
                const int deg = seg_deg ? seg_deg[(int64_t)p * v.rows + r] : fill;
                const int b = pick_bucket(w, n, deg);
                const int width = w[1 + b];
                const int n_ell = (fill + width - 1) / width;
                if (n_ell > kMetaSegMax) atomicOr(&flags[0], 2);
                atomicAdd(&s_cnt[b], n_ell);
            }
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < n)
        blockcnt[(int64_t)(w[12] + threadIdx.x) * nblk + blockIdx.x] = s_cnt[threadIdx.x];
}

struct BucketOffsets {
    long long slot_off;    // first slot of the bucket in the flat slab arrays
    long long row_off;     // first ELL row of the bucket in the flat row arrays
};

// Flat slab layout shared by the builder and its callers: ELL rows of bucket k start at a
// multiple of 64 entries, its slots at a multiple of 1024, so every slab is at least 256-byte
// aligned inside 256-byte aligned allocations.
constexpr int64_t kRowAlign = 64;
constexpr int64_t kSlotAlign = 1024;
__host__ __device__ inline void flat_layout_step(int64_t ell_rows, int64_t width, int64_t* rows, int64_t* slots) {
    *rows += (ell_rows + kRowAlign - 1) / kRowAlign * kRowAlign;
    *slots += (ell_rows * width + kSlotAlign - 1) / kSlotAlign * kSlotAlign;
}

// Exclusive scan over blocks, one workgroup per bucket; totals[k] = ELL rows of bucket k.  The
// workgroup that ends last derives the flat layout from the totals, so that the fill needs
// nothing more from the host, and leaves flags and totals in the host's (pinned) memory, if that is given.
__global__ void __launch_bounds__(1024)
hyb_scan_kernel(int32_t* __restrict__ blockcnt, int nblk, long long* __restrict__ totals,
                const int32_t* __restrict__ widths, int* __restrict__ done, BucketOffsets* __restrict__ offs,
                const int* __restrict__ flags, int* h_flags, long long* h_totals) {
    __shared__ long long s_wave[16];
    __shared__ int s_last;
    int32_t* a = blockcnt + (int64_t)blockIdx.x * nblk;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // a thread's consecutive blocks, then one scan over the threads (a scan over 1024 blocks at a time, with its barriers,
    // was 18 us for 9571 blocks, this is 7)
    const int per = (nblk + 1023) / 1024, from = min((int)threadIdx.x * per, nblk), to = min(from + per, nblk);
    long long mine = 0;
#pragma unroll 8
    for (int i = from; i < to; ++i) mine += a[i];
    long long incl = mine;
    for (int d = 1; d < 64; d <<= 1) {
        const long long y = __shfl_up(incl, d);
        if (lane >= d) incl += y;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    long long before = incl - mine, all = 0;
    for (int w = 0; w < 16; ++w) {
        before += w < wave ? s_wave[w] : 0;
        all += s_wave[w];
    }
#pragma unroll 8
    for (int i = from; i < to; ++i) {
        const int x = a[i];
        a[i] = (int32_t)before;
        before += x;
    }
    if (threadIdx.x == 0) {
        __hip_atomic_store(&totals[blockIdx.x], all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // (release: the total above is visible before the count; acquire: so are the others')
        s_last = __hip_atomic_fetch_add(done, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
    }
    __syncthreads();
    if (!s_last) return;
    const int nb = gridDim.x;
    if (h_flags && threadIdx.x == 0) *h_flags = *flags;           // (hyb_count_kernel's)
    int64_t row = 0, slot = 0;                        // carried by thread 0
    for (int base = 0; base < nb; base += 1024) {     // staged through LDS: the layout is a serial sum
        __shared__ long long s_rows[1024];
        __shared__ int s_width[1024];
        const int i = base + threadIdx.x;
        if (i < nb) {
            s_rows[threadIdx.x] = __hip_atomic_load(&totals[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_width[threadIdx.x] = widths[i];
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int k = 0; k < 1024 && base + k < nb; ++k) {
                offs[base + k] = BucketOffsets{slot, row};
                flat_layout_step(s_rows[k], s_width[k], &row, &slot);
            }
        }
        if (h_totals && i < nb) h_totals[i] = s_rows[threadIdx.x];
        __syncthreads();
    }
}

// Fills the slabs.  One workgroup per 256 source rows, four column partitions at a time.
//   * one thread per (row, partition) segment finds the segment's bucket and its first ELL
//     row (per-wavefront counts per bucket - bit counts, or a shuffle scan where segments
//     split - combined through LDS with a single barrier) and writes the rows / meta entries;
//   * the workgroup then walks the concatenation of the 256 segments, each padded to whole
//     ELL rows: consecutive threads take consecutive groups of four slots (group -> segment
//     by a binary search over LDS prefix sums), so the CSR entries are read in order and
//     each segment's ELL rows, which are consecutive in the slab, are written in order,
//     padding included, with 16-byte accesses wherever a group lies inside one row.
// Reading in row order matters: a source row is ~130 bytes at an arbitrary offset, and when
// the slabs were filled bucket by bucket every row cost two full cache lines (1.27 GB fetched
// for 0.65 GB of entries on an 81.6M-nonzero matrix).  Bound by memory: that matrix, 0.65 GB read and 0.75 GB written, takes 295 us, 4.8
// TB/s (322 with the loads of a group behind conditions, which made a step of four groups wait four times).
constexpr int kFillUnroll = 4;
constexpr int kPartGroup = 4;        // column partitions whose segments are walked together
// four consecutive 32-bit values at a 4-byte aligned address (one 16-byte load)
struct __attribute__((packed, aligned(4))) Packed4i { int x, y, z, w; };
struct __attribute__((packed, aligned(4))) Packed4f { float x, y, z, w; };

__global__ void __launch_bounds__(kBlock)
hyb_fill_kernel(SegView v, const int32_t* __restrict__ seg_deg, const int32_t* __restrict__ wtab,
                int nblk, const int32_t* __restrict__ blockoff, const BucketOffsets* __restrict__ offs,
                const int32_t* __restrict__ indices, const float* __restrict__ values,
                int32_t* __restrict__ out_rows, int32_t* __restrict__ out_meta,
                int32_t* __restrict__ out_cols, float* __restrict__ out_vals, float* __restrict__ out_mask) {
    // segment tables of the walk, entry t * pg + pp for row t and the pp-th partition of the
    // group of pg <= kPartGroup partitions in hand: row-major, so the walk reads each row's CSR
    // entries once and in order however many partitions cut it
    constexpr int kSegs = kBlock * kPartGroup;
    __shared__ int s_cnt[kBlock / 64][LF_MAX_CLASSES + 1];
    // exclusive prefix of the padded segment lengths; 32 bits are enough: a segment is padded
    // by less than 1024 slots and the matrix holds fewer than 2^31 entries
    __shared__ uint32_t s_off[kSegs + 1];
    __shared__ long long s_dst[kSegs];         // first slab slot of each segment
    __shared__ int s_start[kSegs];
    __shared__ int s_fill[kSegs];
    __shared__ uint32_t s_len[kSegs];
    __shared__ uint32_t s_wave[kBlock / 64];
    const int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nnz = v.indptr[v.rows];

    for (int p0 = 0; p0 < v.parts; p0 += kPartGroup) {
        const int pg = min(kPartGroup, v.parts - p0);
        uint32_t vl[kPartGroup];
#pragma unroll
        for (int pp = 0; pp < kPartGroup; ++pp) {
            vl[pp] = 0;
            if (pp >= pg) continue;                    // uniform
            const int p = p0 + pp;
            const int32_t* w = wtab + p * kWtabStride;
            const int n = w[0];
            const int kbase = w[12];
            int start = 0, fill = 0, mine = -1, width = 1, n_ell = 0;
            if (r < v.rows && n > 0) {
                seg_range(v, r, p, start, fill);
                if (fill > 0) {
                    const int deg = seg_deg ? seg_deg[(int64_t)p * v.rows + r] : fill;
                    mine = pick_bucket(w, n, deg);
                    width = w[1 + mine];
                    n_ell = (fill + width - 1) / width;
                }
            }
            // ELL rows of the same bucket that precede this segment inside its wavefront.  Only
            // the widest bucket splits segments; where every segment is one ELL row a bit count
            // does it.
            int in_wave = 0;
            for (int b = 0; b < n; ++b) {
                const unsigned long long members = __ballot(mine == b);
                if (__ballot(mine == b && n_ell != 1) == 0) {
                    if (mine == b) in_wave = __popcll(members & ((1ull << lane) - 1ull));
                    if (lane == 0) s_cnt[wave][b] = __popcll(members);
                } else {
                    const int x = mine == b ? n_ell : 0;
                    int incl = x;
                    for (int d = 1; d < 64; d <<= 1) {
                        const int y = __shfl_up(incl, d);
                        if (lane >= d) incl += y;
                    }
                    if (mine == b) in_wave = incl - x;
                    if (lane == 63) s_cnt[wave][b] = incl;
                }
            }
            __syncthreads();
            long long first = 0;      // flat ELL-row index of this segment's first ELL row
            long long dst = 0;
            if (mine >= 0) {
                int wave_off = 0;
                for (int wv = 0; wv < wave; ++wv) wave_off += s_cnt[wv][mine];
                const BucketOffsets bo = offs[kbase + mine];
                const long long local = (long long)blockoff[(int64_t)(kbase + mine) * nblk + blockIdx.x] + wave_off + in_wave;
                first = bo.row_off + local;
                dst = bo.slot_off + local * width;
            }
            const uint32_t slen = (uint32_t)n_ell * (uint32_t)width;   // slots of the segment's ELL rows
            vl[pp] = (slen + 3u) & ~3u;
            const int idx = threadIdx.x * pg + pp;
            s_dst[idx] = dst;
            s_start[idx] = start;
            s_fill[idx] = fill;
            s_len[idx] = slen;

            const bool is_long = n_ell > 8;
            if (n_ell > 0 && !is_long) {
                for (int i = 0; i < n_ell; ++i) {
                    const int len = min(width, fill - i * width);
                    out_rows[first + i] = (int32_t)r;
                    out_meta[first + i] = make_meta(len, i, n_ell);
                }
            }
            unsigned long long pending = __ballot(is_long);
            while (pending) {
                const int src = __ffsll((long long)pending) - 1;
                pending &= pending - 1;
                const long long f0 = __shfl(first, src);
                const int fl = __shfl(fill, src);
                const int wd = __shfl(width, src);
                const int ne = __shfl(n_ell, src);
                const int rr = (int)((int64_t)blockIdx.x * kBlock + (wave << 6) + src);
                for (int i = lane; i < ne; i += 64) {
                    const int len = min(wd, fl - i * wd);
                    out_rows[f0 + i] = rr;
                    out_meta[f0 + i] = make_meta(len, i, ne);
                }
            }
            __syncthreads();          // s_cnt is rewritten for the next partition
        }

        // exclusive prefix of the padded lengths over (row, partition)
        uint32_t mine_total = 0;
#pragma unroll
        for (int pp = 0; pp < kPartGroup; ++pp) mine_total += vl[pp];
        uint32_t vincl = mine_total;
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(vincl, d);
            if (lane >= d) vincl += y;
        }
        if (lane == 63) s_wave[wave] = vincl;
        __syncthreads();
        uint32_t voff = vincl - mine_total;
        for (int wv = 0; wv < wave; ++wv) voff += s_wave[wv];
#pragma unroll
        for (int pp = 0; pp < kPartGroup; ++pp) {
            if (pp < pg) s_off[threadIdx.x * pg + pp] = voff;
            voff += vl[pp];
        }
        if (threadIdx.x == kBlock - 1) s_off[kBlock * pg] = voff;
        __syncthreads();

        // groups of four consecutive slots; the prefix sums are multiples of four, so a group
        // never straddles two segments
        const int n_seg = kBlock * pg;
        const int steps = 8 + (pg > 1) + (pg > 2);       // ceil(log2(n_seg))
        const uint32_t total = s_off[n_seg];
        // Every lane loads four entries, whatever the group holds of them: behind a condition each load would be waited for before the
        // next.  The last groups of the index array move back to end where it ends and shift.
        auto walk = [&](auto tiny) {                  // tiny: the array has fewer than four entries
            for (uint32_t j0 = 0; j0 < total; j0 += kBlock * kFillUnroll * 4) {
                long long at[kFillUnroll];
                int len[kFillUnroll];                 // slots of the group inside its segment (0: none)
                int live[kFillUnroll], shift[kFillUnroll];
                int4 c[kFillUnroll];
                float4 x[kFillUnroll];
#pragma unroll
                for (int u = 0; u < kFillUnroll; ++u) {
                    const uint32_t mine = j0 + (u * kBlock + threadIdx.x) * 4, j = min(mine, total - 4);
                    int lo = 0, hi = n_seg - 1;        // last segment whose offset is <= j
                    for (int step = 0; step < steps; ++step) {
                        const int mid = (lo + hi + 1) >> 1;
                        if (s_off[mid] <= j) lo = mid; else hi = mid - 1;
                    }
                    const int q = (int)(j - s_off[lo]);
                    live[u] = s_fill[lo] - q;          // entries of the source row from q on
                    at[u] = s_dst[lo] + q;
                    len[u] = mine < total ? min(4, (int)s_len[lo] - q) : 0;
                    const int from = tiny ? 0 : lf::group_source(s_start[lo], q, nnz);
                    shift[u] = live[u] > 0 ? s_start[lo] + q - from : 0;
                    x[u] = make_float4(1.f, 1.f, 1.f, 1.f);
                    if constexpr (tiny) {
                        const int last = max(nnz - 1, 0);
                        if (nnz > 0) {
                            c[u] = make_int4(indices[0], indices[min(1, last)], indices[min(2, last)], 0);
                            if (values) x[u] = make_float4(values[0], values[min(1, last)], values[min(2, last)], 0.f);
                        }
                    } else {
                        const Packed4i ci = *reinterpret_cast<const Packed4i*>(indices + from);
                        c[u] = make_int4(ci.x, ci.y, ci.z, ci.w);
                        if (values) {
                            const Packed4f xv = *reinterpret_cast<const Packed4f*>(values + from);
                            x[u] = make_float4(xv.x, xv.y, xv.z, xv.w);
                        }
                    }
                }
#pragma unroll
                for (int u = 0; u < kFillUnroll; ++u) {
                    if (__ballot(shift[u] != 0) != 0)
                        for (int i = 0; i < 3; ++i)
                            if (shift[u] > i) {
                                c[u].x = c[u].y, c[u].y = c[u].z, c[u].z = c[u].w;
                                x[u].x = x[u].y, x[u].y = x[u].z, x[u].z = x[u].w;
                            }
                    const bool v0 = live[u] > 0, v1 = live[u] > 1, v2 = live[u] > 2, v3 = live[u] > 3;
                    const int4 cc4 = make_int4(v0 ? c[u].x : 0, v1 ? c[u].y : 0, v2 ? c[u].z : 0, v3 ? c[u].w : 0);
                    const float4 xx4 = make_float4(v0 ? x[u].x : 0.f, v1 ? x[u].y : 0.f, v2 ? x[u].z : 0.f, v3 ? x[u].w : 0.f);
                    const float4 mm4 = make_float4(v0, v1, v2, v3);
                    if (len[u] == 4 && (at[u] & 3) == 0) {
                        *reinterpret_cast<int4*>(out_cols + at[u]) = cc4;
                        *reinterpret_cast<float4*>(out_vals + at[u]) = xx4;
                        if (out_mask) *reinterpret_cast<float4*>(out_mask + at[u]) = mm4;
                    } else {
                        const int cc[4] = {cc4.x, cc4.y, cc4.z, cc4.w};
                        const float xx[4] = {xx4.x, xx4.y, xx4.z, xx4.w};
                        const float mm[4] = {mm4.x, mm4.y, mm4.z, mm4.w};
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            if (i < len[u]) {
                                out_cols[at[u] + i] = cc[i];
                                out_vals[at[u] + i] = xx[i];
                                if (out_mask) out_mask[at[u] + i] = mm[i];
                            }
                        }
                    }
                }
            }
        };
        if (nnz >= 4) walk(std::false_type{});
        else walk(std::true_type{});
        __syncthreads();          // the tables are rewritten for the next group of partitions
    }
}

// ---------------------------------------------------------------------------- host helpers
struct StatsLayout {
    size_t bnd, planes, lists, counts, bitmaps, table, stats, hist, total;
};

StatsLayout stats_layout(int64_t rows, int64_t cols, int parts) {
    StatsLayout L{};
    size_t off = 0;
    L.bnd = off;
    if (parts > 1) off += align_up((size_t)(parts + 1) * rows * 4, 256);
    const MarkShape m = mark_shape(rows, cols, parts);
    L.planes = L.lists = L.bitmaps = L.table = off;      // byte planes, or segment lists and bitmaps
    if (m.slices > 0) {
        off += align_up((size_t)parts * (size_t)rows * 8, 256);
        L.counts = off;
        off += align_up(count_at(parts, 0, 0) * 4, 256);
        L.bitmaps = off;
        off += align_up((size_t)m.groups * (size_t)m.words * 4, 256);
        L.table = off;
        off += align_up((size_t)(kMarkItems + 1) * 4, 256);
    } else {
        off += align_up((size_t)LF_MAX_CLASSES * (size_t)cols, 256);
    }
    L.stats = off;
    off += align_up(stat_at(parts, 0, 0) * 8, 256);
    L.hist = off;
    off += align_up((size_t)parts * (1 << LF_MAX_CLASSES) * 8, 256);
    L.total = off;
    return L;
}

struct HybLayout {
    size_t bnd, wtab, widths, flags, totals, scatter, blockcnt, total;
    int nblk;
};

HybLayout hyb_layout(int64_t rows, int parts, int total_buckets) {
    HybLayout L{};
    L.nblk = (int)((rows + kBlock - 1) / kBlock);
    if (L.nblk < 1) L.nblk = 1;
    size_t off = 0;
    L.bnd = off;
    if (parts > 1) off += align_up((size_t)(parts + 1) * rows * 4, 256);
    L.wtab = off;
    off += align_up((size_t)parts * kWtabStride * 4, 256);
    L.widths = off;                     // (behind wtab: they go up together)
    off += align_up((size_t)std::max(total_buckets, 1) * 4, 256);
    L.flags = off;                      // error flags, finished workgroups of the scan
    off += 256;
    L.totals = off;                     // (behind the flags: cleared and read back together)
    off += align_up((size_t)std::max(total_buckets, 1) * 8, 256);
    L.scatter = off;
    off += align_up((size_t)std::max(total_buckets, 1) * sizeof(BucketOffsets), 256);
    L.blockcnt = off;
    off += align_up((size_t)std::max(total_buckets, 1) * L.nblk * 4, 256);
    L.total = off;
    return L;
}

void flat_layout(const int64_t* ell_rows, const int32_t* widths, int nb, int64_t* row_off,
                 int64_t* slot_off, int64_t* total_rows, int64_t* total_slots) {
    int64_t r = 0, s = 0;
    for (int k = 0; k < nb; ++k) {
        row_off[k] = r;
        slot_off[k] = s;
        flat_layout_step(ell_rows[k], widths[k], &r, &s);
    }
    *total_rows = r;
    *total_slots = s;
}

int check_common(const int32_t* d_indptr, const int32_t* d_indices, int64_t rows, int64_t cols, int parts) {
    LF_REQUIRE(d_indptr != nullptr, LF_ERR_INVALID, "indptr is null");
    LF_REQUIRE(rows >= 0 && cols >= 1, LF_ERR_INVALID, "bad shape %lld x %lld", (long long)rows, (long long)cols);
    LF_REQUIRE(rows < (1ll << 31) && cols < (1ll << 31), LF_ERR_UNSUPPORTED, "shape exceeds int32 indices");
    LF_REQUIRE(parts >= 1 && parts <= 65535, LF_ERR_INVALID, "num_parts must be in 1..65535 (got %d)", parts);
    (void)d_indices;
    return LF_OK;
}

int check_widths(int parts, const int32_t* flat, const int32_t* off) {
    LF_REQUIRE(flat && off, LF_ERR_INVALID, "width table is null");
    LF_REQUIRE(off[0] == 0, LF_ERR_INVALID, "widths_off[0] must be 0");
    for (int p = 0; p < parts; ++p) {
        const int n = off[p + 1] - off[p];
        LF_REQUIRE(n >= 0 && n <= LF_MAX_CLASSES, LF_ERR_INVALID,
                   "partition %d has %d widths (max %d)", p, n, LF_MAX_CLASSES);
        for (int b = 0; b < n; ++b) {
            const int w = flat[off[p] + b];
            LF_REQUIRE(lf::is_pow2(w) && w <= (1 << (LF_MAX_CLASSES - 1)), LF_ERR_INVALID,
                       "invalid padding for col_indices[%d][%d] and bucket_width=%d", p, b, w);
            LF_REQUIRE(b == 0 || flat[off[p] + b - 1] < w, LF_ERR_INVALID,
                       "widths of partition %d are not strictly ascending", p);
        }
    }
    return LF_OK;
}

}  // namespace

// ============================================================================ C ABI
extern "C" {

size_t lf_stats_workspace_bytes(int64_t num_rows, int64_t num_cols, int32_t num_parts) {
    if (num_rows < 0 || num_cols < 0 || num_parts < 1) return 0;
    return stats_layout(num_rows, num_cols, num_parts).total;
}

const int32_t* lf_stats_seg_bounds(const void* d_stats_workspace, int64_t num_rows, int32_t num_parts) {
    if (d_stats_workspace == nullptr || num_parts <= 1 || num_rows <= 0) return nullptr;
    return (const int32_t*)((const char*)d_stats_workspace + stats_layout(num_rows, 1, num_parts).bnd);
}

int lf_coo_degrees(const int32_t* d_coo_row, const int32_t* d_coo_col, int64_t nnz, int64_t num_rows,
                   int64_t num_cols, int32_t num_parts, int32_t* d_seg_deg, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(d_seg_deg, LF_ERR_INVALID, "seg_deg is null");
    LF_REQUIRE(nnz == 0 || (d_coo_row && d_coo_col), LF_ERR_INVALID, "COO arrays are null");
    LF_REQUIRE(num_parts >= 1 && num_cols >= 1, LF_ERR_INVALID, "bad num_parts / num_cols");
    const int64_t psize = lf::ceil_div(num_cols, num_parts);
    LF_HIP(fill_u32(d_seg_deg, (int64_t)num_parts * num_rows, 0u, s));
    if (nnz > 0) {
        const int grid = (int)std::min<int64_t>((nnz + 255) / 256, 65535);
        coo_degree_kernel<<<grid, 256, 0, s>>>(d_coo_row, d_coo_col, nnz, num_rows, psize, d_seg_deg);
        LF_HIP(hipGetLastError());
    }
    return LF_OK;
}

int lf_bucket_stats(const int32_t* d_indptr, const int32_t* d_indices, const int32_t* d_seg_deg,
                    int64_t num_rows, int64_t num_cols, int32_t num_parts, int32_t width_limit,
                    void* d_workspace, size_t workspace_bytes, int64_t* h_stats, int64_t* h_colhist,
                    lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    if (int rc = check_common(d_indptr, d_indices, num_rows, num_cols, num_parts)) return rc;
    LF_REQUIRE(h_stats, LF_ERR_INVALID, "h_stats is null");
    LF_REQUIRE(lf::is_pow2(width_limit) && width_limit <= (1 << (LF_MAX_CLASSES - 1)), LF_ERR_INVALID,
               "width_limit must be a power of two <= %d", 1 << (LF_MAX_CLASSES - 1));
    const StatsLayout L = stats_layout(num_rows, num_cols, num_parts);
    LF_REQUIRE(d_workspace && workspace_bytes >= L.total, LF_ERR_WORKSPACE,
               "workspace has %zu bytes, %zu needed", workspace_bytes, L.total);
    char* ws = (char*)d_workspace;
    int32_t* bnd = (int32_t*)(ws + L.bnd);
    uint8_t* planes = (uint8_t*)(ws + L.planes);
    unsigned long long* stats = (unsigned long long*)(ws + L.stats);
    unsigned long long* hist = (unsigned long long*)(ws + L.hist);
    const int64_t psize = lf::ceil_div(num_cols, num_parts);
    const size_t hist_bytes = (size_t)num_parts * (1 << LF_MAX_CLASSES) * 8;

    const MarkShape mark = mark_shape(num_rows, num_cols, num_parts);
    const bool use_planes = h_colhist && mark.slices == 0;
    if (use_planes)
        LF_HIP(fill_u32(planes, (L.total - L.planes) / 4, 0u, s));   // planes, stats and hist
    else
        LF_HIP(fill_u32(stats, (L.total - L.stats) / 4, 0u, s));
    if (num_rows > 0) {
        const int nblk = (int)((num_rows + kBlock - 1) / kBlock);
        if (num_parts > 1) {
            seg_bounds_kernel<<<nblk, kBlock, 0, s>>>(d_indptr, d_indices, num_rows, num_parts, psize, bnd);
            LF_HIP(hipGetLastError());
        }
        SegView v{d_indptr, bnd, num_rows, num_parts};
        const int num_classes = lf::ilog2(width_limit) + 1;
        const dim3 count_grid((unsigned)std::min<int64_t>(lf::ceil_div(num_rows, kCountThreads), kCountGrid), (unsigned)num_parts);
        int32_t* counts = h_colhist && !use_planes ? (int32_t*)(ws + L.counts) : nullptr;
        class_count_kernel<<<count_grid, kCountThreads, 0, s>>>(v, d_seg_deg, num_classes - 1, stats, counts);
        LF_HIP(hipGetLastError());
        if (counts) {
            int2* lists = (int2*)(ws + L.lists);
            uint32_t* bitmaps = (uint32_t*)(ws + L.bitmaps);
            int32_t* table = (int32_t*)(ws + L.table);
            class_list_kernel<<<count_grid, kCountThreads, 0, s>>>(v, d_seg_deg, num_classes - 1, counts, lists);
            LF_HIP(hipGetLastError());
            LF_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(mark_columns_kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kMarkMaxWords * 4));
            mark_columns_kernel<<<mark.groups, kMarkThreads, (size_t)mark.words * 4, s>>>(
                d_indices, lists, num_rows, num_parts, num_classes, mark, psize, num_cols, stats, table, bitmaps);
            LF_HIP(hipGetLastError());
            colbits_hist_kernel<<<dim3(std::min((mark.words + 63) / 64, kHistGrid), num_parts * mark.slices), kHistThreads, 0, s>>>(
                bitmaps, table, num_classes, mark, psize, num_cols, hist);
            LF_HIP(hipGetLastError());
        }
        if (use_planes) {
            mark_planes_kernel<<<dim3(std::min(nblk, kStatsGrid), num_parts, num_classes), kBlock, 0, s>>>(
                v, d_indices, d_seg_deg, num_classes - 1, planes, num_cols);
            LF_HIP(hipGetLastError());
            const int hgrid = (int)std::min<int64_t>((psize + kBlock - 1) / kBlock, 1024);
            colmask_hist_kernel<<<dim3(hgrid, num_parts), kBlock, 0, s>>>(planes, num_classes, num_cols, psize, hist);
            LF_HIP(hipGetLastError());
        }
    }
    const size_t lines_bytes = L.hist - L.stats;
    lf::PinnedLoan back(lines_bytes + (h_colhist ? hist_bytes : 0));
    LF_REQUIRE(back.ok(), LF_ERR_HIP, "out of host memory");
    const unsigned long long* h_lines = back.as<unsigned long long>();
    LF_HIP(hipMemcpyAsync(back.as<char>(), stats, lines_bytes + (h_colhist ? hist_bytes : 0), hipMemcpyDeviceToHost, s));      // (hist is behind stats)
    LF_HIP(hipStreamSynchronize(s));
    for (int p = 0; p < num_parts; ++p)
        for (int k = 0; k < LF_MAX_CLASSES; ++k)
            for (int f = 0; f < LF_STATS_FIELDS; ++f)
                h_stats[((size_t)p * LF_MAX_CLASSES + k) * LF_STATS_FIELDS + f] = f < 3 ? (int64_t)h_lines[stat_at(p, k, f)] : 0;
    if (h_colhist) std::memcpy(h_colhist, back.as<char>(lines_bytes), hist_bytes);
    return LF_OK;
}

int lf_row_features(const int32_t* d_indptr, int64_t num_rows, void* d_scratch, int64_t* h_out,
                    lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(h_out, LF_ERR_INVALID, "h_out is null");
    LF_REQUIRE(num_rows >= 0 && num_rows < (1ll << 31), LF_ERR_INVALID, "bad num_rows");
    h_out[0] = h_out[1] = h_out[2] = h_out[3] = 0;
    if (num_rows == 0) return LF_OK;
    LF_REQUIRE(d_indptr && d_scratch, LF_ERR_INVALID, "null argument");
    LF_REQUIRE((uintptr_t)d_scratch % 8 == 0, LF_ERR_INVALID, "scratch must be 8-byte aligned");
    unsigned long long* acc = (unsigned long long*)d_scratch;
    LF_HIP(fill_u32(acc, 2, 0xFFFFFFFFu, s));
    LF_HIP(fill_u32(acc + 1, 6, 0u, s));
    const int grid = (int)std::min<int64_t>((num_rows + kBlock - 1) / kBlock, 1024);
    row_features_kernel<<<grid, kBlock, 0, s>>>(d_indptr, num_rows, acc);
    LF_HIP(hipGetLastError());
    LF_HIP(lf::read_back(h_out, acc, 32, s));
    return LF_OK;
}

int lf_row_overlap(const int32_t* d_indptr, const int32_t* d_indices, int64_t num_rows, int64_t sample_stride,
                   void* d_scratch, int64_t* h_out, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(h_out, LF_ERR_INVALID, "h_out is null");
    LF_REQUIRE(num_rows >= 0 && num_rows < (1ll << 31) && sample_stride >= 1, LF_ERR_INVALID, "bad num_rows / stride");
    h_out[0] = h_out[1] = 0;
    if (num_rows < 2) return LF_OK;
    LF_REQUIRE(d_indptr && d_indices && d_scratch, LF_ERR_INVALID, "null argument");
    LF_REQUIRE((uintptr_t)d_scratch % 8 == 0, LF_ERR_INVALID, "scratch must be 8-byte aligned");
    unsigned long long* acc = (unsigned long long*)d_scratch;
    LF_HIP(fill_u32(acc, 4, 0u, s));
    LF_HIP(launch_row_overlap(d_indptr, d_indices, num_rows, sample_stride, acc, s));
    LF_HIP(lf::read_back(h_out, acc, 16, s));
    return LF_OK;
}

size_t lf_shape_stats_workspace_bytes(int32_t total_parts) {
    if (total_parts < 1 || total_parts > kShapeParts) return 0;
    const size_t out = ((size_t)total_parts * LF_MAX_CLASSES * LF_STATS_FIELDS + 2) * 8;
    return align_up(out, 256) + (size_t)kShapeGrid * shape_words(total_parts) * 8;
}

int lf_shape_stats(const int32_t* d_indptr, const int32_t* d_indices, int64_t num_rows, int64_t num_cols,
                   const int32_t* h_parts, int32_t n_candidates, int32_t width_limit, int64_t sample_stride,
                   void* d_workspace, size_t workspace_bytes, int64_t* h_stats, int64_t* h_overlap, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(h_parts && h_stats && h_overlap, LF_ERR_INVALID, "null argument");
    LF_REQUIRE(n_candidates >= 1 && n_candidates <= kShapeCands, LF_ERR_UNSUPPORTED, "1..%d candidates (got %d)", kShapeCands, n_candidates);
    LF_REQUIRE(sample_stride >= 1, LF_ERR_INVALID, "bad sample stride");
    LF_REQUIRE(lf::is_pow2(width_limit) && width_limit <= (1 << (LF_MAX_CLASSES - 1)), LF_ERR_INVALID,
               "width_limit must be a power of two <= %d", 1 << (LF_MAX_CLASSES - 1));
    ShapeCands cands{};
    cands.n = n_candidates;
    for (int c = 0; c < n_candidates; ++c) {
        if (int rc = check_common(d_indptr, d_indices, num_rows, num_cols, h_parts[c])) return rc;
        LF_REQUIRE(cands.total + h_parts[c] <= kShapeParts, LF_ERR_UNSUPPORTED, "at most %d partitions of all candidates together", kShapeParts);
        cands.parts[c] = h_parts[c];
        cands.total += h_parts[c];
    }
    LF_REQUIRE(d_workspace && workspace_bytes >= lf_shape_stats_workspace_bytes(cands.total), LF_ERR_WORKSPACE,
               "workspace has %zu bytes, %zu needed", workspace_bytes, lf_shape_stats_workspace_bytes(cands.total));
    const size_t n_stats = (size_t)cands.total * LF_MAX_CLASSES * LF_STATS_FIELDS;
    std::memset(h_stats, 0, n_stats * 8);
    h_overlap[0] = h_overlap[1] = 0;
    if (num_rows == 0) return LF_OK;
    LF_REQUIRE(d_indices, LF_ERR_INVALID, "indices is null");
    unsigned long long* out = (unsigned long long*)d_workspace;       // statistics, then the two overlap sums
    unsigned long long* partial = (unsigned long long*)((char*)d_workspace + align_up((n_stats + 2) * 8, 256));
    const int grid = (int)std::min<int64_t>((num_rows + kBlock - 1) / kBlock, kShapeGrid);
    const int kmax = lf::ilog2(width_limit);
    shape_stats_kernel<<<grid, kBlock, 0, s>>>(d_indptr, d_indices, num_rows, num_cols, cands, kmax, partial, out, (int)n_stats + 2);
    LF_HIP(hipGetLastError());
    shape_reduce_kernel<<<(shape_words(cands.total) + 63) / 64 + (num_rows > 1 ? overlap_groups(num_rows, sample_stride) : 0), 1024, 0, s>>>(
        partial, grid, cands.total, kmax, out, d_indptr, d_indices, num_rows, sample_stride);
    LF_HIP(hipGetLastError());
    lf::PinnedLoan back((n_stats + 2) * 8);
    LF_REQUIRE(back.ok(), LF_ERR_HIP, "out of host memory");
    LF_HIP(hipMemcpyAsync(back.as<char>(), out, (n_stats + 2) * 8, hipMemcpyDeviceToHost, s));
    LF_HIP(hipStreamSynchronize(s));
    std::memcpy(h_stats, back.as<char>(), n_stats * 8);
    std::memcpy(h_overlap, back.as<char>(n_stats * 8), 16);
    return LF_OK;
}

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_lock;
unsigned long long* g_scratch_ptr[kMaxDevices];     // device address of lf_static_scratch, per device

// Address of the current device's copy of lf_static_scratch, looked up once per device.
int static_scratch(unsigned long long** out) {
    int dev = -1;
    LF_HIP(hipGetDevice(&dev));
    LF_REQUIRE(dev >= 0 && dev < kMaxDevices, LF_ERR_UNSUPPORTED, "device index %d is out of range", dev);
    std::lock_guard<std::mutex> hold(g_scratch_lock);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        LF_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(lf_static_scratch)));
        LF_REQUIRE(p != nullptr, LF_ERR_HIP, "hipGetSymbolAddress returned a null address");
        g_scratch_ptr[dev] = (unsigned long long*)p;
    }
    *out = g_scratch_ptr[dev];
    return LF_OK;
}

__global__ void copy_features_kernel(const unsigned long long* __restrict__ acc, int64_t* __restrict__ out) {
    if (threadIdx.x < 4) out[threadIdx.x] = (int64_t)acc[threadIdx.x];
}

}  // namespace

int lf_row_features_static(const int32_t* d_indptr, int64_t num_rows, int64_t* d_out, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(d_out, LF_ERR_INVALID, "d_out is null");
    LF_REQUIRE(num_rows >= 0, LF_ERR_INVALID, "bad num_rows");
    LF_REQUIRE(num_rows <= LF_ROW_FEATURES_STATIC_MAX_ROWS, LF_ERR_UNSUPPORTED,
               "lf_row_features_static handles at most %lld rows (got %lld)",
               (long long)LF_ROW_FEATURES_STATIC_MAX_ROWS, (long long)num_rows);
    LF_REQUIRE(num_rows == 0 || d_indptr, LF_ERR_INVALID, "indptr is null");
    LF_REQUIRE((uintptr_t)d_out % 8 == 0, LF_ERR_INVALID, "d_out must be 8-byte aligned");
    unsigned long long* acc = nullptr;
    if (int rc = static_scratch(&acc)) return rc;
    // the array keeps the last call's values: min starts at all ones, the rest at zero
    // (num_rows == 0: the minimum is cleared too, which gives {0, 0, 0, 0})
    LF_HIP(fill_u32(acc, 2, num_rows > 0 ? 0xFFFFFFFFu : 0u, s));
    LF_HIP(fill_u32(acc + 1, 6, 0u, s));
    if (num_rows > 0) {
        const int grid = (int)std::min<int64_t>((num_rows + kBlock - 1) / kBlock, 1024);
        row_features_kernel<<<grid, kBlock, 0, s>>>(d_indptr, num_rows, acc);
        LF_HIP(hipGetLastError());
    }
    copy_features_kernel<<<1, 64, 0, s>>>(acc, d_out);
    LF_HIP(hipGetLastError());
    return LF_OK;
}

size_t lf_hyb_workspace_bytes(int64_t num_rows, int32_t num_parts, int32_t total_buckets) {
    if (num_rows < 0 || num_parts < 1 || total_buckets < 0) return 0;
    return hyb_layout(num_rows, num_parts, total_buckets).total;
}

int lf_hyb_layout(const int64_t* h_ell_rows, const int32_t* h_widths_flat, int32_t total_buckets,
                  int64_t* h_row_off, int64_t* h_slot_off, int64_t* h_total_rows, int64_t* h_total_slots) {
    LF_REQUIRE(total_buckets >= 0, LF_ERR_INVALID, "negative bucket count");
    LF_REQUIRE(h_total_rows && h_total_slots, LF_ERR_INVALID, "null output");
    LF_REQUIRE(total_buckets == 0 || (h_ell_rows && h_widths_flat && h_row_off && h_slot_off), LF_ERR_INVALID,
               "null argument");
    flat_layout(h_ell_rows, h_widths_flat, total_buckets, h_row_off, h_slot_off, h_total_rows, h_total_slots);
    return LF_OK;
}

int lf_hyb_plan(const int32_t* d_indptr, const int32_t* d_indices, const int32_t* d_seg_deg,
                const int32_t* d_seg_bounds, int64_t num_rows, int64_t num_cols, int32_t num_parts, const int32_t* h_widths_flat,
                const int32_t* h_widths_off, void* d_workspace, size_t workspace_bytes,
                int64_t* h_ell_rows, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    if (int rc = check_common(d_indptr, d_indices, num_rows, num_cols, num_parts)) return rc;
    if (int rc = check_widths(num_parts, h_widths_flat, h_widths_off)) return rc;
    const int nb = h_widths_off[num_parts];
    LF_REQUIRE(h_ell_rows || nb == 0, LF_ERR_INVALID, "h_ell_rows is null");
    const HybLayout L = hyb_layout(num_rows, num_parts, nb);
    LF_REQUIRE(d_workspace && workspace_bytes >= L.total, LF_ERR_WORKSPACE,
               "workspace has %zu bytes, %zu needed", workspace_bytes, L.total);
    char* ws = (char*)d_workspace;
    int32_t* bnd = (int32_t*)(ws + L.bnd);
    int32_t* wtab = (int32_t*)(ws + L.wtab);
    int32_t* flags = (int32_t*)(ws + L.flags);
    long long* totals = (long long*)(ws + L.totals);
    int32_t* blockcnt = (int32_t*)(ws + L.blockcnt);
    const int64_t psize = lf::ceil_div(num_cols, num_parts);

    const size_t up_bytes = L.flags - L.wtab, back_bytes = L.totals - L.flags + (size_t)nb * 8;
    lf::PinnedLoan up(up_bytes), back(back_bytes);
    LF_REQUIRE(up.ok() && back.ok(), LF_ERR_HIP, "out of host memory");
    int32_t* h_wtab = up.as<int32_t>();
    std::memset(h_wtab, 0, up_bytes);
    for (int p = 0; p < num_parts; ++p) {
        const int n = h_widths_off[p + 1] - h_widths_off[p];
        h_wtab[(size_t)p * kWtabStride] = n;
        for (int b = 0; b < n; ++b) h_wtab[(size_t)p * kWtabStride + 1 + b] = h_widths_flat[h_widths_off[p] + b];
        h_wtab[(size_t)p * kWtabStride + 12] = h_widths_off[p];
    }
    if (nb > 0) std::memcpy(up.as<char>(L.widths - L.wtab), h_widths_flat, (size_t)nb * 4);
    // The loans go back when this returns: every way out from here on waits for the stream first.
    struct Wait { hipStream_t s; ~Wait() { (void)hipStreamSynchronize(s); } } wait{s};
    LF_HIP(lf::move_words({h_wtab, wtab, up_bytes}, up.pinned(), flags, back_bytes, {}, true, s));
    const bool direct = back.pinned() && num_rows > 0 && nb > 0;
    if (num_rows > 0) {
        if (num_parts > 1 && d_seg_bounds) {       // bounds already known (the statistics pass made them)
            LF_HIP(hipMemcpyAsync(bnd, d_seg_bounds, (size_t)(num_parts + 1) * num_rows * 4,
                                  hipMemcpyDeviceToDevice, s));
        } else if (num_parts > 1) {
            seg_bounds_kernel<<<L.nblk, kBlock, 0, s>>>(d_indptr, d_indices, num_rows, num_parts, psize, bnd);
            LF_HIP(hipGetLastError());
        }
        SegView v{d_indptr, bnd, num_rows, num_parts};
        hyb_count_kernel<<<dim3(L.nblk, num_parts), kBlock, 0, s>>>(v, d_seg_deg, wtab, L.nblk, blockcnt, flags);
        LF_HIP(hipGetLastError());
        if (nb > 0) {
            hyb_scan_kernel<<<nb, 1024, 0, s>>>(blockcnt, L.nblk, totals, (const int32_t*)(ws + L.widths), flags + 1,
                                                (BucketOffsets*)(ws + L.scatter), flags, direct ? back.as<int>() : nullptr,
                                                direct ? back.as<long long>(L.totals - L.flags) : nullptr);
            LF_HIP(hipGetLastError());
        }
    }
    if (!direct) LF_HIP(hipMemcpyAsync(back.as<char>(), flags, back_bytes, hipMemcpyDeviceToHost, s));
    LF_HIP(hipStreamSynchronize(s));
    const int32_t h_flags = *back.as<int32_t>();
    if (h_flags & 1)
        return lf::fail(LF_ERR_CONFIG, "list index out of range: a partition with nonzeros has no bucket widths");
    if (h_flags & 2)
        return lf::fail(LF_ERR_UNSUPPORTED, "a row is split over more than %d ELL rows", kMetaSegMax);
    for (int k = 0; k < nb; ++k) h_ell_rows[k] = num_rows > 0 ? back.as<long long>(L.totals - L.flags)[k] : 0;
    return LF_OK;
}

int lf_hyb_build(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values,
                 const int32_t* d_seg_deg, int64_t num_rows, int64_t num_cols, int32_t num_parts,
                 const int32_t* h_widths_flat, const int32_t* h_widths_off, const int64_t* h_ell_rows,
                 void* d_workspace, size_t workspace_bytes, int32_t* d_rows, int32_t* d_meta,
                 int32_t* d_cols, float* d_vals, float* d_mask, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    if (int rc = check_common(d_indptr, d_indices, num_rows, num_cols, num_parts)) return rc;
    if (int rc = check_widths(num_parts, h_widths_flat, h_widths_off)) return rc;
    const int nb = h_widths_off[num_parts];
    if (nb == 0 || num_rows == 0) return LF_OK;
    LF_REQUIRE(h_ell_rows, LF_ERR_INVALID, "h_ell_rows is null");
    int64_t total_rows = 0;
    for (int k = 0; k < nb; ++k) {
        LF_REQUIRE(h_ell_rows[k] >= 0, LF_ERR_INVALID, "negative ELL row count");
        total_rows += h_ell_rows[k];
    }
    if (total_rows == 0) return LF_OK;
    LF_REQUIRE(d_rows && d_meta && d_cols && d_vals && d_indices, LF_ERR_INVALID, "slab pointers are null");
    const HybLayout L = hyb_layout(num_rows, num_parts, nb);
    LF_REQUIRE(d_workspace && workspace_bytes >= L.total, LF_ERR_WORKSPACE,
               "workspace has %zu bytes, %zu needed", workspace_bytes, L.total);
    char* ws = (char*)d_workspace;
    int32_t* bnd = (int32_t*)(ws + L.bnd);
    int32_t* wtab = (int32_t*)(ws + L.wtab);
    BucketOffsets* offs = (BucketOffsets*)(ws + L.scatter);
    int32_t* blockoff = (int32_t*)(ws + L.blockcnt);

    // (the bucket offsets are in the workspace: hyb_scan_kernel left them there)
    SegView v{d_indptr, bnd, num_rows, num_parts};
    hyb_fill_kernel<<<L.nblk, kBlock, 0, s>>>(v, d_seg_deg, wtab, L.nblk, blockoff, offs, d_indices, d_values,
                                              d_rows, d_meta, d_cols, d_vals, d_mask);
    LF_HIP(hipGetLastError());
    return LF_OK;
}

}  // extern "C"
