// Fused hyb SpMM for gfx950 (MI355X):  C[rows][N] = A_hyb . B[cols][N], fp32 accumulate.
//
// Takes over the kernel that the reference generates through SparseTIR/TVM in
// bench_hyb_with_config (playground_pipline/format_algos.py:388-605): all (partition,
// bucket) ELL blocks of the hyb format are walked by one launch per column partition.
// The reference binds 32 threads to 32 features and 8 ELL rows to a thread block and uses
// atomicAdd where several ELL rows feed one output row (format_algos.py:508-533).  Here:
//
//   * a "sub-wave" of LPR lanes owns one ELL row at a time; each lane holds VEC consecutive
//     features (float4, or 8 x bf16 = 16 bytes), so one B row is read with one 16-byte load
//     per lane, coalesced along the feature dimension (N = 128 fp32 -> 32 lanes, two rows
//     per 64-lane wavefront);
//   * narrow buckets stage their (row of B, value) tile in LDS with coalesced 16-byte loads
//     and read it back as broadcasts; rows too wide to stage are streamed by one or several sub-waves each, their slots
//     broadcast by DPP;
//   * a source row split over several ELL rows is summed by one owner; rows longer than
//     coop_slots (64, 128 or 256) are reduced by a whole workgroup in chunks of 512 to 8192 slots: a row
//     that fits one chunk is written directly, a longer one leaves one partial row per chunk, which the
//     workgroup that comes last adds up (rows of very many chunks: a small second kernel);
//   * partitions run as consecutive launches: partition 0 stores every output row (rows it
//     does not touch are cleared by the same launch), later partitions add.  No sum is made with
//     atomics and the order of every sum is fixed, so results are bit-reproducible; the one atomic of a
//     product counts the chunks of a long row that have left their partial row.
//
// The workgroup -> tile mapping is XCD-aware: workgroup i runs on XCD i % 8, an XCD computes an eighth of the features'
// slices, and within a slice a contiguous range of each group of tiles, so that neighbouring ELL rows (which tend to
// share B rows in structured matrices) meet in the same L2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "lf_cells.h"
#include "lf_internal.h"
#include "lf_spmm_device.h"

namespace {

// ------------------------------------------------------------------------------------
// Tile bodies.  s_pairs / s_rm point into the workgroup's LDS: tile_slots(LPR) (key of B's row, val)
// pairs followed by kTileRows (row, meta) entries.

// Narrow bucket: W slots per ELL row, rows independent (one ELL row per source row).
// RPI rows are processed together by a sub-wave so that kUnroll gathers are in flight
// even when W < kUnroll.
template <int W, int LPR, int CH, typename BT, bool WIDE>
__device__ __forceinline__ void ell_tile_narrow(const RowsOfB<LPR, CH, BT, WIDE>& b, const int2* s_pairs, const int2* s_rm, int n,
                                                const LaunchArgs& a, int sw, int sl) {
    constexpr int VEC = Dense<BT>::kVec;
    constexpr int SW = kWG / LPR;
    constexpr int RPI = kUnroll / W;
    const Lane<LPR, CH, VEC> ln(sl, a.feat, a.ldb, a.ldc);
    for (int r0 = sw * RPI; r0 < n; r0 += SW * RPI) {
        uint32_t k[kUnroll];
        float v[kUnroll];
#pragma unroll
        for (int q = 0; q < RPI; ++q) {
            const int r = min(r0 + q, n - 1);
            const int len = r0 + q < n ? s_rm[r].y & kMetaLenMask : 0;
#pragma unroll
            for (int j = 0; j < W; ++j) {
                const int2 kv = s_pairs[r * W + j];
                k[q * W + j] = j < len ? (uint32_t)kv.x : b.kNone;
                v[q * W + j] = __int_as_float(kv.y);
            }
        }
        typename Dense<BT>::Raw x[kUnroll][CH];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
#pragma unroll
            for (int cc = 0; cc < CH; ++cc) x[u][cc] = b.load(cc, k[u]);
#pragma unroll
        for (int q = 0; q < RPI; ++q) {
            Acc<CH, VEC> acc;
            acc.clear();
#pragma unroll
            for (int j = 0; j < W; ++j)
#pragma unroll
                for (int cc = 0; cc < CH; ++cc) fma_dense<BT>(v[q * W + j], x[q * W + j][cc], acc.v[cc]);
            if (r0 + q < n) store_row<LPR, CH, VEC>(a.C, s_rm[r0 + q].x, ln, acc, a.accumulate);
        }
    }
}

// U staged slots of an ELL row from position j; slots at or past `len` are padding (their value is 0).
template <int U, int LPR, int CH, typename BT, bool WIDE>
__device__ __forceinline__ void staged_group(const RowsOfB<LPR, CH, BT, WIDE>& b, const int2* rp, int j, int len,
                                             Acc<CH, Dense<BT>::kVec>& acc) {
    uint32_t k[U];
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int2 kv = rp[j + u];
        k[u] = j + u < len ? (uint32_t)kv.x : b.kNone;
        v[u] = __int_as_float(kv.y);
    }
    gather_fma<U>(b, k, v, acc);
}

// Bucket with W >= kUnroll (a multiple of it) staged in LDS: one ELL row per sub-wave at a time.
template <int LPR, int CH, typename BT, bool WIDE>
__device__ __forceinline__ void ell_tile_wide(const RowsOfB<LPR, CH, BT, WIDE>& b, const int2* s_pairs, const int2* s_rm, int n, int log_w,
                                              const LaunchArgs& a, int sw, int sl) {
    constexpr int VEC = Dense<BT>::kVec;
    constexpr int SW = kWG / LPR;
    const Lane<LPR, CH, VEC> ln(sl, a.feat, a.ldb, a.ldc);
#pragma unroll 1
    for (int r = sw; r < n; r += SW) {
        const int2 rm = s_rm[r];
        const int len = rm.y & kMetaLenMask;
        const int2* rp = s_pairs + (r << log_w);
        Acc<CH, VEC> acc;
        acc.clear();
        // Whole groups of kUnroll slots, then a tail of kUnroll or kUnroll / 2 gathers.  The
        // short tail saves padding gathers (a 27-slot stencil row: 28 instead of 32); with
        // many rows per wavefront (small N) the extra branch costs more than it saves.
        constexpr bool kShortTail = LPR >= 32;
        if constexpr (kShortTail) {
            int j = 0;
#pragma unroll 1
            for (; j + kUnroll <= len; j += kUnroll) staged_group<kUnroll>(b, rp, j, len, acc);
            if (len > j && len - j <= kUnroll / 2) staged_group<kUnroll / 2>(b, rp, j, len, acc);
            else if (len > j) staged_group<kUnroll>(b, rp, j, len, acc);
        } else {
#pragma unroll 1
            for (int j = 0; j < len; j += kUnroll) staged_group<kUnroll>(b, rp, j, len, acc);
        }
        store_row<LPR, CH, VEC>(a.C, rm.x, ln, acc, a.accumulate);
    }
}

// Staged tile of a bucket whose source rows may span several consecutive ELL rows (the widest
// bucket of a partition): the first ELL row of a segment owns it.  The part of the segment
// inside the tile is read from LDS, a part that runs past the tile's end is streamed from
// global memory.  Continuation rows and rows that take the cooperative path are skipped.
template <int LPR, int CH, typename BT, bool WIDE>
__device__ __forceinline__ void ell_tile_segments(const RowsOfB<LPR, CH, BT, WIDE>& b, const Group& g, long long e0, const int2* s_pairs,
                                                  const int2* s_rm, int n, const LaunchArgs& a, int* s_next,
                                                  int sl) {
    constexpr int VEC = Dense<BT>::kVec;
    const Lane<LPR, CH, VEC> ln(sl, a.feat, a.ldb, a.ldc);
    const int log_w = g.log_w;
    // Segments differ in length and continuation rows carry no work, so the sub-waves take
    // the tile's ELL rows from a shared counter as they become free instead of by a fixed
    // stride.  Which sub-wave sums a row does not change the order of its additions.
    for (;;) {
        int r = 0;
        if (sl == 0) r = atomicAdd(s_next, 1);
        r = __shfl(r, 0, LPR);
        if (r >= n) break;
        const int2 rm = s_rm[r];
        if (rm.y < 0) continue;                                  // continuation row
        const int seg = (int)((uint32_t)rm.y >> kMetaLenBits);
        if (((long long)seg << log_w) > a.coop_slots) continue; // reduced by a whole workgroup
        int total = rm.y & kMetaLenMask;
        if (seg > 1) {
            const int last = r + seg - 1;
            const int last_meta = last < n ? s_rm[last].y : g.meta[e0 + last];
            total = ((seg - 1) << log_w) + (last_meta & kMetaLenMask);
        }
        const int staged = min(total, (n - r) << log_w);
        const int2* rp = s_pairs + (r << log_w);
        Acc<CH, VEC> acc;
        acc.clear();
#pragma unroll 1
        for (int j = 0; j < staged; j += kUnroll) {
            uint32_t k[kUnroll];
            float v[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const bool in = j + u < staged;
                const int2 kv = rp[in ? j + u : 0];
                k[u] = in ? (uint32_t)kv.x : b.kNone;
                v[u] = in ? __int_as_float(kv.y) : 0.f;
            }
            gather_fma<kUnroll>(b, k, v, acc);
        }
        if (total > staged)
            Teams<LPR, CH, BT, WIDE>(b, 0).sum(g.cols, g.vals, ((e0 + r) << log_w) + staged, total - staged, total - staged, acc);
        store_row<LPR, CH, VEC>(a.C, rm.x, ln, acc, a.accumulate);
    }
}

// The same bucket with the work spread evenly: every ELL row of the tile is summed by the
// sub-wave it falls to, a row that is only part of a segment leaves its sum in LDS, and after
// a barrier the first ELL row of each segment adds the sums of its rows in order.  With the
// variant above a tile of a folded configuration offers fewer segments than sub-waves at
// small N (about 20 for 32 at N = 32), and the lanes in flight bound the gather rate.
// Rows that continue a segment begun in an earlier tile are summed by that tile, as above.
template <int LPR, int CH, typename BT, bool WIDE>
__device__ __forceinline__ void ell_tile_segments_balanced(const RowsOfB<LPR, CH, BT, WIDE>& b, const Group& g, long long e0, const int2* s_pairs,
                                                           const int2* s_rm, int n, const LaunchArgs& a,
                                                           float* s_part, int sw, int sl) {
    constexpr int VEC = Dense<BT>::kVec;
    constexpr int SW = kWG / LPR;
    const Lane<LPR, CH, VEC> ln(sl, a.feat, a.ldb, a.ldc);
    const int log_w = g.log_w;
    for (int r = sw; r < n; r += SW) {
        const int2 rm = s_rm[r];
        const bool cont = rm.y < 0;
        const int head = cont ? r - (int)(((uint32_t)rm.y & 0x7FFFFFFFu) >> kMetaLenBits) : r;
        if (head < 0) continue;                                  // belongs to the previous tile's last segment
        const int seg = (int)((uint32_t)s_rm[head].y >> kMetaLenBits);
        if (((long long)seg << log_w) > a.coop_slots) continue; // reduced by a whole workgroup
        const int len = rm.y & kMetaLenMask;
        const int2* rp = s_pairs + (r << log_w);
        Acc<CH, VEC> acc;
        acc.clear();
#pragma unroll 1
        for (int j = 0; j < len; j += kUnroll) {
            uint32_t k[kUnroll];
            float v[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const bool in = j + u < len;          // W may be below kUnroll: stay inside the row
                const int2 kv = rp[in ? j + u : 0];
                k[u] = in ? (uint32_t)kv.x : b.kNone;
                v[u] = in ? __int_as_float(kv.y) : 0.f;
            }
            gather_fma<kUnroll>(b, k, v, acc);
        }
        if (seg == 1) {
            store_row<LPR, CH, VEC>(a.C, rm.x, ln, acc, a.accumulate);
        } else {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                if (!ln.on[c]) continue;
                float* dst = s_part + r * a.feat + ln.f[c];
#pragma unroll
                for (int i = 0; i < VEC; i += 4)
                    *reinterpret_cast<float4*>(dst + i) =
                        make_float4(acc.v[c][i], acc.v[c][i + 1], acc.v[c][i + 2], acc.v[c][i + 3]);
            }
        }
    }
    __syncthreads();
    for (int r = sw; r < n; r += SW) {
        const int2 rm = s_rm[r];
        if (rm.y < 0) continue;
        const int seg = (int)((uint32_t)rm.y >> kMetaLenBits);
        if (seg == 1 || ((long long)seg << log_w) > a.coop_slots) continue;
        Acc<CH, VEC> acc;
        acc.clear();
        const int inside = min(seg, n - r);
        for (int k = 0; k < inside; ++k) {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                if (!ln.on[c]) continue;
                const float* src = s_part + (r + k) * a.feat + ln.f[c];
#pragma unroll
                for (int i = 0; i < VEC; i += 4) {
                    const float4 x = *reinterpret_cast<const float4*>(src + i);
                    acc.v[c][i] += x.x; acc.v[c][i + 1] += x.y; acc.v[c][i + 2] += x.z; acc.v[c][i + 3] += x.w;
                }
            }
        }
        if (inside < seg) {                                      // the segment runs past the tile: stream the rest
            const int total = ((seg - 1) << log_w) + (g.meta[e0 + r + seg - 1] & kMetaLenMask);
            const int staged = inside << log_w;
            Teams<LPR, CH, BT, WIDE>(b, 0).sum(g.cols, g.vals, ((e0 + r) << log_w) + staged, total - staged, total - staged, acc);
        }
        store_row<LPR, CH, VEC>(a.C, rm.x, ln, acc, a.accumulate);
    }
}

template <int LPR, int CH, typename BT, bool WIDE>
__device__ __forceinline__ void run_ell_tile(const RowsOfB<LPR, CH, BT, WIDE>& b, const Group& g, long long tile, int2* s_pairs, int2* s_rm,
                                             int* s_next, float* s_part, const LaunchArgs& a) {
    const int tid = threadIdx.x;
    const long long e0 = tile * g.rows_per_tile;
    const int n = (int)min((long long)g.rows_per_tile, g.n_items - e0);
    const int n_slots = n << g.log_w;
    const long long s0 = e0 << g.log_w;
    for (int i = tid * 4; i < n_slots; i += kWG * 4) {
        if (i + 4 <= n_slots) {            // s0 and i are multiples of 4, slabs are 16-byte aligned
            const lf_i32x4 c = load_i32x4(g.cols + s0 + i, a.accumulate & kStreamSlabs);
            const lf_i32x4 v = load_i32x4(g.vals + s0 + i, a.accumulate & kStreamSlabs);
            s_pairs[i + 0] = make_int2((int)b.key(c.x), v.x);
            s_pairs[i + 1] = make_int2((int)b.key(c.y), v.y);
            s_pairs[i + 2] = make_int2((int)b.key(c.z), v.z);
            s_pairs[i + 3] = make_int2((int)b.key(c.w), v.w);
        } else {
            for (int k = i; k < n_slots; ++k)
                s_pairs[k] = make_int2((int)b.key(g.cols[s0 + k]), __float_as_int(g.vals[s0 + k]));
        }
    }
    for (int i = tid; i < n; i += kWG) s_rm[i] = make_int2(g.rows[e0 + i], g.meta[e0 + i]);
    if (tid == 0) *s_next = 0;
    __syncthreads();
    const int sw = tid / LPR, sl = tid % LPR;
    if (g.type == kEllSeg) {
        if (g.balanced) ell_tile_segments_balanced(b, g, e0, s_pairs, s_rm, n, a, s_part, sw, sl);
        else ell_tile_segments(b, g, e0, s_pairs, s_rm, n, a, s_next, sl);
        return;
    }
    switch (g.log_w) {
        case 0: ell_tile_narrow<1>(b, s_pairs, s_rm, n, a, sw, sl); break;
        case 1: ell_tile_narrow<2>(b, s_pairs, s_rm, n, a, sw, sl); break;
        case 2: ell_tile_narrow<4>(b, s_pairs, s_rm, n, a, sw, sl); break;
        default: ell_tile_wide(b, s_pairs, s_rm, n, g.log_w, a, sw, sl); break;
    }
}

// Bucket whose source rows may span several ELL rows, or whose rows are too wide to stage: the first ELL row of a
// segment owns it, a team of sub-waves sums all of its slots, each its share; continuation rows and segments
// above coop_slots (handled as chunks) are skipped.
template <int LPR, int CH, typename BT, bool WIDE>
__device__ __forceinline__ void run_seg_tile(const RowsOfB<LPR, CH, BT, WIDE>& b, const Group& g, long long tile, const LaunchArgs& a) {
    constexpr int VEC = Dense<BT>::kVec;
    const int lane = threadIdx.x & 63;
    const Lane<LPR, CH, VEC> ln(lane % LPR, a.feat, a.ldb, a.ldc);
    const Teams<LPR, CH, BT, WIDE> team(b, min(g.balanced, Teams<LPR, CH, BT, WIDE>::kLgSubs));
    const int lanes = LPR << team.lg;
    const long long e0 = tile * g.rows_per_tile;
    const int n = (int)min((long long)g.rows_per_tile, g.n_items - e0);
    for (int r = (int)threadIdx.x / lanes; r < n; r += kWG / lanes) {
        const long long e = e0 + r;
        const int m = g.meta[e];
        if (m < 0) continue;                                   // continuation row
        const int seg = (int)((uint32_t)m >> kMetaLenBits);
        if (((long long)seg << g.log_w) > a.coop_slots) continue;
        int total = m & kMetaLenMask;
        if (seg > 1) total = ((seg - 1) << g.log_w) + (g.meta[e + seg - 1] & kMetaLenMask);
        Acc<CH, VEC> acc;
        acc.clear();
        team.sum(g.cols, g.vals, e << g.log_w, total, total, acc);
        team.combine(acc);
        if (team.sub == 0) store_row<LPR, CH, VEC>(a.C, g.rows[e], ln, acc, a.accumulate);
    }
}

template <int LPR, int CH, typename BT>
__device__ __forceinline__ void run_zero_tile(const Group& g, long long tile, const LaunchArgs& a) {
    constexpr int VEC = Dense<BT>::kVec;
    constexpr int SW = kWG / LPR;
    const int tid = threadIdx.x;
    const int sw = tid / LPR, sl = tid % LPR;
    const Lane<LPR, CH, VEC> ln(sl, a.feat, a.ldb, a.ldc);
    const long long e0 = tile * g.rows_per_tile;
    const int n = (int)min((long long)g.rows_per_tile, g.n_items - e0);
    Acc<CH, VEC> zero;
    zero.clear();
    for (int r = sw; r < n; r += SW) store_row<LPR, CH, VEC>(a.C, g.rows[e0 + r], ln, zero, a.accumulate & kStreamC);
}

// Two floats at agent scope: stored to, and read from, where all XCDs see them.
__device__ __forceinline__ void store_pair_agent(float* dst, float x, float y) {
    const unsigned long long v = (unsigned long long)__float_as_uint(x) | (unsigned long long)__float_as_uint(y) << 32;
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(dst), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void load_pair_agent(const float* src, float& x, float& y) {
    const unsigned long long v = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(src), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    x = __uint_as_float((unsigned int)v);
    y = __uint_as_float((unsigned int)(v >> 32));
}

// Streamed rows: as many sub-waves to a row as have 64 of its slots each, 8 rows to a tile, 4 where rows of B take 32 lanes and
// more.  A sub-wave to a row, with tiles of 16 and 32 rows, is a chain of up to 32 batches; all of a wavefront to a row leaves
// batches of its sub-waves half empty, and an eighth row waits for two before it where a wavefront is one sub-wave.  Log-normal rows,
// us, a sub-wave / a wavefront / this: 16000 x 128, N = 32 25.7 / 19.1 / 18.4, N = 64 35.6 / 28.2 / 28.1; 132K x 300 in eight
// partitions, N = 32 363 / 371 / 359, N = 64 605 / 617 / 610; 207K x 175, N = 32 323 / 339 / 329; 4.5K x 91, N = 416 34.4 /
// 37.2 / 29.6; 6.5K x 311, N = 416 149 / 153 / 138.  300 matrices of 3K to 250K rows of 50 to 400: 0.93 to 1.0 of
// the time with a wavefront to a row; 16 rows to a tile are 1 % better above 32K such rows and up to 25 % worse below 16K.
constexpr int kSegRows = 8, kLgTeamSlots = 6;
constexpr int kSlice = 8;
constexpr int kSlicedSlots = 128;

// One chunk of a heavy source row: the workgroup's wavefronts take consecutive parts of the chunk, a part's
// slots are spread over the wavefront's sub-waves, the sums are combined through LDS in wavefront order.
template <int LPR, int CH, typename BT, bool WIDE>
__device__ __forceinline__ void run_chunk_tile(const RowsOfB<LPR, CH, BT, WIDE>& b, const Group& g, long long tile, float* s_red,
                                               const LaunchArgs& a) {
    constexpr int VEC = Dense<BT>::kVec;
    constexpr int SW = kWG / LPR;
    const int tid = threadIdx.x;
    const int sw = tid / LPR, sl = tid % LPR;
    const Lane<LPR, CH, VEC> ln(sl, a.feat, a.ldb, a.ldc);
    const Chunk ck = g.chunks[tile];
    Acc<CH, VEC> acc;
    acc.clear();
    if (ck.partial < 0 && ck.n_slots <= kSlicedSlots) {
        // A short row in slices of kSlice slots, added in their order: the same sums whatever the lane
        // count, so that such rows do not depend on the feature windows of the plan.
        Acc<CH, VEC> sum;
        sum.clear();
        for (int s0 = 0; s0 * kSlice < ck.n_slots; s0 += SW) {
            const int at = (s0 + sw) * kSlice;
            acc.clear();
            Teams<LPR, CH, BT, WIDE>(b, 0).sum(g.cols, g.vals, ck.slot_begin + at, min(kSlice, ck.n_slots - at), kSlice, acc);
            if (s0 > 0) __syncthreads();             // the slices before have been read
#pragma unroll
            for (int c = 0; c < CH; ++c)
#pragma unroll
                for (int i = 0; i < VEC; ++i) s_red[((sw * CH + c) * LPR + sl) * VEC + i] = acc.v[c][i];
            __syncthreads();
            const int n = min(SW, (ck.n_slots + kSlice - 1) / kSlice - s0);
#pragma unroll
            for (int c = 0; c < CH; ++c)
                for (int s = 0; s < n && sw == 0; ++s)
#pragma unroll
                    for (int i = 0; i < VEC; ++i) sum.v[c][i] += s_red[((s * CH + c) * LPR + sl) * VEC + i];
        }
        if (sw == 0) store_row<LPR, CH, VEC>(a.C, ck.row, ln, sum, a.accumulate);
        return;
    }
    constexpr int kWaves = kWG / 64, kStep = Teams<LPR, CH, BT, WIDE>::kBatch << Teams<LPR, CH, BT, WIDE>::kLgSubs;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per = ((ck.n_slots + kWaves - 1) / kWaves + kStep - 1) / kStep * kStep;
    const int lo = min(wave * per, ck.n_slots), part = min(per, ck.n_slots - lo);
    const Teams<LPR, CH, BT, WIDE> team(b, Teams<LPR, CH, BT, WIDE>::kLgSubs);
    team.sum(g.cols, g.vals, ck.slot_begin + lo, part, part, acc);
    team.combine(acc);
    // s_red[wave][c][sl][i]
    if ((tid & 63) < LPR) {
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
            for (int i = 0; i < VEC; ++i) s_red[((wave * CH + c) * LPR + sl) * VEC + i] = acc.v[c][i];
    }
    __syncthreads();
    if (tid >= 64) return;
    acc.clear();
    if (sw == 0) {
#pragma unroll
        for (int c = 0; c < CH; ++c)
            for (int w = 0; w < kWaves; ++w)
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc.v[c][i] += s_red[((w * CH + c) * LPR + sl) * VEC + i];
    }
    if (ck.partial < 0) {                            // the row's only chunk
        if (sw == 0) store_row<LPR, CH, VEC>(a.C, ck.row, ln, acc, a.accumulate);
        return;
    }
    // The first wavefront leaves the chunk's partial row, counts it, and adds the row's partial rows
    // up if it was the last: sub-wave s takes partial rows s, s + n_sub, ..., the sub-waves' sums are
    // added in sub-wave order - the same order whoever comes last.  Partial rows are written and read at
    // agent scope, past the L2s that the XCDs do not share, and are complete (the wait) before they
    // are counted.  A release and acquire at the counter would do the same by writing back and invalidating the
    // whole L2 of the XCD, once per chunk: 500k x 2M matrix with 4911 partial rows 1.34 -> 1.72 ms.
    // (170K-row graph with 27 such rows: one launch less, 85.7 -> 81.9 us a product.)  Where a row has
    // many chunks they are short and the wait and the count would hold up their workgroups more than
    // a launch costs (that matrix: 1.37 ms): those rows are left to spmm_finalize_wide_kernel.
    if (sw == 0) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            if (!ln.on[c]) continue;
            float* dst = a.partials + (size_t)ck.partial * a.feat + ln.f[c];
#pragma unroll
            for (int i = 0; i < VEC; i += 2) store_pair_agent(dst + i, acc.v[c][i], acc.v[c][i + 1]);
        }
    }
    HeavyRow* hr = a.heavy + ck.heavy;
    const int n = hr->n_partials;
    if (n > kWideFinalPartials) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int before = 0;
    if (tid == 0) before = __hip_atomic_fetch_add(&hr->done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(before) != n - 1) return;
    if (tid == 0) hr->done = 0;                      // for the next launch
    constexpr int kSub = 64 / LPR;
    constexpr int U = VEC * CH <= 4 ? 8 : VEC * CH <= 8 ? 4 : 2;   // partial rows in flight per sub-wave
    acc.clear();
    for (int k0 = sw; k0 < n; k0 += kSub * U) {
        float x[U][CH][VEC];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(k0 + u * kSub, n - 1); // (clamped loads, masked below)
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const float* src = a.partials + (size_t)(hr->partial_begin + k) * a.feat + (ln.on[c] ? ln.f[c] : 0);
#pragma unroll
                for (int i = 0; i < VEC; i += 2) load_pair_agent(src + i, x[u][c][i], x[u][c][i + 1]);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = k0 + u * kSub < n;
#pragma unroll
            for (int c = 0; c < CH; ++c)
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc.v[c][i] += in ? x[u][c][i] : 0.f;
        }
    }
    Acc<CH, VEC> sum = acc;
    for (int s = 1; s < kSub; ++s)
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
            for (int i = 0; i < VEC; ++i) sum.v[c][i] += __shfl(acc.v[c][i], s * LPR + sl);
    if (sw == 0) store_row<LPR, CH, VEC>(a.C, ck.row, ln, sum, a.accumulate);
}

// ------------------------------------------------------------------------------------
// The fused kernel: one workgroup per tile, all tile groups of one column partition in one
// launch.  Workgroup i runs on XCD i % 8 and takes entry i / 8 of that XCD's tile list: for
// every group the contiguous range of its tiles that belongs to the XCD, groups
// concatenated, and where the XCD has a part of a second feature slice, the same for that.  The hardware hands out workgroups in index order as slots free up, which
// keeps the tiles in flight on an XCD next to each other and balances the load; a resident
// grid that strides over the tiles measured 2-7 % slower on every workload.
//
// RESIDENT: the partition's part of B stays in the XCD's L2.  Gathers that hit are short, so what counts is how many
// wavefronts are there to issue them: registers are held to 6 wavefronts per SIMD (two chunks per lane 4), and a tile
// of a float product holds twice the slots, since the wait for a tile's slots is a larger part of it.  132K-row graph,
// 300 entries a row, 16 partitions, N = 96, with the kernels of its time: 1186 -> 1046 us (occupancy alone 1100, tiles
// alone 1096); 1023 now.  (The loops over a row's slots are not unrolled beyond one batch of gathers: two batches in
// flight spilled here, 1497 us, and elsewhere cost a wavefront per SIMD.)  Where gathers miss, more of them in flight
// gain nothing and bf16 pays for the spills (500k x 2M matrix 1.32 -> 1.39 ms).
constexpr int partition_min_waves(int lpr, int ch, bool bf16, bool resident) {
    if (ch != 1) return resident ? 4 : 1;
    if (!bf16) return lpr == 8 || resident ? 6 : 1;
    return resident ? 6 : 1;
}
constexpr bool has_resident_kernel(int lpr, int ch, bool bf16) { return bf16 ? ch == 1 : ch <= 2 && lpr > 8; }

__device__ __forceinline__ Group load_group(const __attribute__((address_space(4))) Group* from) {
    Group g;
    g.type = from->type;
    g.log_w = from->log_w;
    g.rows_per_tile = from->rows_per_tile;
    g.balanced = from->balanced;
    g.n_items = from->n_items;
    g.n_tiles = from->n_tiles;
    g.rows = from->rows;
    g.meta = from->meta;
    g.cols = from->cols;
    g.vals = from->vals;
    g.chunks = from->chunks;
    return g;
}

template <int LPR, int CH, typename BT, bool RESIDENT, bool WIDE>
__global__ void __launch_bounds__(kWG, partition_min_waves(LPR, CH, Dense<BT>::kVec == 8, RESIDENT))
spmm_partition_kernel(LaunchArgs a, XcdParts parts) {
    // one LDS buffer, used either as the staged tile ((col, val) pairs then (row, meta)
    // entries) or as the reduction scratch of a chunk tile (one accumulator per thread)
    constexpr int kTileSlots = tile_slots(LPR, RESIDENT && Dense<BT>::kVec == 4);
    constexpr int kStageBytes = (kTileSlots + kTileRows) * (int)sizeof(int2);
    constexpr int kReduceBytes = kWG * CH * Dense<BT>::kVec * (int)sizeof(float);
    __shared__ __align__(16) char s_raw[kStageBytes > kReduceBytes ? kStageBytes : kReduceBytes];
    int2* s_pairs = reinterpret_cast<int2*>(s_raw);
    int2* s_rm = s_pairs + kTileSlots;
    __shared__ int s_next;                     // next ELL row of a tile whose rows are taken dynamically
    extern __shared__ __align__(16) float s_dyn[];   // per-ELL-row sums of a balanced segment tile

    // Position in this XCD's tile list -> group and tile.  The groups' tile counts come with the
    // arguments: reading the groups one after the other took a round trip to memory each.  The group itself is read
    // whole, by scalar loads (through the constant address space: nothing writes it while the launch runs): field by
    // field, where it is used, each read was a round trip of its own.
    XcdPart part = xcd_part(parts, blockIdx.x % kXcds);
    using ConstGroup = const __attribute__((address_space(4))) Group;
    ConstGroup* groups = (ConstGroup*)(uintptr_t)a.groups;
    int v = blockIdx.x / kXcds;
    // a group to a lane, the shares' prefix sums by DPP, the group from one ballot: group by group the walk to the
    // last of eleven was 300 scalar instructions
    int n_tiles = 0, gi;
#pragma unroll
    for (int i = 0; i < kInlineGroups; ++i) n_tiles = (int)(threadIdx.x & 63) == i ? a.n_tiles[i] : n_tiles;
    for (;;) {
        const int first = tiles_before(n_tiles, part.from), count = tiles_before(n_tiles, part.upto) - first;
        int until = count;
        until += __builtin_amdgcn_update_dpp(0, until, 0x111, 0xF, 0xF, true);       // row_shr:1, 2, 4, 8
        until += __builtin_amdgcn_update_dpp(0, until, 0x112, 0xF, 0xF, true);
        until += __builtin_amdgcn_update_dpp(0, until, 0x114, 0xF, 0xF, true);
        until += __builtin_amdgcn_update_dpp(0, until, 0x118, 0xF, 0xF, true);
        const int behind = (int)(__ballot(v < until) & ((1ull << kInlineGroups) - 1));
        if (behind) {
            gi = __builtin_ctz(behind);
            v += __builtin_amdgcn_readlane(first - (until - count), gi);
            break;
        }
        v -= __builtin_amdgcn_readlane(until, kInlineGroups - 1);
        int skipped = 0;
        for (gi = kInlineGroups; gi < a.n_groups; ++gi) {
            const int n = (int)groups[gi].n_tiles;
            skipped = tiles_before(n, part.from);
            const int mine = tiles_before(n, part.upto) - skipped;
            if (v < mine) break;
            v -= mine;
        }
        if (gi < a.n_groups) {
            v += skipped;
            break;
        }
        if (part.next == 0) return;
        part = XcdPart{part.slice + 1, 0, part.next, 0};
    }
    const size_t skip = (size_t)part.slice * a.feat;
    a.C += skip;
    a.partials += (size_t)part.slice * a.slice_partials;
    a.heavy += (size_t)part.slice * a.slice_heavy;
    a.feat = min(a.feat, a.all_feat - (int)skip);
    const Group g = load_group(groups + gi);
    const RowsOfB<LPR, CH, BT, WIDE> b((const char*)a.B + skip * Dense<BT>::kElemBytes, a.b_bytes - skip * Dense<BT>::kElemBytes,
                                       Lane<LPR, CH, Dense<BT>::kVec>(threadIdx.x % LPR, a.feat, a.ldb, a.ldc));
    switch (g.type) {
        case kEll:
        case kEllSeg: run_ell_tile(b, g, v, s_pairs, s_rm, &s_next, s_dyn, a); break;
        case kSeg: run_seg_tile(b, g, v, a); break;
        case kZero: run_zero_tile<LPR, CH, BT>(g, v, a); break;
        default: run_chunk_tile(b, g, v, reinterpret_cast<float*>(s_raw), a); break;
    }
}

// Rows of many partial rows (dense rows cut into short chunks; more than kWideFinalPartials): one workgroup per
// row, sub-wave s adds partial rows s, s + SW, s + 2 SW, ... four at a time, and the sub-waves'
// sums are added in sub-wave order - a fixed order, so the result does not depend on scheduling.
template <int LPR, int CH, typename BT>
__global__ void __launch_bounds__(kWG)
spmm_finalize_wide_kernel(const HeavyRow* __restrict__ heavy, int n_heavy, LaunchArgs a) {
    constexpr int VEC = Dense<BT>::kVec;
    constexpr int SW = kWG / LPR;
    constexpr int U = 4;
    __shared__ float s_red[kWG * CH * VEC];
    const int sw = threadIdx.x / LPR, sl = threadIdx.x % LPR;
    const int skip = blockIdx.y * a.feat;                   // the feature slice
    a.C += skip;
    a.partials += (size_t)blockIdx.y * a.slice_partials;
    a.feat = min(a.feat, a.all_feat - skip);
    const Lane<LPR, CH, VEC> ln(sl, a.feat, a.ldb, a.ldc);
    const int h = blockIdx.x;
    if (h >= n_heavy) return;
    const HeavyRow hr = heavy[h];
    if (hr.n_partials <= kWideFinalPartials) return;
    Acc<CH, VEC> acc;
    acc.clear();
    for (int k0 = sw; k0 < hr.n_partials; k0 += SW * U) {
        float x[U][CH][VEC];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(k0 + u * SW, hr.n_partials - 1);      // (clamped loads, masked below)
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const float* src = a.partials + (size_t)(hr.partial_begin + k) * a.feat + (ln.on[c] ? ln.f[c] : 0);
#pragma unroll
                for (int i = 0; i < VEC; i += 4) {
                    const float4 v = *reinterpret_cast<const float4*>(src + i);
                    x[u][c][i] = v.x; x[u][c][i + 1] = v.y; x[u][c][i + 2] = v.z; x[u][c][i + 3] = v.w;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k0 + u * SW >= hr.n_partials) break;
#pragma unroll
            for (int c = 0; c < CH; ++c)
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc.v[c][i] += x[u][c][i];
        }
    }
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int i = 0; i < VEC; ++i) s_red[((sw * CH + c) * LPR + sl) * VEC + i] = acc.v[c][i];
    __syncthreads();
    if (sw == 0) {
        Acc<CH, VEC> sum;
        sum.clear();
#pragma unroll
        for (int c = 0; c < CH; ++c)
            for (int s2 = 0; s2 < SW; ++s2)
#pragma unroll
                for (int i = 0; i < VEC; ++i) sum.v[c][i] += s_red[((s2 * CH + c) * LPR + sl) * VEC + i];
        store_row<LPR, CH, VEC>(a.C, hr.row, ln, sum, a.accumulate);
    }
}

// ------------------------------------------------------------------------------------
// Row groups.  In a banded, stencil or block-structured matrix consecutive rows hold mostly
// the same columns; a bucket of such rows is rewritten at plan time as groups of four
// consecutive ELL rows with the union of their columns ("merged entries": column, four
// values, a 4-bit presence mask), and one gather of a B row then feeds up to four output
// rows.  The 27-point stencil needs 54 gathers per four rows instead of 4 x 28.  Only
// buckets whose merged entries are well below their slots take this path (measured at plan
// time); a matrix without shared columns never does.  Separate kernel, so that its registers
// (four accumulators) do not weigh on the main one.
constexpr int kGroupRows = 4;
#ifndef LF_MERGED_CAP
#define LF_MERGED_CAP 1024
#endif
constexpr int kMergedCap = LF_MERGED_CAP;   // merged entries staged per workgroup at most
constexpr int kMergedTileGroups = 64;  // row groups per tile at most
constexpr long long kRowGroupMinRows = 4096;   // smaller buckets are not worth the analysis
constexpr int kRowGroupSample = 4096;          // the decision looks at about this many groups of a bucket first
constexpr int kRowGroupMaxPercent = 70;        // merged entries / plain gathers at most, in percent
constexpr int kRowGroupSampleEntries = 24;     // merged entries of a group that the sampling pass looks at
constexpr int kLdsOfCu = 160 << 10, kLdsStep = 1280;
constexpr double kFarSliceBytes = 64e6;

struct MergedBucket {
    long long n_groups;        // row groups
    long long n_rows;          // ELL rows of the bucket (the last group may hold fewer than four)
    long long n_tiles;
    int groups_per_tile;
    int pad_;
    const int32_t* rows;       // [n_rows] source rows of the bucket
    const int32_t* goff;       // [n_groups + 1] first merged entry of each group
    const int32_t* ecol;       // [entries]
    const float4* eval;        // [entries] the four rows' values, 0 where a row lacks the column
    const uint8_t* emask;      // [entries] bit r: row r of the group holds the column
};

// Merges the (ascending) column lists of the rows of group g; calls emit(col, vals[4], mask)
// per merged entry when kEmit, and returns the number of merged entries.
template <bool kEmit, typename Emit>
__device__ __forceinline__ int merge_group(const int32_t* __restrict__ cols, const float* __restrict__ vals,
                                           const int32_t* __restrict__ meta, long long g, long long n_rows,
                                           int log_w, Emit emit) {
    // Four columns (and values) of every row are held in registers and refilled with one
    // 16-byte load: a row starts at a multiple of its width (>= 8 slots), so the loads are
    // aligned, and the chain of dependent loads is a quarter as long.
    int len[kGroupRows], pos[kGroupRows];
    long long base[kGroupRows];
    int4 cbuf[kGroupRows];
    float4 vbuf[kGroupRows];
#pragma unroll
    for (int r = 0; r < kGroupRows; ++r) {
        const long long e = g * kGroupRows + r;
        len[r] = e < n_rows ? (meta[e] & (int)kMetaLenMask) : 0;
        base[r] = e << log_w;
        pos[r] = 0;
        cbuf[r] = make_int4(0, 0, 0, 0);
        vbuf[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (len[r] > 0) {
            cbuf[r] = *reinterpret_cast<const int4*>(cols + base[r]);
            if (kEmit) vbuf[r] = *reinterpret_cast<const float4*>(vals + base[r]);
        }
    }
    auto pick = [](const int4& q, int i) { return i == 0 ? q.x : i == 1 ? q.y : i == 2 ? q.z : q.w; };
    auto pickf = [](const float4& q, int i) { return i == 0 ? q.x : i == 1 ? q.y : i == 2 ? q.z : q.w; };
    int m = 0;
    for (;;) {
        int head[kGroupRows];
        int cmin = 0x7FFFFFFF;
#pragma unroll
        for (int r = 0; r < kGroupRows; ++r) {
            head[r] = pos[r] < len[r] ? pick(cbuf[r], pos[r] & 3) : 0x7FFFFFFF;
            cmin = min(cmin, head[r]);
        }
        if (cmin == 0x7FFFFFFF) break;
        float v[kGroupRows];
        uint32_t mask = 0;
#pragma unroll
        for (int r = 0; r < kGroupRows; ++r) {
            v[r] = 0.f;
            if (head[r] == cmin) {
                if (kEmit) v[r] = pickf(vbuf[r], pos[r] & 3);
                mask |= 1u << r;
                ++pos[r];
                if ((pos[r] & 3) == 0 && pos[r] < len[r]) {
                    cbuf[r] = *reinterpret_cast<const int4*>(cols + base[r] + pos[r]);
                    if (kEmit) vbuf[r] = *reinterpret_cast<const float4*>(vals + base[r] + pos[r]);
                }
            }
        }
        if (kEmit) emit(m, cmin, v, mask);
        ++m;
    }
    return m;
}

// One bucket of the row-group analysis.
struct RowGroupCand {
    const int32_t* cols;
    const int32_t* meta;
    long long n_rows;
    long long n_groups;
    int32_t* m_out;            // merged length of every group
    int log_w;
    int pad_;
};

// One atomic per wavefront and counter: [0] sum of m, [1] sum of plain, [2] largest m.
__device__ __forceinline__ void add_rowgroup_counters(int sm, int sp, int mx, unsigned long long* __restrict__ c) {
    for (int d = 32; d > 0; d >>= 1) {
        sm += __shfl_xor(sm, d);
        sp += __shfl_xor(sp, d);
        mx = max(mx, __shfl_xor(mx, d));
    }
    if ((threadIdx.x & 63) == 0 && sp > 0) {
        atomicAdd(&c[0], (unsigned long long)sm);
        atomicAdd(&c[1], (unsigned long long)sp);
        atomicMax(&c[2], (unsigned long long)mx);
    }
}

// counters[3 * i + ...] of bucket i = blockIdx.y: merged entries, gathers of the plain path (row
// lengths rounded up to the unroll), longest group.
__global__ void __launch_bounds__(256)
rowgroup_count_kernel(const RowGroupCand* __restrict__ cands, unsigned long long* __restrict__ counters) {
    const RowGroupCand cd = cands[blockIdx.y];
    const long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    int m = 0, plain = 0;
    if (g < cd.n_groups) {
        m = merge_group<false>(cd.cols, nullptr, cd.meta, g, cd.n_rows, cd.log_w, [](int, int, const float*, uint32_t) {});
        for (int r = 0; r < kGroupRows; ++r) {
            const long long e = g * kGroupRows + r;
            if (e < cd.n_rows) plain += ((cd.meta[e] & (int)kMetaLenMask) + kUnroll - 1) / kUnroll * kUnroll;
        }
        cd.m_out[g] = m;
    }
    add_rowgroup_counters(m, plain, m, counters + 3 * blockIdx.y);
}

__global__ void __launch_bounds__(256)
rowgroup_fill_kernel(const int32_t* __restrict__ cols, const float* __restrict__ vals,
                     const int32_t* __restrict__ meta, long long n_rows, int log_w, long long n_groups,
                     const int32_t* __restrict__ goff, int32_t* __restrict__ ecol, float4* __restrict__ eval,
                     uint8_t* __restrict__ emask) {
    const long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_groups) return;
    const long long at = goff[g];
    merge_group<true>(cols, vals, meta, g, n_rows, log_w, [&](int j, int c, const float* v, uint32_t mask) {
        ecol[at + j] = c;
        eval[at + j] = make_float4(v[0], v[1], v[2], v[3]);
        emask[at + j] = (uint8_t)mask;
    });
}

// One workgroup per tile of row groups, XCD-aware like the main kernel.  CH == 1 only.
template <int LPR, typename BT>
__global__ void __launch_bounds__(kWG)
spmm_rowgroup_kernel(const MergedBucket* __restrict__ buckets, int n_buckets, LaunchArgs a) {
    constexpr int VEC = Dense<BT>::kVec;
    constexpr int SW = kWG / LPR;
    // Gathers of a sub-wave, and staged entries of a thread, requested together.  27-point stencils, N = 128 .. 256 bf16, 4 and 8 gathers: 30.6,
    // 28.8 us (38 x 71 x 22), 31.3, 29.1 (34 x 40 x 45); N = 448, where a sub-wave is a wavefront and skips rows: 111, 120.  Entries by 1, 2, 4:
    // N = 448 111, 107, 100; N = 128 30.6, 29.7, 30.2; f32 N = 224 32.4, 31.7, 32.1.
    constexpr bool kWideRow = VEC == 8 && LPR == 64;
    constexpr int U = kWideRow ? 4 : 8, kStage = kWideRow ? 4 : 2;
    __shared__ float4 s_val[kMergedCap];
    __shared__ int s_col[kMergedCap];
    __shared__ int s_goff[kMergedTileGroups + 1];
    __shared__ uint8_t s_msk[kMergedCap];

    const int xcd = blockIdx.x % kXcds;
    long long v = blockIdx.x / kXcds;
    for (int bi = 0; bi < n_buckets; ++bi) {
        const MergedBucket& b = buckets[bi];
        const long long lo = b.n_tiles * xcd / kXcds;
        const long long hi = b.n_tiles * (xcd + 1) / kXcds;
        if (v >= hi - lo) { v -= hi - lo; continue; }
        const long long g0 = (lo + v) * b.groups_per_tile;
        const int n = (int)min((long long)b.groups_per_tile, b.n_groups - g0);
        const int tid = threadIdx.x;
        // (pointers out of a table are generic to the compiler: flat loads, which wait for the LDS counter too)
        typedef const int32_t __attribute__((address_space(1)))* GlobalInts;
        typedef float Four __attribute__((ext_vector_type(4)));
        const GlobalInts goff = (GlobalInts)(uintptr_t)b.goff, ecol = (GlobalInts)(uintptr_t)b.ecol, rows = (GlobalInts)(uintptr_t)b.rows;
        const auto eval = (const Four __attribute__((address_space(1)))*)(uintptr_t)b.eval;
        const auto emask = (const uint8_t __attribute__((address_space(1)))*)(uintptr_t)b.emask;
        for (int i = tid; i <= n; i += kWG) s_goff[i] = goff[g0 + i];
        __syncthreads();
        const int sw = tid / LPR, sl = tid % LPR;
        const Lane<LPR, 1, VEC> ln(sl, a.feat, a.ldb, a.ldc);
        // The tile's groups are staged in rounds of as many whole groups as the buffer holds
        // (one group always fits: the plan checks the longest group against the capacity).
        for (int ga = 0; ga < n;) {
            const int base = s_goff[ga];
            int gb = ga + 1;
            while (gb < n && s_goff[gb + 1] - base <= kMergedCap) ++gb;      // uniform
            const int n_entries = s_goff[gb] - base;
            for (int i0 = tid; i0 < n_entries; i0 += kStage * kWG) {
                Four v[kStage];
                int c[kStage];
                uint8_t k[kStage];
#pragma unroll
                for (int u = 0; u < kStage; ++u) {
                    const int i = base + min(i0 + u * kWG, n_entries - 1);
                    v[u] = eval[i];
                    c[u] = ecol[i];
                    k[u] = emask[i];
                }
#pragma unroll
                for (int u = 0; u < kStage; ++u) {
                    const int i = min(i0 + u * kWG, n_entries - 1);
                    s_col[i] = c[u];
                    s_val[i] = make_float4(v[u].x, v[u].y, v[u].z, v[u].w);
                    s_msk[i] = k[u];
                }
            }
            __syncthreads();
            for (int gi = ga + sw; gi < gb; gi += SW) {
                const int e0 = s_goff[gi] - base;
                const int m = s_goff[gi + 1] - s_goff[gi];
                Acc<1, VEC> acc[kGroupRows];
#pragma unroll
                for (int r = 0; r < kGroupRows; ++r) acc[r].clear();
                for (int j = 0; j < m; j += U) {
                    int c[U];
                    float4 w[U];
                    uint32_t k[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const bool in = j + u < m;
                        const int idx = e0 + (in ? j + u : 0);   // past the end: the first column again, nothing added
                        c[u] = s_col[idx];
                        w[u] = in ? s_val[idx] : make_float4(0.f, 0.f, 0.f, 0.f);
                        k[u] = in ? s_msk[idx] : 0u;
                    }
                    typename Dense<BT>::Raw raw[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) raw[u] = load_dense<BT>(a.B, ln, 0, c[u]);
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        float x[VEC];
                        Dense<BT>::unpack(raw[u], x);
                        const float wr[kGroupRows] = {w[u].x, w[u].y, w[u].z, w[u].w};
#pragma unroll
                        for (int r = 0; r < kGroupRows; ++r) {
                            if constexpr (LPR == 64) {
                                // one group per wavefront: rows without the column are skipped outright
                                if (__builtin_amdgcn_readfirstlane(k[u]) & (1u << r)) {
#pragma unroll
                                    for (int i = 0; i < VEC; ++i) acc[r].v[0][i] = fmaf(wr[r], x[i], acc[r].v[0][i]);
                                }
                            } else {
                                // several groups per wavefront: the value is 0 where the row lacks the
                                // column (like a padded slot, this adds 0 * B: only non-finite B differs)
#pragma unroll
                                for (int i = 0; i < VEC; ++i) acc[r].v[0][i] = fmaf(wr[r], x[i], acc[r].v[0][i]);
                            }
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < kGroupRows; ++r) {
                    const long long e = (g0 + gi) * kGroupRows + r;
                    if (e < b.n_rows) store_row<LPR, 1, VEC>(a.C, rows[e], ln, acc[r], a.accumulate);
                }
            }
            ga = gb;
            if (ga < n) __syncthreads();                 // the buffer is refilled
        }
        return;
    }
}

// ------------------------------------------------------------------------------------
// Plan-time kernels.

// Inclusive scans over a 256-thread workgroup: the largest value at or before a thread, the
// smallest value at or after it.  s_wave: 4 ints of LDS.
__device__ __forceinline__ int block_scan_max_fwd(int x, int* s_wave) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d);
        if (lane >= d) x = max(x, y);
    }
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    for (int w = 0; w < wave; ++w) x = max(x, s_wave[w]);
    __syncthreads();
    return x;
}

__device__ __forceinline__ int block_scan_min_bwd(int x, int* s_wave) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_down(x, d);
        if (lane + d < 64) x = min(x, y);
    }
    if (lane == 0) s_wave[wave] = x;
    __syncthreads();
    for (int w = wave + 1; w < 4; ++w) x = min(x, s_wave[w]);
    __syncthreads();
    return x;
}

// meta from rows / vals for slabs that come without one (the reference passes rows, cols and
// values only, format_algos.py:552-578): len = position of the last nonzero value + 1 (at
// least 1); a run of equal row ids is one segment.  Two passes, so that a long run costs a
// scan and not a walk per ELL row: the first notes, per block of 256 ELL rows, its first and
// its last segment head (an ELL row whose predecessor carries another row id); the second
// finds for every ELL row the head at or before it and, for a head, the next head.
__global__ void __launch_bounds__(256)
derive_heads_kernel(const int32_t* __restrict__ rows, long long n_rows, int32_t* __restrict__ blk_first,
                    int32_t* __restrict__ blk_last) {
    __shared__ int s_wave[4];
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    const bool head = e < n_rows && (e == 0 || rows[e - 1] != rows[e]);
    const int last = block_scan_max_fwd(head ? (int)e : -1, s_wave);
    const int first = block_scan_min_bwd(head ? (int)e : 0x7FFFFFFF, s_wave);
    if (threadIdx.x == 255) blk_last[blockIdx.x] = last;
    if (threadIdx.x == 0) blk_first[blockIdx.x] = first;
}

// flags[3] is raised when a segment is longer than the meta word can say.
__global__ void __launch_bounds__(256)
derive_meta_kernel(const int32_t* __restrict__ rows, const float* __restrict__ vals, long long n_rows,
                   int log_w, const int32_t* __restrict__ blk_first, const int32_t* __restrict__ blk_last,
                   int n_blocks, int32_t* __restrict__ meta, int* __restrict__ flags) {
    __shared__ int s_wave[4];
    __shared__ int s_prev, s_next;
    if (threadIdx.x == 0) {                      // heads outside this block (block 0 starts with one)
        int b = (int)blockIdx.x - 1;
        while (b >= 0 && blk_last[b] < 0) --b;
        s_prev = b >= 0 ? blk_last[b] : 0;
        b = (int)blockIdx.x + 1;
        while (b < n_blocks && blk_first[b] == 0x7FFFFFFF) ++b;
        s_next = b < n_blocks ? blk_first[b] : (int)n_rows;
    }
    __syncthreads();
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    const bool in = e < n_rows;
    const bool head = in && (e == 0 || rows[e - 1] != rows[e]);
    int prev = block_scan_max_fwd(head ? (int)e : -1, s_wave);
    // the next head strictly after e: the smallest head at or after the thread's successor
    __shared__ int s_at_or_after[257];
    s_at_or_after[threadIdx.x] = block_scan_min_bwd(head ? (int)e : 0x7FFFFFFF, s_wave);
    if (threadIdx.x == 0) s_at_or_after[256] = 0x7FFFFFFF;
    __syncthreads();
    int next = s_at_or_after[threadIdx.x + 1];
    if (!in) return;
    if (prev < 0) prev = s_prev;
    if (next == 0x7FFFFFFF) next = min(s_next, (int)n_rows);
    const int w = 1 << log_w;
    const float* rv = vals + (e << log_w);
    int len = 1;
    for (int j = w - 1; j > 0; --j)
        if (rv[j] != 0.f) { len = j + 1; break; }
    uint32_t field, cont = 0;
    if (head) {
        field = (uint32_t)(next - (int)e);
    } else {
        field = (uint32_t)((int)e - prev);
        cont = 0x80000000u;
    }
    if (field >= (1u << (31 - kMetaLenBits))) {
        flags[3] = 1;
        field = 1;                                 // keep the word well formed; the plan is refused
    }
    meta[e] = (int32_t)((uint32_t)len | (field << kMetaLenBits) | cont);
}

// One ELL row as the chunk planner sees it.
struct ChunkedRow {
    long long total;     // slots of its segment
    int n_chunks;        // 0: no head of a segment that takes the cooperative path
    int chunk_slots;
    int found;           // 1 part of a split row, 2 dense row, 4 more than kWideFinalPartials chunks
};

// Row e of a bucket, whose meta word is m; tail: the meta word at tail_of(m, e, n_rows).
__device__ __forceinline__ long long tail_of(int m, long long e, long long n_rows) {
    return m < 0 ? e : min(max(e + (int)((uint32_t)m >> kMetaLenBits) - 1, e), n_rows - 1);
}
__device__ __forceinline__ ChunkedRow chunked_row(int m, int tail, long long e, long long n_rows, int log_w, int coop_slots, int chunk_slots,
                                                  long long dense_min_slots) {
    ChunkedRow x{0, 0, chunk_slots, 0};
    if (m < 0) {
        x.found = 1;
        return x;
    }
    const int seg = (int)((uint32_t)m >> kMetaLenBits);
    if (seg > 1) x.found = 1;
    // The counting pass is enqueued together with the slab checks, before their verdict has been
    // read: a head that announces more ELL rows than the bucket holds (which the checks flag and
    // the plan is then refused) must not be followed past the array.
    if (((long long)seg << log_w) > coop_slots && e + seg <= n_rows) {
        x.total = ((long long)(seg - 1) << log_w) + (tail & (int)kMetaLenMask);
        if (x.total >= dense_min_slots) {
            x.chunk_slots = kDenseChunkSlots;
            x.found |= 2;
        }
        x.n_chunks = (int)((x.total + x.chunk_slots - 1) / x.chunk_slots);
        if (x.n_chunks > kWideFinalPartials) x.found |= 4;
    }
    return x;
}

// One bucket as the plan-time kernels see it.
struct PlanBucket {
    const int32_t* rows;
    const int32_t* meta;
    const int32_t* cols;
    long long n_rows;
    int log_w;
    int part;
    int n_blocks;              // workgroups of plan_scan_kernel, behind n_first others
    int n_first;               // one for the span, and those of the row-group sampling; none without n_blocks
    int sample_stride;         // row-group sampling: every sample_stride-th group is looked at (0: no candidate)
    int span_stride;           // every span_stride-th row is looked at for the span of neighbours' columns
    int all_cols;              // columns of a partition
    int first_line, n_lines;   // of its counters
};

// One pass over all buckets of a plan:
//   * checks what the SpMM kernels take on trust: source rows inside the matrix, column indices
//     inside B, 1..W valid slots per ELL row, and segments (a head that announces n ELL rows followed
//     by continuation rows 1..n-1 with the same row id) that are complete and stay inside the
//     bucket.  flags[0] bad column, [1] bad row, [2] bad meta;
//   * counts what lf_spmm_create sizes its tables by: counter i, in each of the bucket's lines, of bucket
//     k = chunks of the rows of more than kCoopSlots slots, rows with several chunks, their partial
//     rows, rows of 65 .. 128 and of 129 .. kCoopSlots slots (a chunk each if they take the cooperative
//     path), ChunkedRow::found of all rows; and by a workgroup of its own, not to lengthen the others, the columns that
//     groups of kGroupRows neighbours span (every span_stride-th row and those behind it, in kSpanUnits of all columns; all,
//     where one is a part of a row, which says nothing);
//   * marks the rows that partition 0 writes;
//   * samples the row-group candidates: of every sample_stride-th group of four rows, samples[3 k ..] = merged entries among the
//     first kRowGroupSampleEntries, the slots they consumed, the largest count.  By workgroups of their own, which start first
//     and stage the first slots of their rows in LDS (merged out of memory, a group to a lane, each step waited for a load: 19 us of
//     the 21 that the scan of a 170K-row graph took, now 10 of 13; 115 behind the stream of a large one, now 20).  (Nothing here is
//     followed out of the slabs, whatever the meta words say; where a check fails the samples are not read.)
// Bound by the stream of the column slabs.  Workgroup -> bucket by the first workgroups of the
// buckets, so that all of them share one launch however many there are: three launches per bucket
// (checks, counts, marks) were 60 us of GPU time for the 11 buckets of a 170K-row graph, whose slabs
// take 3 us to read, and each read the row ids or the meta words again.  Together the workgroups fill the GPU once: 1024 to a
// bucket left a second, nearly empty round of them.  No load is behind a condition, where it would wait for the one before.
// 2.45M-row graph, widths 1 .. 32, behind the builder: 147 + 26 us with the samples, now 123, of which 60 take its slabs at 5.7 TB/s
// and as many the rows.
constexpr int kScanSlotsPerBlock = 16384, kScanRowsPerBlock = 1024;  // at least
constexpr int kScanBlocksPerCu = 7;
constexpr int kScanRows = 4;               // ELL rows of a thread requested together
constexpr int kScanUnroll = 4;             // 16-byte loads of columns in flight per thread
constexpr int kScanCounters = 7, kScanFound = 5, kScanSpan = 6;
constexpr int kSampleGroups = 64, kSampleRound = 32;       // of a workgroup, and staged together
constexpr int kSpanUnits = 4096, kSpanSamples = 1024;      // (twice the samples at most: sums below 2^24)
// Atomics on one line are taken one after the other, 17 to 40 ns each, and the workgroups of a bucket end together: up to 16
// lines share them.
constexpr int kScanLinesMost = 16, kScanBlocksPerLine = 64;
constexpr int kCounterLine = 32;           // words between the cursors of a bucket: each has a 128-byte line of its
                                           // own, as atomics on one line are taken one after the other (17 ns each)
__global__ void __launch_bounds__(256)
plan_scan_kernel(const PlanBucket* __restrict__ buckets, const int32_t* __restrict__ first_block, int n_buckets,
                 long long num_rows, long long num_cols, int chunk_slots, long long dense_min_slots,
                 int* __restrict__ counters, int* __restrict__ flags, uint8_t* __restrict__ covered,
                 unsigned long long* __restrict__ samples) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int k = -1;                                       // last bucket whose first workgroup is not behind this one
    for (int i = 0; i < n_buckets; i += 64)
        k += __popcll(__ballot(i + lane < n_buckets && first_block[i + lane] <= (int)blockIdx.x));
    k = __builtin_amdgcn_readfirstlane(k);
    const PlanBucket bk = buckets[k];
    const long long stride = (long long)bk.n_blocks * 256;
    const int place = (int)blockIdx.x - first_block[k];
    const long long t0 = ((long long)place - bk.n_first) * 256 + threadIdx.x;
    // (pointers out of a table are generic to the compiler: flat loads, which wait for the LDS counter too)
    typedef const int32_t __attribute__((address_space(1)))* GlobalInts;
    typedef int Four __attribute__((ext_vector_type(4), aligned(4)));
    typedef const Four __attribute__((address_space(1)))* GlobalFours;
    const GlobalInts rows = (GlobalInts)(uintptr_t)bk.rows, meta = (GlobalInts)(uintptr_t)bk.meta, cols = (GlobalInts)(uintptr_t)bk.cols;
    const int log_w = bk.log_w;
    const long long n_rows = bk.n_rows;
    if (place > 0 && place < bk.n_first) {                    // samples
        constexpr int kSlots = kRowGroupSampleEntries, kFours = kSlots / 4, kLine = kGroupRows * kSlots + 1;      // slots of a row that are looked at
        __shared__ int s_cols[kSampleRound][kLine];
        __shared__ int s_len[kSampleRound][kGroupRows];
        const int width = 1 << log_w;
        int merged = 0, plain = 0, most = 0;
        for (int g0 = 0; g0 < kSampleGroups; g0 += kSampleRound) {
            auto row_at = [&](int g, int r) { return ((long long)(place - 1) * kSampleGroups + g0 + g) * bk.sample_stride * kGroupRows + r; };
            Four c[kSampleRound * kGroupRows * kFours / 256];
#pragma unroll
            for (int t = 0; t < kSampleRound * kGroupRows * kFours / 256; ++t) {
                const int i = t * 256 + threadIdx.x, q = i % kFours, r = i / kFours % kGroupRows, g = i / (kFours * kGroupRows);
                c[t] = *(GlobalFours)(cols + (min(row_at(g, r), n_rows - 1) << log_w) + min(q * 4, width - 4));
            }
            if (threadIdx.x < kSampleRound * kGroupRows) {
                const int r = threadIdx.x % kGroupRows, g = threadIdx.x / kGroupRows;
                const int m = meta[min(row_at(g, r), n_rows - 1)];
                s_len[g][r] = row_at(g, r) < n_rows ? min(m & (int)kMetaLenMask, width) : 0;      // (not checked yet)
            }
#pragma unroll
            for (int t = 0; t < kSampleRound * kGroupRows * kFours / 256; ++t) {
                const int i = t * 256 + threadIdx.x, q = i % kFours, r = i / kFours % kGroupRows, g = i / (kFours * kGroupRows);
                int* to = &s_cols[g][r * kSlots + q * 4];
                to[0] = c[t].x, to[1] = c[t].y, to[2] = c[t].z, to[3] = c[t].w;
            }
            __syncthreads();
            if (threadIdx.x < kSampleRound) {
                const int g = threadIdx.x;
                int pos[kGroupRows] = {}, head[kGroupRows], m = 0;
                for (; m < kRowGroupSampleEntries; ++m) {
                    int least = 0x7FFFFFFF;
#pragma unroll
                    for (int r = 0; r < kGroupRows; ++r) {
                        head[r] = pos[r] < s_len[g][r] ? s_cols[g][r * kSlots + pos[r]] : 0x7FFFFFFF;
                        least = min(least, head[r]);
                    }
                    if (least == 0x7FFFFFFF) break;
#pragma unroll
                    for (int r = 0; r < kGroupRows; ++r) pos[r] += head[r] == least;
                }
                plain += pos[0] + pos[1] + pos[2] + pos[3];
                merged += m;
                most = max(most, m);
            }
            __syncthreads();
        }
        if (threadIdx.x < 64) add_rowgroup_counters(merged, plain, most, samples + 3 * k);
        return;
    }
    if (place == 0) {                                         // span
        int span = 0;
        for (long long e = (long long)threadIdx.x * bk.span_stride; e < n_rows; e += 256ll * bk.span_stride) {
            int first = 0x7FFFFFFF, last = 0;
            bool whole = true;
#pragma unroll
            for (int r = 0; r < kGroupRows; ++r) {
                const long long q = min(e + r, n_rows - 1), at = q << log_w;
                const int m = meta[q], n = min(max(m & (int)kMetaLenMask, 1), 1 << log_w);       // (not checked yet)
                whole = whole && m >> kMetaLenBits == 1;
                first = min(first, cols[at]);
                last = max(last, cols[at + n - 1]);
            }
            const long long columns = whole ? max((long long)last - first, 0ll) : bk.all_cols;
            span += (int)min((long long)kSpanUnits, columns * kSpanUnits / bk.all_cols);
        }
        for (int d = 32; d > 0; d >>= 1) span += __shfl_xor(span, d);
        if (lane == 0 && span > 0) atomicAdd(counters + (size_t)bk.first_line * kCounterLine + kScanSpan, span);
        return;
    }
    bool bad_col = false, bad_row = false, bad_meta = false;
    const long long n_slots = n_rows << log_w;
    const unsigned limit = (unsigned)num_cols;               // < 2^31
    const long long round = stride * 4 * kScanUnroll;       // from the end: what the builder wrote last may still be in the memory-side cache (143 -> 131 us)
    if (n_slots < 4) {
        if (t0 < n_slots) bad_col = (unsigned)cols[t0] >= limit;
    } else {
        for (long long i = t0 * 4 + (n_slots - 1) / round * round; i >= 0; i -= round) {
            Four c[kScanUnroll];
#pragma unroll
            for (int u = 0; u < kScanUnroll; ++u)                // (no load behind a condition: they would wait for one another)
                c[u] = *(GlobalFours)(cols + min(i + u * stride * 4, n_slots - 4));
#pragma unroll
            for (int u = 0; u < kScanUnroll; ++u)
                bad_col |= (unsigned)c[u].x >= limit || (unsigned)c[u].y >= limit || (unsigned)c[u].z >= limit || (unsigned)c[u].w >= limit;
        }
    }
    constexpr int kSums = kScanFound;
    int sum[kSums] = {}, found = 0;
    for (long long e0 = t0; e0 < n_rows; e0 += stride * kScanRows) {
        int row_of[kScanRows], meta_of[kScanRows], next_of[kScanRows];
#pragma unroll
        for (int u = 0; u < kScanRows; ++u) {                 // requested together
            const long long e = min(e0 + u * stride, n_rows - 1);
            row_of[u] = rows[e];
            meta_of[u] = meta[e];
            next_of[u] = meta[min(e + 1, n_rows - 1)];
        }
        int there_meta[kScanRows], there_row[kScanRows];      // of a segment's head its last ELL row, of the others the head
#pragma unroll
        for (int u = 0; u < kScanRows; ++u) {
            const long long e = min(e0 + u * stride, n_rows - 1), back = (long long)(((uint32_t)meta_of[u] & 0x7FFFFFFFu) >> kMetaLenBits);
            const long long there = meta_of[u] < 0 ? max(e - back, 0ll) : tail_of(meta_of[u], e, n_rows);
            there_meta[u] = meta[there];
            there_row[u] = rows[there];
        }
#pragma unroll
        for (int u = 0; u < kScanRows; ++u) {
            const long long e = e0 + u * stride;
            if (e >= n_rows) break;
            const int row = row_of[u];
            const bool row_ok = (unsigned)row < (unsigned long long)num_rows;
            bad_row |= !row_ok;
            if (bk.part == 0 && row_ok) covered[row] = 1;
            const int m = meta_of[u];
            const int len = m & (int)kMetaLenMask;
            bad_meta |= len < 1 || len > (1 << log_w);
            const long long field = (long long)(((uint32_t)m & 0x7FFFFFFFu) >> kMetaLenBits);
            // what the next ELL row must be: a continuation row with index `want`, or a head (0)
            long long want = 0;
            if (m >= 0) {
                bad_meta |= field < 1 || e + field > n_rows;
                want = field > 1 ? 1 : 0;
            } else {
                const long long h = e - field;
                if (field < 1 || h < 0) {
                    bad_meta = true;
                } else {
                    const int hm = there_meta[u];
                    const long long n = (long long)((uint32_t)hm >> kMetaLenBits);
                    bad_meta |= hm < 0 || field >= n || there_row[u] != row;
                    want = field + 1 < n ? field + 1 : 0;
                }
            }
            if (e == 0) bad_meta |= m < 0;
            if (e + 1 < n_rows) {
                const int nm = next_of[u];
                const long long nf = (long long)(((uint32_t)nm & 0x7FFFFFFFu) >> kMetaLenBits);
                bad_meta |= want == 0 ? nm < 0 : (nm >= 0 || nf != want);
            } else {
                bad_meta |= want != 0;
            }
            const ChunkedRow x = chunked_row(m, there_meta[u], e, n_rows, log_w, kCoopSlots, chunk_slots, dense_min_slots);
            found |= x.found;
            sum[0] += x.n_chunks;
            sum[1] += x.n_chunks > 1;
            sum[2] += x.n_chunks > 1 ? x.n_chunks : 0;
            const long long slots = m >= 0 ? field << log_w : 0;     // of the row that starts here
            sum[3] += slots > 64 && slots <= 128;
            sum[4] += slots > 128 && slots <= kCoopSlots;
        }
    }
    if (__ballot(bad_col) != 0 && lane == 0) flags[0] = 1;
    if (__ballot(bad_row) != 0 && lane == 0) flags[1] = 1;
    if (__ballot(bad_meta) != 0 && lane == 0) flags[2] = 1;
    // one atomic per workgroup and counter
    __shared__ int s_sum[4][kSums + 1];
    for (int d = 32; d > 0; d >>= 1) {
        found |= __shfl_xor(found, d);
        for (int i = 0; i < kSums; ++i) sum[i] += __shfl_xor(sum[i], d);
    }
    if (lane == 0) {
        for (int i = 0; i < kSums; ++i) s_sum[wave][i] = sum[i];
        s_sum[wave][kSums] = found;
    }
    __syncthreads();
    const int i = threadIdx.x;
    int* mine = counters + (size_t)(bk.first_line + place % bk.n_lines) * kCounterLine + min(i, kSums);
    if (i < kSums) {
        const int all = s_sum[0][i] + s_sum[1][i] + s_sum[2][i] + s_sum[3][i];
        if (all) atomicAdd(mine, all);
    } else if (i == kSums) {
        const int all = s_sum[0][i] | s_sum[1][i] | s_sum[2][i] | s_sum[3][i];
        // what the shared word holds already need not be added again
        if ((all & ~__hip_atomic_load(mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0) atomicOr(mine, all);
    }
}

// Fills the chunk tables of up to kChunkBuckets buckets (rows of more than coop_slots slots, cut into chunks) and their
// parts of the heavy-row table.  cursors (kCounterLine words apart): chunks, rows with several chunks
// and their partial rows handed out so far.  Table order depends on scheduling, results do not: every row's partials are
// private and are summed in chunk order.
// A workgroup takes kChunkRows ELL rows, all their loads in flight together, and its ranges of the tables with one atomic
// per counter.  With one atomic per wavefront and counter, counting and filling the widest bucket of a folded 2.45M-row graph (850K
// ELL rows) took 1.35 ms, all of it updates of one cache line; a sweep that counts and one that fills, 448 rows to a wavefront one after the
// other, 43 us; now 26.  (One workgroup to 1024 rows 40: the atomics.)  One launch for the buckets of a plan: each waited for the one before.
constexpr int kChunkBuckets = 12, kChunkThreads = 1024, kChunkRowsOfThread = 4, kChunkRows = kChunkThreads * kChunkRowsOfThread;
struct ChunkBucket {
    const int32_t *rows, *meta, *cols;
    long long n_rows;
    Chunk* chunks;
    int* cursors;
    int log_w, partial_base, heavy_base, first_block;
};
struct ChunkBuckets {
    ChunkBucket of[kChunkBuckets];
    int n;
};
__global__ void __launch_bounds__(kChunkThreads)
plan_chunks_kernel(ChunkBuckets buckets, HeavyRow* __restrict__ heavy, int n_heavy, int slices, int coop_slots, int chunk_slots,
                   long long dense_min_slots) {
    __shared__ int s_wave[3][kChunkThreads / 64];
    __shared__ int s_base[3];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int k = 0;
    while (k + 1 < buckets.n && buckets.of[k + 1].first_block <= (int)blockIdx.x) ++k;
    const ChunkBucket& b = buckets.of[k];
    const int log_w = b.log_w;
    const long long e0 = ((long long)blockIdx.x - b.first_block) * kChunkRows + threadIdx.x;
    ChunkedRow x[kChunkRowsOfThread];
    int m[kChunkRowsOfThread], tail[kChunkRowsOfThread];
#pragma unroll
    for (int u = 0; u < kChunkRowsOfThread; ++u) m[u] = b.meta[min(e0 + u * kChunkThreads, b.n_rows - 1)];
#pragma unroll
    for (int u = 0; u < kChunkRowsOfThread; ++u) tail[u] = b.meta[tail_of(m[u], min(e0 + u * kChunkThreads, b.n_rows - 1), b.n_rows)];
    int mine[3] = {0, 0, 0};                 // chunks, rows with several, their partial rows
#pragma unroll
    for (int u = 0; u < kChunkRowsOfThread; ++u) {
        const long long e = e0 + u * kChunkThreads;
        x[u] = ChunkedRow{0, 0, chunk_slots, 0};
        if (e < b.n_rows) x[u] = chunked_row(m[u], tail[u], e, b.n_rows, log_w, coop_slots, chunk_slots, dense_min_slots);
        mine[0] += x[u].n_chunks;
        mine[1] += x[u].n_chunks > 1;
        mine[2] += x[u].n_chunks > 1 ? x[u].n_chunks : 0;
    }
    if (__syncthreads_or(mine[0]) == 0) return;
    int at[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        int incl = mine[i];
        for (int d = 1; d < 64; d <<= 1) {
            const int y = __shfl_up(incl, d);
            if (lane >= d) incl += y;
        }
        if (lane == 63) s_wave[i][wave] = incl;
        at[i] = incl - mine[i];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        int all = 0;
        for (int w = 0; w < kChunkThreads / 64; ++w) all += s_wave[threadIdx.x][w];
        s_base[threadIdx.x] = all ? atomicAdd(&b.cursors[threadIdx.x * kCounterLine], all) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        at[i] += s_base[i];
        for (int w = 0; w < wave; ++w) at[i] += s_wave[i][w];
    }
#pragma unroll
    for (int u = 0; u < kChunkRowsOfThread; ++u) {
        if (x[u].n_chunks == 0) continue;
        const long long e = e0 + u * kChunkThreads;
        const bool several = x[u].n_chunks > 1;
        const int row = b.rows[e], partial = b.partial_base + at[2], h = b.heavy_base + at[1];
        for (int i = 0; i < x[u].n_chunks; ++i) {
            const long long first = (long long)i * x[u].chunk_slots;
            Chunk ck;
            ck.slot_begin = (e << log_w) + first;
            ck.n_slots = (int)min((long long)x[u].chunk_slots, x[u].total - first) | (x[u].found & 2 ? kChunkDenseBit : 0);
            ck.partial = several ? partial + i : -1;
            ck.row = row;
            ck.first_col = b.cols[ck.slot_begin];
            ck.heavy = h;
            ck.pad_ = 0;
            b.chunks[at[0] + i] = ck;
        }
        for (int i = 0; i < slices && several; ++i)          // every feature slice counts its chunks
            heavy[(size_t)i * n_heavy + h] = HeavyRow{row, partial, x[u].n_chunks, 0};
        at[0] += x[u].n_chunks;
        at[1] += several;
        at[2] += several ? x[u].n_chunks : 0;
    }
}

// Rows that no bucket of partition 0 writes: counted (list == nullptr) or listed.  Each
// wavefront owns a contiguous range of rows and each workgroup takes its slice of the list
// with a single atomic: one atomic per wavefront was 38K updates of one address for 2.45M
// rows, 0.3 ms per pass.
__global__ void __launch_bounds__(256)
collect_uncovered_kernel(const uint8_t* __restrict__ covered, long long n_rows,
                         int* __restrict__ count, int32_t* __restrict__ list) {
    __shared__ int s_total[4];
    __shared__ int s_base;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long per_wave = ((n_rows + (long long)gridDim.x * 4 - 1) / ((long long)gridDim.x * 4) + 63) / 64 * 64;
    const long long lo = ((long long)blockIdx.x * 4 + wave) * per_wave;
    const long long hi = lo + per_wave < n_rows ? lo + per_wave : n_rows;
    int total = 0;
    for (long long r0 = lo; r0 < hi; r0 += 64) {
        const long long r = r0 + lane;
        total += __popcll(__ballot(r < hi && !covered[r]));
    }
    if (lane == 0) s_total[wave] = total;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int sum = s_total[0] + s_total[1] + s_total[2] + s_total[3];
        s_base = sum ? atomicAdd(count, sum) : 0;
    }
    __syncthreads();
    if (list == nullptr) return;
    int at = s_base;
    for (int w = 0; w < wave; ++w) at += s_total[w];
    for (long long r0 = lo; r0 < hi; r0 += 64) {
        const long long r = r0 + lane;
        const bool mine = r < hi && !covered[r];
        const unsigned long long votes = __ballot(mine);
        if (mine) list[at + __popcll(votes & ((1ull << lane) - 1ull))] = (int32_t)r;
        at += __popcll(votes);
    }
}

__global__ void fill_bytes_kernel(uint32_t* __restrict__ p, long long n_words, uint32_t value) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n_words;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = value;
}

double slices_and_subs(int slices, int lg_subs, double us) { return us + 0.5 * std::log2((double)slices) + 0.35 * lg_subs; }

}  // namespace

// ====================================================================================
struct lf_spmm_plan {
    int feat = 0, b_dtype = 0, num_parts = 0;
    int64_t num_rows = 0, num_cols = 0;
    int lpr = 0, ch = 0;
    int window = 0;                  // features of a window
    int slices = 1;                  // feature slices that the XCDs share out within a launch, of `feat` features (the last up to that)
    XcdParts parts;
    int windows = 1;                 // feature windows that a run covers
    int device = 0, num_cus = 0, grid = 0;
    struct Launch {
        int group_begin = 0, n_groups = 0, grid = 0;
        int dyn_lds = 0;             // bytes of dynamic LDS (balanced segment tiles, or to have fewer tiles on a CU)
        int merged_begin = 0, n_merged = 0, merged_grid = 0;   // row-group buckets of this partition
        int cell_begin = 0, n_cell_buckets = 0, cell_grid = 0; // buckets rewritten as cells
        long long tiles = 0;
        int heavy_begin = 0, n_heavy = 0;
        bool wide_rows = false;      // some rows have more than kWideFinalPartials partial rows
        int n_tiles[kInlineGroups] = {0};    // of the first groups
        bool stream_c = false;       // store C past the caches (when this is the run's last partition)
    };
    std::vector<Launch> launches;
    int coop_slots = kCoopSlots;        // source rows of more slab slots are reduced by whole workgroups
    bool resident = false;              // parts of B that the L2s hold: the kernels of that case
    bool stream_slabs = false;          // read the slabs non-temporally
    MergedBucket* d_merged = nullptr;   // row-group buckets, grouped by partition
    LfCellBucket* d_cells = nullptr;    // buckets rewritten as cells, grouped by partition
    std::vector<void*> owned;        // device allocations released by destroy
    std::vector<void*> temp;         // plan-time scratch, released when lf_spmm_create returns
    Group* d_groups = nullptr;
    HeavyRow* d_heavy = nullptr;        // [slices][n_heavy]
    float* d_partials = nullptr;        // [slices][partial rows][feat]
    int n_heavy = 0;
    long long slice_partials = 0;
    // d_partials and HeavyRow::done are written by every run; see order_behind_last_run
    hipEvent_t order_event = nullptr;    // made when a second stream appears
    hipStream_t last_stream = nullptr;
    std::thread::id last_thread;
    bool has_run = false;
    std::mutex order_mutex;              // from the wait for the run before to this run's last launch
    int64_t info[LF_SPMM_INFO_FIELDS] = {0};
};

namespace {

template <typename T> int dev_alloc(lf_spmm_plan* p, T** out, size_t count, bool temporary = false) {
    *out = nullptr;
    if (count == 0) return LF_OK;
    void* ptr = nullptr;
    LF_HIP(hipMalloc(&ptr, count * sizeof(T)));
    (temporary ? p->temp : p->owned).push_back(ptr);
    *out = (T*)ptr;
    return LF_OK;
}

int free_temporaries(lf_spmm_plan* p) {
    int rc = LF_OK;
    for (void* ptr : p->temp)
        if (hipFree(ptr) != hipSuccess) rc = LF_ERR_HIP;
    p->temp.clear();
    return rc;
}

using KernelFn = void (*)(LaunchArgs, XcdParts);
using FinalFn = void (*)(const HeavyRow*, int, LaunchArgs);

using RowGroupFn = void (*)(const MergedBucket*, int, LaunchArgs);

struct KernelSet {
    KernelFn tiles = nullptr;
    KernelFn tiles_resident = nullptr;   // the same where there is no such kernel
    KernelFn tiles_wide = nullptr;       // B past what 32-bit keys reach; its LDS holds the tiles of either
    FinalFn finalize_wide = nullptr;
    RowGroupFn rowgroup = nullptr;   // one 16-byte chunk per lane only
};

template <int LPR, int CH> void pick_kernels(int dtype, KernelSet* k) {
    if constexpr (CH == 1) {
        if (dtype == LF_DTYPE_BF16) k->rowgroup = spmm_rowgroup_kernel<LPR, bf16_t>;
        else k->rowgroup = spmm_rowgroup_kernel<LPR, float>;
    }
    if (dtype == LF_DTYPE_BF16) {
        k->tiles = spmm_partition_kernel<LPR, CH, bf16_t, false, false>;
        k->tiles_resident = spmm_partition_kernel<LPR, CH, bf16_t, has_resident_kernel(LPR, CH, true), false>;
        k->tiles_wide = spmm_partition_kernel<LPR, CH, bf16_t, has_resident_kernel(LPR, CH, true), true>;
        k->finalize_wide = spmm_finalize_wide_kernel<LPR, CH, bf16_t>;
    } else {
        k->tiles = spmm_partition_kernel<LPR, CH, float, false, false>;
        k->tiles_resident = spmm_partition_kernel<LPR, CH, float, has_resident_kernel(LPR, CH, false), false>;
        k->tiles_wide = spmm_partition_kernel<LPR, CH, float, has_resident_kernel(LPR, CH, false), true>;
        k->finalize_wide = spmm_finalize_wide_kernel<LPR, CH, float>;
    }
}

int select_kernels(int lpr, int ch, int dtype, KernelSet* k) {
    if (ch == 1) {
        switch (lpr) {
            case 8: pick_kernels<8, 1>(dtype, k); break;
            case 16: pick_kernels<16, 1>(dtype, k); break;
            case 32: pick_kernels<32, 1>(dtype, k); break;
            case 64: pick_kernels<64, 1>(dtype, k); break;
        }
    } else if (lpr == 64 && ch == 2) {
        pick_kernels<64, 2>(dtype, k);
    } else if (lpr == 64 && ch == 4) {
        pick_kernels<64, 4>(dtype, k);
    }
    LF_REQUIRE(k->tiles != nullptr, LF_ERR_UNSUPPORTED, "no kernel for %d lanes x %d chunks", lpr, ch);
    return LF_OK;
}

}  // namespace

extern "C" {

int lf_spmm_destroy(lf_spmm_plan* plan) {
    if (!plan) return LF_OK;
    int rc = free_temporaries(plan);
    if (plan->order_event && hipEventDestroy(plan->order_event) != hipSuccess) rc = LF_ERR_HIP;
    for (void* p : plan->owned)
        if (hipFree(p) != hipSuccess) rc = LF_ERR_HIP;
    delete plan;
    if (rc != LF_OK) return lf::fail(rc, "the runtime failed to release the plan's memory");
    return LF_OK;
}

int lf_spmm_create(lf_spmm_plan** out_plan, const lf_bucket_desc* h_buckets, int32_t num_buckets,
                   int32_t num_parts, int64_t num_rows, int64_t num_cols, int32_t feat_size,
                   int32_t b_dtype, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(out_plan, LF_ERR_INVALID, "out_plan is null");
    *out_plan = nullptr;
    LF_REQUIRE(num_buckets >= 0 && (num_buckets == 0 || h_buckets), LF_ERR_INVALID, "bucket list is null");
    LF_REQUIRE(num_parts >= 1, LF_ERR_INVALID, "num_parts must be >= 1");
    LF_REQUIRE(num_rows >= 0 && num_rows < (1ll << 31) && num_cols >= 1 && num_cols < (1ll << 31),
               LF_ERR_INVALID, "bad shape");
    LF_REQUIRE(b_dtype == LF_DTYPE_F32 || b_dtype == LF_DTYPE_BF16, LF_ERR_INVALID, "unknown B dtype %d", b_dtype);
    int lpr, ch;
    if (int rc = feature_shape(feat_size, b_dtype, &lpr, &ch)) return rc;
    for (int k = 0; k < num_buckets; ++k) {
        const lf_bucket_desc& b = h_buckets[k];
        LF_REQUIRE(lf::is_pow2(b.width) && b.width <= 1024, LF_ERR_INVALID, "bucket %d: width %d", k, b.width);
        LF_REQUIRE(b.part >= 0 && b.part < num_parts, LF_ERR_INVALID, "bucket %d: partition %d", k, b.part);
        LF_REQUIRE(b.num_ell_rows >= 0 && b.num_ell_rows < (1ll << 31), LF_ERR_INVALID, "bucket %d: row count", k);
        LF_REQUIRE(k == 0 || h_buckets[k - 1].part <= b.part, LF_ERR_INVALID, "buckets must be ordered by partition");
        if (b.num_ell_rows > 0) {
            LF_REQUIRE(b.d_rows && b.d_cols && b.d_vals, LF_ERR_INVALID, "bucket %d: null slab", k);
            LF_REQUIRE(((uintptr_t)b.d_cols % 16 == 0) && ((uintptr_t)b.d_vals % 16 == 0), LF_ERR_INVALID,
                       "bucket %d: slabs must be 16-byte aligned", k);
        }
    }

    lf_spmm_plan* plan = new lf_spmm_plan();
    plan->feat = plan->window = feat_size;
    plan->parts = xcd_parts(1, 1);
    plan->b_dtype = b_dtype;
    plan->num_parts = num_parts;
    plan->num_rows = num_rows;
    plan->num_cols = num_cols;
    plan->lpr = lpr;
    plan->ch = ch;
    auto bail = [&](int rc) {
        std::string keep = lf::last_error();
        (void)hipStreamSynchronize(s);       // nothing enqueued may outlive the scratch and the read-back buffers
        lf_spmm_destroy(plan);
        lf::last_error() = keep;
        return rc;
    };
#define LF_TRY(expr)                        \
    do {                                    \
        int _rc = (expr);                   \
        if (_rc != LF_OK) return bail(_rc); \
    } while (0)
#define LF_TRY_HIP(call)                                                                          \
    do {                                                                                          \
        hipError_t _e = (call);                                                                   \
        if (_e != hipSuccess)                                                                     \
            return bail(lf::fail(LF_ERR_HIP, "%s failed: %s", #call, hipGetErrorString(_e)));     \
    } while (0)

    hipDeviceProp_t prop;
    LF_TRY_HIP(hipGetDevice(&plan->device));
    LF_TRY_HIP(hipGetDeviceProperties(&prop, plan->device));
    plan->num_cus = prop.multiProcessorCount;

    // ---- meta: derive where missing; check the slabs; count the chunks of rows that take the
    // cooperative path; find the rows that nothing writes; sample the row-group candidates.  All of it
    // is enqueued together and read back with one copy and one synchronisation.
    std::vector<const int32_t*> meta((size_t)num_buckets, nullptr);
    struct ChunkCount { int chunks = 0, heavy = 0, partials = 0; };
    std::vector<ChunkCount> counts((size_t)num_buckets);
    // Chunk size of the rows that a whole workgroup reduces.  The smaller the matrix, the more a chunk's
    // chain of gathers is of the whole: short chunks; where there is work enough to hide it, longer ones
    // leave fewer partial rows.  By total slots because nothing else is known before the scan; the
    // steps lie where the sizes crossed on the first matrices measured (13K rows, 58K entries, N = 320 bf16,
    // chunks of 2048 / 1024 / 512: 47 / 29 / 19 us, 30K rows, 130K entries, N = 192 41 / 26 / 25, 149K
    // rows, 640K entries, N = 128 58 / 59 / 60) and are not all at the best place.  Power-law graphs of
    // 8K to 1.5M rows, rows cut at 13,000 or 1500, N = 64, 128 and bf16 320, every size tried:
    //   below 128K slots    512: the fastest, 2048 takes up to 2.6 times as long
    //   128K - 192K        1024: loses 24 - 32 % to 512 at 135K slots
    //   192K - 512K        1536: loses 22 - 51 % to 512 at 205K, 4 - 8 % to 1024 at 366K - 435K
    //   512K - 4M          2048: within 4 % of the fastest (9 % at 670K), 8192 takes up to 2.5 times as long
    //   from 4M on         8192: within 5 %; where long rows hold most entries it loses more (1M rows, 400
    //                            of 20,000 entries, N = 128: 1.18 ms, 1024 1.04; 500k x 2M, 150 of 30,000, N =
    //                            64: 0.311, 4096 0.286) or gains a little (the same, bf16 N = 256: 666 against 699)
    long long total_slots = 0;
    for (int k = 0; k < num_buckets; ++k) total_slots += h_buckets[k].num_ell_rows * h_buckets[k].width;
    const int chunk_slots = total_slots >= kLargeMatrixSlots ? kChunkSlotsLarge
                            : total_slots >= (512 << 10)     ? kChunkSlots
                            : total_slots >= (192 << 10)     ? kChunkSlots / 4 * 3
                            : total_slots >= (128 << 10)     ? kChunkSlots / 2
                                                             : kChunkSlots / 4;
    // Slabs of a large matrix are read past the caches' retention (2.45M-row graph 6.15 -> 6.09 ms,
    // 500k x 2M matrix 1.457 -> 1.443); those of a small one are worth keeping between products
    // (170k-row graph, 6 MB of slabs: 0.073 ms cached, 0.076 ms streamed).
    plan->stream_slabs = total_slots >= kLargeMatrixSlots;
    const char* env_dense = getenv("LF_DENSE_ROWS");       // "0": dense rows are chunked like the other long rows
    // (where the memory-side cache holds the partition's part of B anyway there is nothing to order)
    const long long cols_p = lf::ceil_div(num_cols, num_parts);
    const bool b_is_cached = cols_p * feat_size * (b_dtype == LF_DTYPE_BF16 ? 2 : 4) <= kDenseMinBBytes;
    const long long dense_min_slots = (env_dense && env_dense[0] == '0') || b_is_cached
                                          ? (1ll << 62)
                                          : std::max<long long>(kDenseRowMinSlots, cols_p / kDenseRowShare);

    // Scratch: the words that are read back (chunk counters and fill cursors of every bucket, sampling
    // counters, flags), then the coverage bytes - cleared by one launch - then the bucket table.
    const size_t nb_s = (size_t)num_buckets;
    long long scan_units = 0;                              // of kScanSlotsPerBlock slots or kScanRowsPerBlock rows
    auto units_of = [](const lf_bucket_desc& b) {
        return std::max<long long>(lf::ceil_div(b.num_ell_rows, (int64_t)kScanRowsPerBlock), lf::ceil_div(b.num_ell_rows * b.width, (int64_t)kScanSlotsPerBlock));
    };
    for (int k = 0; k < num_buckets; ++k) scan_units += units_of(h_buckets[k]);
    const long long units_per_block = std::max<long long>(1, lf::ceil_div(scan_units, (int64_t)kScanBlocksPerCu * plan->num_cus));
    auto scan_blocks_of = [&](int k) { return (int)lf::ceil_div(units_of(h_buckets[k]), units_per_block); };
    auto scan_lines_of = [&](int k) { return std::min(kScanLinesMost, std::max(1, scan_blocks_of(k) / kScanBlocksPerLine)); };
    int scan_lines = 0;
    for (int k = 0; k < num_buckets; ++k) scan_lines += scan_lines_of(k);
    const size_t o_counters = 0, o_cursors = o_counters + (size_t)scan_lines * kCounterLine * 4, o_flags = o_cursors + nb_s * 3 * kCounterLine * 4;
    const size_t o_zero = o_flags + 16, o_sample = o_zero + 16, back_bytes = o_sample + nb_s * 24;
    const size_t o_covered = (back_bytes + 255) / 256 * 256;
    const size_t o_table = (o_covered + (size_t)num_rows + 255) / 256 * 256;
    const size_t table_bytes = nb_s * (sizeof(PlanBucket) + 4);
    char* d_scratch = nullptr;
    LF_TRY(dev_alloc(plan, &d_scratch, o_table + std::max<size_t>(table_bytes, 16), true));
    int* d_counters = (int*)(d_scratch + o_counters);
    int* d_cursors = (int*)(d_scratch + o_cursors);
    int* d_flags = (int*)(d_scratch + o_flags);          // bad column, bad row, bad meta; derive_meta_kernel
    int* d_zero_count = (int*)(d_scratch + o_zero);      // rows to clear; listed so far
    unsigned long long* d_sample = (unsigned long long*)(d_scratch + o_sample);
    uint8_t* d_cov = (uint8_t*)(d_scratch + o_covered);
    lf::PinnedLoan back(back_bytes);
    lf::PinnedLoan table(table_bytes);
    if (!back.ok() || !table.ok()) return bail(lf::fail(LF_ERR_HIP, "out of host memory"));
    const int* h_counters = back.as<int>(o_counters);
    auto read_back = [&]() {
        hipError_t e = hipMemcpyAsync(back.as<char>(), d_scratch, back_bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        return e;
    };
    const char* env_groups = getenv("LF_ROW_GROUPS");
    std::vector<int> cand;                                 // buckets that may be rewritten as row groups or cells
    PlanBucket* h_table = table.as<PlanBucket>();
    int32_t* h_first = table.as<int32_t>(nb_s * sizeof(PlanBucket));
    const PlanBucket* d_table = (const PlanBucket*)(d_scratch + o_table);
    const int32_t* d_first = (const int32_t*)(d_scratch + o_table + nb_s * sizeof(PlanBucket));
    int scan_blocks = 0;
    std::vector<std::pair<int, int32_t*>> derived;         // buckets that come without meta words
    scan_lines = 0;
    for (int k = 0; k < num_buckets; ++k) {
        const lf_bucket_desc& b = h_buckets[k];
        const int log_w = lf::ilog2(b.width);
        if (b.num_ell_rows > 0 && !b.d_meta) {
            int32_t* m = nullptr;
            LF_TRY(dev_alloc(plan, &m, (size_t)b.num_ell_rows));
            derived.push_back({k, m});
            meta[k] = m;
        } else if (b.num_ell_rows > 0) {
            meta[k] = b.d_meta;
        }
        PlanBucket& t = h_table[k];
        t.rows = b.d_rows;
        t.meta = meta[k];
        t.cols = b.d_cols;
        t.n_rows = b.num_ell_rows;
        t.log_w = log_w;
        t.part = b.part;
        t.n_blocks = scan_blocks_of(k);
        t.first_line = scan_lines;
        t.n_lines = scan_lines_of(k);
        scan_lines += t.n_lines;
        t.n_first = t.n_blocks > 0 ? 1 : 0;
        t.span_stride = (int)std::max<long long>(kGroupRows, b.num_ell_rows / kSpanSamples);
        t.all_cols = (int)cols_p;
        t.sample_stride = 0;
        if (ch == 1 && !(env_groups && env_groups[0] == '0') && b.num_ell_rows >= kRowGroupMinRows && b.width >= kUnroll && b.width <= 64) {
            const long long n_groups = lf::ceil_div(b.num_ell_rows, kGroupRows);
            t.sample_stride = (int)std::max<long long>(1, n_groups / kRowGroupSample);
            t.n_first += (int)lf::ceil_div(lf::ceil_div(n_groups, (long long)t.sample_stride), (long long)kSampleGroups);
            cand.push_back(k);
        }
        h_first[k] = scan_blocks;
        scan_blocks += t.n_first + t.n_blocks;
    }
    LF_TRY_HIP(lf::move_words({h_table, d_scratch + o_table, table_bytes}, table.pinned(), d_scratch, o_table, {}, true, s));
    for (const auto& [k, m] : derived) {
        const lf_bucket_desc& b = h_buckets[k];
        int32_t *blk_first = nullptr, *blk_last = nullptr;
        const int n_blocks = (int)((b.num_ell_rows + 255) / 256);
        LF_TRY(dev_alloc(plan, &blk_first, (size_t)n_blocks, true));
        LF_TRY(dev_alloc(plan, &blk_last, (size_t)n_blocks, true));
        derive_heads_kernel<<<n_blocks, 256, 0, s>>>(b.d_rows, b.num_ell_rows, blk_first, blk_last);
        LF_TRY_HIP(hipGetLastError());
        derive_meta_kernel<<<n_blocks, 256, 0, s>>>(b.d_rows, b.d_vals, b.num_ell_rows, lf::ilog2(b.width), blk_first,
                                                    blk_last, n_blocks, m, d_flags);
        LF_TRY_HIP(hipGetLastError());
    }
    if (scan_blocks > 0) {
        plan_scan_kernel<<<scan_blocks, 256, 0, s>>>(d_table, d_first, num_buckets, num_rows, num_cols, chunk_slots,
                                                     dense_min_slots, d_counters, d_flags, d_cov, d_sample);
        LF_TRY_HIP(hipGetLastError());
    }
    const int rgrid = (int)std::min<int64_t>((num_rows + 255) / 256, 1024);
    if (num_rows > 0) {
        collect_uncovered_kernel<<<rgrid, 256, 0, s>>>(d_cov, num_rows, d_zero_count, nullptr);
        LF_TRY_HIP(hipGetLastError());
    }
    LF_TRY_HIP(read_back());
    {
        // nothing below (and no SpMM launch) may run on slabs that fail these checks: a column
        // or row index out of range would be an out-of-range gather or store
        const int* f = back.as<int>(o_flags);
        if (f[0]) return bail(lf::fail(LF_ERR_INVALID, "a bucket holds a column index outside [0, %lld)", (long long)num_cols));
        if (f[1]) return bail(lf::fail(LF_ERR_INVALID, "a bucket holds a row index outside [0, %lld)", (long long)num_rows));
        if (f[2]) return bail(lf::fail(LF_ERR_INVALID, "a bucket's meta array is inconsistent (valid slots outside 1..W, "
                                                        "or a segment that is incomplete or leaves the bucket)"));
        if (f[3]) return bail(lf::fail(LF_ERR_UNSUPPORTED, "a row is split over more than %d ELL rows", (1 << (31 - kMetaLenBits)) - 1));
    }
    std::vector<int> scan_sums(nb_s * kScanCounters, 0);
    for (int k = 0; k < num_buckets; ++k)
        for (int l = 0; l < h_table[k].n_lines; ++l)
            for (int i = 0; i < kScanCounters; ++i) {
                const int x = h_counters[(size_t)(h_table[k].first_line + l) * kCounterLine + i];
                int& sum = scan_sums[(size_t)kScanCounters * k + i];
                sum = i == kScanFound ? sum | x : sum + x;
            }
    auto scanned = [&](int k, int i) { return scan_sums[(size_t)kScanCounters * k + i]; };
    auto is_multi = [&](int k) { return (scanned(k, kScanFound) & 1) != 0; };       // rows split over several ELL rows
    auto has_dense = [&](int k) { return (scanned(k, kScanFound) & 2) != 0; };
    auto has_wide = [&](int k) { return (scanned(k, kScanFound) & 4) != 0; };
    const int n_zero = *back.as<int>(o_zero);
    // Candidates whose sample shows shared columns.  Neither the groups nor the cells know segments, they store every
    // ELL row as a row of C: a bucket that holds a split row stays with the tiles.
    std::vector<int> chosen;
    for (int k : cand) {
        const unsigned long long* c = back.as<unsigned long long>(o_sample) + 3 * k;
        if (!is_multi(k) && c[1] > 0 && c[0] * 100 <= c[1] * kRowGroupMaxPercent) chosen.push_back(k);
    }

    // Columns that neighbouring rows span, on average; 0: not known.
    double span = 0.0;
    {
        double slots = 0.0;
        for (int k = 0; k < num_buckets; ++k) {
            if (h_buckets[k].num_ell_rows == 0) continue;
            const double mine = (double)h_buckets[k].num_ell_rows * h_buckets[k].width;
            const double samples = (double)lf::ceil_div(h_buckets[k].num_ell_rows, (int64_t)h_table[k].span_stride);
            span += mine * scanned(k, kScanSpan) / samples / kSpanUnits * (double)cols_p;
            slots += mine;
        }
        if (slots > 0.0) span /= slots;
    }

    // ---- Feature slices; matrices whose kernels share gathers between rows read B through the L2s as it is.
    // A doubling of S costs 0.5 us in rows' starts and ends, one of the sub-waves to a wavefront 0.35, and sub-waves of fewer
    // lanes are more of them to share a long row's chunk, whose chain of gathers (0.11 us a step; it overlaps with other
    // work) sets the time of small power-law products.  3900 matrices of 2K to 2M rows, log-normal and power-law, N = 32 ..
    // 512, f32 and bf16, every S timed at the shape that was picked then: 0.927 of the time with S = 1 on average,
    // 1.6 % above the best S; 3 % of them more than 3 % slower than S = 1, 30 % at worst (products of 8 to 17
    // us with a B of 4 to 5 MB).  S that are no power of two, us, S = 1 or 2 before -> now: 32K rows of 32 entries, N = 96
    // 40.6 -> 29.6, 160 81 -> 43, 192 78 -> 50, 224 118 -> 58; 64K rows of 32, N = 224 247 -> 168, 352 393 -> 331; 64K rows of
    // 100, N = 288 in 16 partitions 825 -> 662; 132K rows of 300, N = 96 in 16 partitions 1025 -> 993, in 8 1003 -> 891.
    if (chosen.empty()) {
        const int vec = b_dtype == LF_DTYPE_BF16 ? 8 : 4;
        bool chains = false;                               // rows of several chunks
        for (int k = 0; k < num_buckets; ++k) chains = chains || scanned(k, 1) > 0;
        const double row_slots = (double)total_slots / ((double)num_parts * (double)std::max<int64_t>(num_rows, 1));
        auto tile_rows = [&](int lanes) { return tile_slots(lanes, false) / std::max(row_slots, 1.0); };
        const Slices slices = feature_slices(cols_p, total_slots / num_parts, feat_size, b_dtype, Neighbours{span, num_rows}, tile_rows,
                                             [&](int n, int width, int lg_subs, double us) {
            const int lanes = std::min(64, std::max(8, width / vec));
            const double steps = (double)chunk_slots * lanes / (kWG * kUnroll);
            return slices_and_subs(n, lg_subs, us) + (chains ? 0.11 * steps : 0.0);
        });
        plan->slices = slices.n;
        plan->parts = slices.parts;
        plan->feat = feat_size = slices.feat;
        LF_TRY(feature_shape(feat_size, b_dtype, &lpr, &ch));
        plan->lpr = lpr;
        plan->ch = ch;
    }
    const int sw = kWG / lpr;
    // Parts of B that an L2 (4 MB) about holds, and for float products rows that are mostly staged (those of
    // hundreds of slots per partition are streamed: 5774 rows of 368 in two partitions, N = 288
    // 145 -> 149 us).  A single float partition is not latency-bound enough (10K and 20K rows, 2.4 to 22 MB: -2 to
    // + 4 %); a bf16 one is up to 32 lanes per row (10K rows of 182, N = 128: 38.4 -> 36.5 us).  Where the line
    // loses: the same 5774 rows at N = 64 .. 128 would gain 18 - 23 % (53.6 -> 43.6 us), a bf16 B of 4.9 MB in
    // one partition 3 %; two partitions of 12K rows of 60 entries lose 1 - 7 % with it (N = 192: 42.7 -> 45.8).
    {
        const bool bf16 = b_dtype == LF_DTYPE_BF16;
        const long long part_bytes = lf::ceil_div(num_cols, (int64_t)num_parts) * feat_size * (bf16 ? 2 : 4);
        plan->resident = has_resident_kernel(lpr, ch, bf16) &&
                         part_bytes <= (num_parts > 1 ? 2 * kL2XcdBytes : bf16 && lpr <= 32 ? kL2XcdBytes : 0) &&
                         (bf16 || total_slots <= 96 * num_rows * num_parts);
    }
    // A sub-wave sums kUnroll slots of its row per round trip to B, so a row of kCoopSlots is a
    // chain of 32; where a product (all partitions together) holds few rows of more than 64 slots - a few
    // workgroups per CU - they set its length, and whole workgroups take them too: 56K-row power-law graph, bf16,
    // N = 128 33 -> 21 us with 64 instead of 256; 4K rows of 40 entries, N = 32 16 -> 6.5.  With some thousand
    // such rows the workgroups' set-up costs more than the chains (60K rows of 40, N = 64: 64 us with 256, 71
    // with 64).  In between, for small N with its many sub-waves to a workgroup, rows of more than 128 (30K
    // rows of 40, N = 32: 17 us, 64 20, 256 24).  Graphs of 4K to 500K rows, N = 32 .. 256, folded and not: the
    // length taken is within 6 % of the best, but where the first limit has just been passed (8K rows of 40,
    // 1255 of them above 64 slots: 4 - 48 %, 64 would be best up to N = 64, 128 above), up to 25 % for 15K
    // rows and N >= 128, which have no middle step, 11 % for such rows folded, and one folded 170K-row
    // power-law graph at N = 256 (64 taken: 174 us, 256 142).
    // It is rows that count, whatever the bucket: in a folded format they are segments of narrow ELL rows.
    // (Counted by the widths of the buckets, a folded format had none, and every such row became a chunk:
    // 2.45M-row graph, widths 1 .. 32, 302K chunks instead of 20K, N = 32 1.86 -> 1.60 ms now, N = 128 7.03 -> 6.84;
    // 132K rows of 300 entries, widths 1 .. 32 in four partitions, N = 32 0.998 -> 0.450.)
    long long over64 = 0, over128 = 0;
    for (int k = 0; k < num_buckets; ++k) {
        over64 += (long long)scanned(k, 3) + scanned(k, 4);
        over128 += scanned(k, 4);
    }
    if (over64 <= 4 * plan->num_cus) plan->coop_slots = 64;
    else if (lpr <= 16 && over128 <= 8 * plan->num_cus) plan->coop_slots = 128;
    // the rows that this adds are one chunk each
    static_assert(kCoopSlots >= 128 && kCoopSlots <= kChunkSlots / 4 && kCoopSlots <= kDenseChunkSlots && kCoopSlots < kDenseRowMinSlots);
    for (int k = 0; k < num_buckets; ++k) {
        counts[k].chunks = scanned(k, 0) + (plan->coop_slots <= 64 ? scanned(k, 3) : 0) + (plan->coop_slots <= 128 ? scanned(k, 4) : 0);
        counts[k].heavy = scanned(k, 1);
        counts[k].partials = scanned(k, 2);
    }
    // ---- chunk tables, heavy-row table (grouped by bucket, hence by partition) and partial rows
    std::vector<Chunk*> d_chunks((size_t)num_buckets, nullptr);
    std::vector<int> heavy_base((size_t)num_buckets + 1, 0), partial_base((size_t)num_buckets + 1, 0);
    std::vector<long long> chunk_base((size_t)num_buckets + 1, 0);
    for (int k = 0; k < num_buckets; ++k) {
        heavy_base[k + 1] = heavy_base[k] + counts[k].heavy;
        partial_base[k + 1] = partial_base[k] + counts[k].partials;
        chunk_base[k + 1] = chunk_base[k] + counts[k].chunks;
    }
    const int n_heavy_total = heavy_base[num_buckets];
    const int n_partials = partial_base[num_buckets];
    if (n_heavy_total > 0) {
        plan->n_heavy = n_heavy_total;
        plan->slice_partials = (long long)n_partials * feat_size;
        LF_TRY(dev_alloc(plan, &plan->d_heavy, (size_t)n_heavy_total * plan->slices));
        LF_TRY(dev_alloc(plan, &plan->d_partials, (size_t)plan->slice_partials * plan->slices));
    }
    Chunk* d_chunks_all = nullptr;
    LF_TRY(dev_alloc(plan, &d_chunks_all, (size_t)chunk_base[num_buckets]));
    ChunkBuckets chunk_buckets{};
    int chunk_blocks = 0;
    for (int k = 0; k < num_buckets; ++k) {
        const bool last = k + 1 == num_buckets;
        if (counts[k].chunks > 0) {
            const lf_bucket_desc& b = h_buckets[k];
            d_chunks[k] = d_chunks_all + chunk_base[k];
            chunk_buckets.of[chunk_buckets.n++] = ChunkBucket{b.d_rows, meta[k], b.d_cols, b.num_ell_rows, d_chunks[k], d_cursors + (size_t)3 * k * kCounterLine,
                                                              lf::ilog2(b.width), partial_base[k], heavy_base[k], chunk_blocks};
            chunk_blocks += (int)lf::ceil_div(b.num_ell_rows, (int64_t)kChunkRows);
        }
        if (chunk_buckets.n == kChunkBuckets || (last && chunk_buckets.n > 0)) {
            plan_chunks_kernel<<<chunk_blocks, kChunkThreads, 0, s>>>(chunk_buckets, plan->d_heavy, n_heavy_total, plan->slices, plan->coop_slots, chunk_slots, dense_min_slots);
            LF_TRY_HIP(hipGetLastError());
            chunk_buckets.n = chunk_blocks = 0;
        }
    }
    for (int k = 0; k < num_buckets; ++k) {
        if (!has_dense(k) || counts[k].chunks == 0) continue;
        // The chunks of dense rows go behind the others, in column order (ties: by row, so
        // the order is the same in every plan): some thousands of records, sorted on the host.
        std::vector<Chunk> h_chunks((size_t)counts[k].chunks);
        LF_TRY_HIP(hipMemcpyAsync(h_chunks.data(), d_chunks[k], h_chunks.size() * sizeof(Chunk), hipMemcpyDeviceToHost, s));
        LF_TRY_HIP(hipStreamSynchronize(s));
        const auto mid = std::stable_partition(h_chunks.begin(), h_chunks.end(),
                                               [](const Chunk& x) { return (x.n_slots & kChunkDenseBit) == 0; });
        std::sort(mid, h_chunks.end(), [](const Chunk& x, const Chunk& y) {
            if (x.first_col != y.first_col) return x.first_col < y.first_col;
            if (x.row != y.row) return x.row < y.row;
            return x.slot_begin < y.slot_begin;
        });
        for (auto it = mid; it != h_chunks.end(); ++it) it->n_slots &= ~kChunkDenseBit;
        LF_TRY_HIP(hipMemcpyAsync(d_chunks[k], h_chunks.data(), h_chunks.size() * sizeof(Chunk), hipMemcpyHostToDevice, s));
        LF_TRY_HIP(hipStreamSynchronize(s));
    }

    // ---- rows that partition 0 does not write are cleared by its launch
    int32_t* d_zero_rows = nullptr;
    if (n_zero > 0) {
        LF_TRY(dev_alloc(plan, &d_zero_rows, (size_t)n_zero));
        collect_uncovered_kernel<<<rgrid, 256, 0, s>>>(d_cov, num_rows, d_zero_count + 1, d_zero_rows);
        LF_TRY_HIP(hipGetLastError());
    }

    // ---- row groups: buckets whose consecutive rows share most of their columns
    std::vector<MergedBucket> merged;                      // in bucket (hence partition) order
    std::vector<int> merged_of((size_t)num_buckets, -1);
    std::vector<LfCellBucket> cells;                       // in bucket (hence partition) order
    std::vector<int> cell_of((size_t)num_buckets, -1);
    {
        std::vector<unsigned long long> h_rg(chosen.size() * 3, 0);   // three counters per bucket
        // merged lengths of all groups of the buckets `which`, and their totals
        auto count_pass = [&](const std::vector<int>& which, const std::vector<int32_t*>& m_arrays) -> int {
            unsigned long long* d_rg = nullptr;
            RowGroupCand* d_cands = nullptr;
            if (int rc = dev_alloc(plan, &d_rg, which.size() * 3, true)) return rc;
            if (int rc = dev_alloc(plan, &d_cands, which.size(), true)) return rc;
            std::vector<RowGroupCand> h_cands(which.size());
            long long most = 1;
            for (size_t i = 0; i < which.size(); ++i) {
                const lf_bucket_desc& b = h_buckets[which[i]];
                RowGroupCand& c = h_cands[i];
                c.cols = b.d_cols;
                c.meta = meta[which[i]];
                c.n_rows = b.num_ell_rows;
                c.n_groups = lf::ceil_div(b.num_ell_rows, kGroupRows);
                c.m_out = m_arrays[i];
                c.log_w = lf::ilog2(b.width);
                most = std::max<long long>(most, c.n_groups);
            }
            fill_bytes_kernel<<<1, 64, 0, s>>>((uint32_t*)d_rg, (long long)which.size() * 6, 0u);
            LF_HIP(hipGetLastError());
            LF_HIP(hipMemcpyAsync(d_cands, h_cands.data(), h_cands.size() * sizeof(RowGroupCand), hipMemcpyHostToDevice, s));
            rowgroup_count_kernel<<<dim3((unsigned)lf::ceil_div(most, 256), (unsigned)which.size()), 256, 0, s>>>(d_cands, d_rg);
            LF_HIP(hipGetLastError());
            LF_HIP(hipMemcpyAsync(h_rg.data(), d_rg, which.size() * 24, hipMemcpyDeviceToHost, s));
            LF_HIP(hipStreamSynchronize(s));               // also keeps h_cands alive until the copy is done
            return LF_OK;
        };
        if (!chosen.empty()) {
            // fp32 B, one 16-byte load per lane and 32 or 64 lanes per row of B (128 or 256
            // features per pass): the chosen buckets are rewritten as cells of rows that are
            // neighbours in up to three directions where that structure is found, else four
            // consecutive rows at a time (as are all other operand shapes: the cells measured
            // slower there).
            const bool cells_fit = (feat_size == 256 || feat_size == 128) && b_dtype == LF_DTYPE_F32;
            if (cells_fit && !(env_groups && env_groups[0] == '4')) {
                std::vector<int> rest;
                for (int k : chosen) {
                    LfCellBucket cb{};
                    bool ok = false;
                    LF_TRY(lf::cells_build(h_buckets[k], meta[k], num_rows, (int64_t)feat_size * (b_dtype == LF_DTYPE_BF16 ? 2 : 4), s,
                                           &plan->owned, &plan->temp, &cb, &ok));
                    if (ok) {
                        cell_of[k] = (int)cells.size();
                        cells.push_back(cb);
                    } else {
                        rest.push_back(k);
                    }
                }
                chosen.swap(rest);
            }
            if (!chosen.empty()) {
                std::vector<int32_t*> m_arrays(chosen.size(), nullptr);
                for (size_t i = 0; i < chosen.size(); ++i)
                    LF_TRY(dev_alloc(plan, &m_arrays[i], (size_t)lf::ceil_div(h_buckets[chosen[i]].num_ell_rows, kGroupRows), true));
                LF_TRY(count_pass(chosen, m_arrays));
                for (size_t i = 0; i < chosen.size(); ++i) {
                    const int k = chosen[i];
                    const lf_bucket_desc& b = h_buckets[k];
                    const unsigned long long entries = h_rg[3 * i], plain = h_rg[3 * i + 1], longest = h_rg[3 * i + 2];
                    if (entries == 0 || entries >= (1ull << 31) || longest > (unsigned long long)kMergedCap ||
                        entries * 100 > plain * kRowGroupMaxPercent)
                        continue;
                    MergedBucket mb{};
                    mb.n_rows = b.num_ell_rows;
                    mb.n_groups = lf::ceil_div(b.num_ell_rows, kGroupRows);
                    int32_t *goff = nullptr, *ecol = nullptr;
                    float4* eval = nullptr;
                    uint8_t* emask = nullptr;
                    LF_TRY(dev_alloc(plan, &goff, (size_t)mb.n_groups + 1));
                    LF_TRY(dev_alloc(plan, &ecol, (size_t)entries));
                    LF_TRY(dev_alloc(plan, &eval, (size_t)entries));
                    LF_TRY(dev_alloc(plan, &emask, (size_t)entries));
                    const int n_blocks = (int)lf::ceil_div(mb.n_groups, 1024);
                    int32_t* partial = nullptr;
                    LF_TRY(dev_alloc(plan, &partial, (size_t)n_blocks + 1, true));
                    LF_TRY_HIP(exclusive_scan_i32(m_arrays[i], mb.n_groups, partial, goff, s));
                    rowgroup_fill_kernel<<<(int)lf::ceil_div(mb.n_groups, 256), 256, 0, s>>>(
                        b.d_cols, b.d_vals, meta[k], b.num_ell_rows, lf::ilog2(b.width), mb.n_groups, goff, ecol, eval, emask);
                    LF_TRY_HIP(hipGetLastError());
                    // tile: one group per sub-wave (the tile is staged in rounds when its entries
                    // exceed the buffer), fewer when the bucket is small
                    const long long spread = lf::ceil_div(mb.n_groups, (long long)4 * plan->num_cus);
                    const long long per_tile = std::max<long long>(1, std::min<long long>(std::min(sw, kMergedTileGroups), spread));
                    mb.groups_per_tile = (int)per_tile;
                    mb.n_tiles = lf::ceil_div(mb.n_groups, per_tile);
                    mb.rows = b.d_rows;
                    mb.goff = goff;
                    mb.ecol = ecol;
                    mb.eval = eval;
                    mb.emask = emask;
                    merged_of[k] = (int)merged.size();
                    merged.push_back(mb);
                }
            }
        }
    }

    // ---- tile groups per launch: chunks first (longest), then buckets widest first, then clears
    std::vector<Group> groups;
    plan->launches.resize((size_t)num_parts);
    long long total_tiles = 0;
    for (int p = 0; p < num_parts; ++p) {
        lf_spmm_plan::Launch& L = plan->launches[p];
        L.group_begin = (int)groups.size();
        std::vector<int> mine;
        for (int k = 0; k < num_buckets; ++k)
            if (h_buckets[k].part == p && h_buckets[k].num_ell_rows > 0) mine.push_back(k);
        // Streaming stores leave the caches to B (2.45M-row graph, 33 entries per row: 6.23 -> 6.13
        // ms; short rows too: 392K x 680K, 4 entries per row, N = 64 88 -> 77 us, 1.47M x 2.73M, 8
        // per row, N = 96 910 -> 874), except where a lane's eight features of a bf16 product go out
        // as 16 of 32 bytes per instruction: the pieces then need the L2 to be put together, and a
        // launch of mostly short rows is made of stores as much as of gathers (500k x 2M matrix, most
        // rows 2-4 entries, 1.46 -> 1.53 ms; 1.19M x 1.83M, 3.6 per row, N = 128 296 -> 376 us).  A
        // C that the L2s hold is left there.
        long long rows_wide = 0, rows_all = 0;
        for (int k : mine) {
            rows_all += h_buckets[k].num_ell_rows;
            if (h_buckets[k].width >= kStreamMinWidth) rows_wide += h_buckets[k].num_ell_rows;
        }
        const bool c_fits_l2 = (long long)num_rows * plan->window * 4 <= kL2Bytes;
        L.stream_c = rows_wide * 2 >= rows_all || (b_dtype == LF_DTYPE_F32 && !c_fits_l2);
        for (int k : mine) L.wide_rows = L.wide_rows || has_wide(k);
        L.heavy_begin = mine.empty() ? 0 : heavy_base[mine.front()];
        L.n_heavy = mine.empty() ? 0 : heavy_base[mine.back() + 1] - L.heavy_begin;
        for (int k : mine) {
            if (counts[k].chunks == 0) continue;
            Group g{};
            g.type = kChunk;
            g.log_w = lf::ilog2(h_buckets[k].width);
            g.rows_per_tile = 1;
            g.cols = h_buckets[k].d_cols;
            g.vals = h_buckets[k].d_vals;
            g.n_items = g.n_tiles = counts[k].chunks;       // (those of dense rows last, in column order)
            g.chunks = d_chunks[k];
            groups.push_back(g);
        }
        std::sort(mine.begin(), mine.end(), [&](int x, int y) { return h_buckets[x].width > h_buckets[y].width; });
        for (int k : mine) {
            const lf_bucket_desc& b = h_buckets[k];
            if (b.width > plan->coop_slots) continue;           // every row of this bucket is a chunk
            if (merged_of[k] >= 0 || cell_of[k] >= 0) continue;   // served by the row-group or the cell kernel
            Group g{};
            g.log_w = lf::ilog2(b.width);
            const int fit = tile_slots(lpr, plan->resident && b_dtype == LF_DTYPE_F32) >> g.log_w;   // ELL rows whose slots fit the LDS tile
            const bool staged = fit >= sw;
            g.type = staged ? (is_multi(k) ? kEllSeg : kEll) : kSeg;
            g.rows_per_tile = staged ? std::min(kTileRows, fit) : lpr <= 16 ? kSegRows : kSegRows / 2;
            if (!staged) g.balanced = std::max(0, g.log_w - kLgTeamSlots);
            if (staged) {
                // a small bucket is cut into more, shorter tiles so that it still spreads over
                // the CUs: at least one pass of every sub-wave (8 rows at a time in the
                // narrow-bucket code), aiming at four tiles per CU
                const int unit = sw * (b.width < kUnroll ? kUnroll / b.width : 1);
                const long long want = lf::ceil_div(b.num_ell_rows, (long long)4 * plan->num_cus);
                const long long rows = std::max<long long>(unit, lf::ceil_div(want, (long long)unit) * unit);
                g.rows_per_tile = (int)std::min<long long>(g.rows_per_tile, rows);
            }
            if (g.type == kEllSeg) {
                const long long part_bytes = (long long)g.rows_per_tile * feat_size * 4;
                if (part_bytes <= kPartBytesMax) {
                    g.balanced = 1;
                    L.dyn_lds = std::max(L.dyn_lds, (int)part_bytes);
                }
            }
            g.n_items = b.num_ell_rows;
            g.n_tiles = lf::ceil_div(g.n_items, g.rows_per_tile);
            g.rows = b.d_rows;
            g.meta = meta[k];
            g.cols = b.d_cols;
            g.vals = b.d_vals;
            groups.push_back(g);
        }
        if (p == 0 && n_zero > 0) {
            Group g{};
            g.type = kZero;
            // (4096 rows, 1500 of them empty, N = 128: tiles of 1024 32 us, so 6)
            g.rows_per_tile = (int)std::min<long long>(1024, std::max<long long>(4 * sw, lf::ceil_div(n_zero, (long long)4 * plan->num_cus)));
            g.n_items = n_zero;
            g.n_tiles = lf::ceil_div(g.n_items, g.rows_per_tile);
            g.rows = d_zero_rows;
            groups.push_back(g);
        }
        L.n_groups = (int)groups.size() - L.group_begin;
        L.merged_begin = -1;
        for (int k : mine) {
            if (merged_of[k] < 0) continue;
            if (L.merged_begin < 0 || merged_of[k] < L.merged_begin) L.merged_begin = merged_of[k];
            ++L.n_merged;                                  // a partition's buckets are consecutive in `merged`
        }
        L.cell_begin = -1;
        for (int k : mine) {
            if (cell_of[k] < 0) continue;
            if (L.cell_begin < 0 || cell_of[k] < L.cell_begin) L.cell_begin = cell_of[k];
            ++L.n_cell_buckets;                            // a partition's buckets are consecutive in `cells`
        }
        if (L.n_cell_buckets > 0) {
            long long longest_c = 0;
            for (int x = 0; x < kXcds; ++x) {
                long long len = 0;
                for (int i = L.cell_begin; i < L.cell_begin + L.n_cell_buckets; ++i)
                    len += cells[i].n_tiles * (x + 1) / kXcds - cells[i].n_tiles * x / kXcds;
                longest_c = std::max(longest_c, len);
            }
            if (longest_c * kXcds >= (1ll << 31)) return bail(lf::fail(LF_ERR_UNSUPPORTED, "too many cell tiles"));
            L.cell_grid = (int)(longest_c * kXcds);
        }
        if (L.n_merged > 0) {
            long long longest_m = 0;
            for (int x = 0; x < kXcds; ++x) {
                long long len = 0;
                for (int i = L.merged_begin; i < L.merged_begin + L.n_merged; ++i)
                    len += merged[i].n_tiles * (x + 1) / kXcds - merged[i].n_tiles * x / kXcds;
                longest_m = std::max(longest_m, len);
            }
            if (longest_m * kXcds >= (1ll << 31)) return bail(lf::fail(LF_ERR_UNSUPPORTED, "too many row-group tiles"));
            L.merged_grid = (int)(longest_m * kXcds);
        }
        // grid: 8 x the longest per-XCD tile list
        long long longest = 0;
        for (int x = 0; x < kXcds; ++x) {
            long long len = 0;
            for (int gi = L.group_begin; gi < (int)groups.size(); ++gi) len += part_tiles(plan->parts, x, groups[gi].n_tiles);
            longest = std::max(longest, len);
        }
        for (int gi = L.group_begin; gi < (int)groups.size(); ++gi) {
            L.tiles += groups[gi].n_tiles;
            if (gi - L.group_begin < kInlineGroups) L.n_tiles[gi - L.group_begin] = (int)groups[gi].n_tiles;   // (checked below)
        }
        if (longest * kXcds >= (1ll << 31))
            return bail(lf::fail(LF_ERR_UNSUPPORTED, "partition %d needs too many tiles", p));
        L.grid = (int)(longest * kXcds);
        total_tiles += L.tiles;
    }
    // the tables go up together, in one allocation
    const size_t o_merged = (groups.size() * sizeof(Group) + 255) / 256 * 256;
    const size_t o_cells = (o_merged + merged.size() * sizeof(MergedBucket) + 255) / 256 * 256;
    const size_t tables_bytes = o_cells + cells.size() * sizeof(LfCellBucket);
    lf::PinnedLoan h_tables(tables_bytes);
    if (!h_tables.ok()) return bail(lf::fail(LF_ERR_HIP, "out of host memory"));
    lf::Words up;                              // sent with the read-back below
    if (tables_bytes > 0) {
        char* d_tables = nullptr;
        LF_TRY(dev_alloc(plan, &d_tables, tables_bytes));
        auto put = [&](size_t at, const void* src, size_t bytes) {
            if (bytes) std::memcpy(h_tables.as<char>(at), src, bytes);
        };
        put(0, groups.data(), groups.size() * sizeof(Group));
        put(o_merged, merged.data(), merged.size() * sizeof(MergedBucket));
        put(o_cells, cells.data(), cells.size() * sizeof(LfCellBucket));
        up = lf::Words{h_tables.as<char>(), d_tables, tables_bytes};
        plan->d_groups = (Group*)d_tables;
        plan->d_merged = (MergedBucket*)(d_tables + o_merged);
        plan->d_cells = (LfCellBucket*)(d_tables + o_cells);
    }

    KernelSet ks;
    LF_TRY(select_kernels(lpr, ch, b_dtype, &ks));
    hipFuncAttributes attributes;
    LF_TRY_HIP(hipFuncGetAttributes(&attributes, reinterpret_cast<const void*>(plan->resident ? ks.tiles_resident : ks.tiles)));
    // Four tiles to a CU, where five and more would push each other's rows of B out of the caches for nothing:
    // rows of near columns, and all features of them (7-point stencils, us, without a limit, 5 or 6 to a CU / 4 / 3: 226K points,
    // N = 64 32.5 / 29.8 / 32.7; 200K, N = 128 54.0 / 50.7 / 53.6; 729K, N = 64 112 / 107.4 / 105.8), and parts of B of which the
    // L2s hold little (522K rows of 15, bf16 N = 256 648 / 637 / 615; 170K power-law rows, N = 64 38.0 / 35.7 / 36.9; 630
    // matrices with slices of more than 64 MB: 0.994 and 0.993 of the time on average, 1.02 and 1.05 at most; below 16 MB 1.03 to
    // 1.1 and 1.1 to 1.3).  Little more than four to a CU would run in two rounds so (70K points, N = 96: 17.8, 19.7).
    const double slice_bytes = (double)cols_p * feat_size * (b_dtype == LF_DTYPE_BF16 ? 2 : 4);
    if (chosen.empty() && ((is_near(span, cols_p) && plan->slices == 1) || slice_bytes > kFarSliceBytes)) {
        const int most = kLdsOfCu / (kNearGroupsPerCu + 1) + kLdsStep;     // one more would not fit
        for (auto& L : plan->launches)
            if (2 * L.grid > 11 * plan->num_cus) L.dyn_lds = std::max(L.dyn_lds, most - (int)attributes.sharedSizeBytes);
    }
    int dyn_lds = 0;
    plan->grid = 0;
    for (const auto& L : plan->launches) {
        plan->grid = std::max(plan->grid, L.grid);
        dyn_lds = std::max(dyn_lds, L.dyn_lds);
    }

    plan->info[0] = total_tiles;
    plan->info[1] = plan->grid;
    plan->info[2] = num_parts;
    plan->info[3] = (int64_t)attributes.sharedSizeBytes + dyn_lds;
    plan->info[4] = n_heavy_total;
    plan->info[5] = n_partials;
    plan->info[6] = n_zero;
    plan->info[7] = (int64_t)(merged.size() + cells.size());
    plan->info[8] = (int64_t)cells.size();
    LF_TRY_HIP(lf::move_words(up, h_tables.pinned(), nullptr, 0, {d_scratch + o_cursors, back.as<char>(o_cursors), o_flags - o_cursors}, back.pinned(), s));
    LF_TRY_HIP(hipStreamSynchronize(s));     // the tables are complete: the plan may run on any stream
    for (int k = 0; k < num_buckets; ++k) {  // the filling pass must have taken the counted ranges
        const int* c = back.as<int>(o_cursors) + (size_t)3 * k * kCounterLine;
        if (counts[k].chunks > 0 && (c[0] != counts[k].chunks || c[kCounterLine] != counts[k].heavy || c[2 * kCounterLine] != counts[k].partials))
            return bail(lf::fail(LF_ERR_INVALID, "bucket %d changed while the plan was being built", k));
    }
    if (free_temporaries(plan) != LF_OK) return bail(lf::fail(LF_ERR_HIP, "hipFree failed on plan-time scratch"));
    *out_plan = plan;
    return LF_OK;
#undef LF_TRY
#undef LF_TRY_HIP
}

// Launch shape.  A launch (one partition, one window) takes the price of its best feature slices (feature_slices), longer
// where the memory-side cache holds so little of the part of B that HBM is what its misses wait for, by rows of B of which a
// window reads 256 bytes or less, and before a later partition, whose additions to C keep its stores in the caches; 7 TB/s
// for the stores of C and the additions; and 7 us for a launch more.
// Before, lf_model_spmm_ms stood here: fitted to kernels without slices it kept to few partitions.  1120 matrices of 2K to
// 2M rows, log-normal and power-law, N = 32 .. 512, f32 and bf16, up to 32 partitions and 4 windows each timed: its pick was
// 5.2 % above the fastest on average and more than 5 % above for 22 % of them.  This one's is 0.8 % above on these and 725 more, to
// all of which its constants are fitted, and 0.6 % on 302 that were timed afterwards, 15 % at worst.  2.5 % of the matrices take 3 %
// longer than with the pick before, at worst 26 %; the best takes half the time (73K rows of 125, N = 352: 1.63 -> 0.85 ms).
int lf_model_shape_ms(const int64_t* h_stats, int32_t num_parts, int32_t n_windows, int64_t num_rows, int64_t num_cols,
                      int32_t feat_size, int32_t b_dtype, double* h_ms) {
    constexpr double kMallBytes = 140e6, kFabricOverHbm = 1.3, kBytesOfC = 7.0e6, kNextUs = 7.0, kFirstUs = 4.0;
    constexpr double kNarrow = 0.02, kNotLast = 0.05;
    LF_REQUIRE(h_stats && h_ms, LF_ERR_INVALID, "null argument");
    LF_REQUIRE(num_parts >= 1 && n_windows >= 1 && num_rows >= 0 && num_cols >= 1, LF_ERR_INVALID, "bad shape");
    LF_REQUIRE(feat_size >= 1 && feat_size % n_windows == 0, LF_ERR_INVALID, "feat_size %d is not a multiple of %d windows",
               feat_size, n_windows);
    LF_REQUIRE(b_dtype == LF_DTYPE_F32 || b_dtype == LF_DTYPE_BF16, LF_ERR_INVALID, "unknown B dtype %d", b_dtype);
    double nnz = 0, added = 0;                             // of all partitions; rows that a later one adds to
    for (int p = 0; p < num_parts; ++p) {
        for (int k = 0; k < LF_MAX_CLASSES; ++k) {
            const int64_t* st = h_stats + ((size_t)p * LF_MAX_CLASSES + k) * LF_STATS_FIELDS;
            nnz += (double)st[1];
            if (p > 0) added += (double)st[2];
        }
    }
    const int feat = feat_size / n_windows;
    const double g = (double)feat * (b_dtype == LF_DTYPE_BF16 ? 2.0 : 4.0), cols = std::ceil((double)num_cols / num_parts);
    const Slices best = feature_slices((int64_t)cols, (int64_t)(nnz / num_parts), feat, b_dtype,
                                       Neighbours{}, [](int) { return 0.0; },
                                       [](int n, int, int lg_subs, double us) { return slices_and_subs(n, lg_subs, us); });
    const double lg = std::log2((double)n_windows);
    const double narrow = 1.0 + (g < 512.0 ? kNarrow * lg * lg : 0.0);
    const double cached = std::min(1.0, kMallBytes / (cols * g)) * (1.0 - std::min(1.0, (double)num_cols / std::max(nnz, 1.0)));
    const double hbm = std::max(1.0, (1.0 - cached) * kFabricOverHbm);
    const double window_us = (num_parts + kNotLast * (num_parts - 1)) * best.us * narrow * hbm + num_parts * kNextUs +
                             ((double)num_rows * feat * 4.0 + added * feat * 8.0) / kBytesOfC;
    *h_ms = 1e-3 * (window_us * n_windows + kFirstUs - kNextUs);
    return LF_OK;
}

int lf_spmm_info(const lf_spmm_plan* plan, int64_t* h_info) {
    LF_REQUIRE(plan && h_info, LF_ERR_INVALID, "null argument");
    std::memcpy(h_info, plan->info, sizeof(plan->info));
    return LF_OK;
}

// The runs of a plan with rows of several chunks share the plan's partial rows and counters: two that
// overlap mix their sums, and can push a counter past the row's last chunk, whose row of C is then never
// written.  A run on another stream than the one before therefore waits for it.  The event is
// recorded here, on the stream of the run before, and not behind every run: that would add 1.3 to 3 us to
// each (170K-row graph, N = 128: 71.0 -> 72.3 us without a system-scope fence, 73.9 with one), this adds
// nothing to runs on one stream.  Where the runtime refuses the stream of the run before (it has been
// destroyed), or that was another thread's hipStreamPerThread, the device is waited for.  While either
// stream is being recorded into a graph no event may cross over: those runs are ordered by the caller.
// To be called with order_mutex held: a run that another thread has ordered but not launched yet is not
// behind the event.
static int order_behind_last_run(lf_spmm_plan* plan, hipStream_t s) {
    if (!plan->d_heavy) return LF_OK;
    const bool same = plan->has_run && plan->last_stream == s;
    const auto is_own = [](hipStream_t x) { return x == hipStreamPerThread; };
    if (same && (!is_own(s) || plan->last_thread == std::this_thread::get_id())) return LF_OK;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    LF_HIP(hipStreamIsCapturing(s, &capture));
    if (capture != hipStreamCaptureStatusNone) return LF_OK;
    if (plan->has_run) {
        const hipStream_t before = plan->last_stream;
        bool reachable = !is_own(before) || plan->last_thread == std::this_thread::get_id();
        if (reachable) {
            reachable = hipStreamIsCapturing(before, &capture) == hipSuccess;
            if (reachable && capture != hipStreamCaptureStatusNone) return LF_OK;
            if (!plan->order_event) LF_HIP(hipEventCreateWithFlags(&plan->order_event, hipEventDisableTiming));
            reachable = reachable && hipEventRecord(plan->order_event, before) == hipSuccess;
        }
        if (reachable) {
            LF_HIP(hipStreamWaitEvent(s, plan->order_event, 0));
        } else {
            (void)hipGetLastError();
            LF_HIP(hipDeviceSynchronize());
        }
    }
    plan->last_stream = s;
    plan->last_thread = std::this_thread::get_id();
    plan->has_run = true;
    return LF_OK;
}

int lf_spmm_run(lf_spmm_plan* plan, const void* d_B, float* d_C, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(plan, LF_ERR_INVALID, "plan is null");
    if (plan->num_rows == 0) return LF_OK;
    LF_REQUIRE(d_B && d_C, LF_ERR_INVALID, "B or C is null");
    LF_REQUIRE((uintptr_t)d_B % 16 == 0 && (uintptr_t)d_C % 16 == 0, LF_ERR_INVALID, "B and C must be 16-byte aligned");
    KernelSet ks;
    if (int rc = select_kernels(plan->lpr, plan->ch, plan->b_dtype, &ks)) return rc;
    std::unique_lock<std::mutex> order(plan->order_mutex, std::defer_lock);
    if (plan->d_heavy) order.lock();
    if (int rc = order_behind_last_run(plan, s)) return rc;
    // One pass per feature window (all partitions inside), each on its own columns of B and C.
    const size_t b_elem = plan->b_dtype == LF_DTYPE_BF16 ? 2 : 4;
    const int window = plan->window, ld = window * plan->windows;
    const unsigned long long b_bytes = (unsigned long long)plan->num_cols * ld * b_elem;
    const KernelFn tiles = b_bytes > kPastB ? ks.tiles_wide : plan->resident ? ks.tiles_resident : ks.tiles;
    for (int w = 0; w < plan->windows; ++w) {
        for (int p = 0; p < plan->num_parts; ++p) {
            const lf_spmm_plan::Launch& L = plan->launches[p];
            if (L.n_groups == 0 && L.n_merged == 0 && L.n_cell_buckets == 0) continue;
            LaunchArgs a{};
            a.groups = plan->d_groups + L.group_begin;
            a.n_groups = L.n_groups;
            a.accumulate = (p > 0 ? kAccumulateC : 0) | (p + 1 == plan->num_parts && L.stream_c ? kStreamC : 0) |
                           (plan->stream_slabs ? kStreamSlabs : 0);
            a.feat = plan->feat;
            a.all_feat = window;
            a.ldb = a.ldc = ld;
            a.B = (const char*)d_B + (size_t)w * window * b_elem;
            a.C = d_C + (size_t)w * window;
            a.b_bytes = b_bytes - (size_t)w * window * b_elem;
            a.slice_heavy = plan->n_heavy;
            a.slice_partials = plan->slice_partials;
            a.partials = plan->d_partials;
            a.heavy = plan->d_heavy;
            a.coop_slots = plan->coop_slots;
            std::memcpy(a.n_tiles, L.n_tiles, sizeof(a.n_tiles));
            if (L.grid > 0) {
                tiles<<<L.grid, kWG, L.dyn_lds, s>>>(a, plan->parts);
                LF_HIP(hipGetLastError());
            }
            if (L.n_merged > 0) {
                ks.rowgroup<<<L.merged_grid, kWG, 0, s>>>(plan->d_merged + L.merged_begin, L.n_merged, a);
                LF_HIP(hipGetLastError());
            }
            if (L.n_cell_buckets > 0) {
                if (int rc = lf::cells_launch(plan->d_cells + L.cell_begin, L.n_cell_buckets, L.cell_grid, plan->b_dtype,
                                              a.B, a.C, a.feat, a.ldb, a.ldc, a.accumulate, s))
                    return rc;
            }
            if (L.wide_rows) {
                ks.finalize_wide<<<dim3((unsigned)L.n_heavy, (unsigned)plan->slices), kWG, 0, s>>>(plan->d_heavy + L.heavy_begin, L.n_heavy, a);
                LF_HIP(hipGetLastError());
            }
        }
    }
    return LF_OK;
}

int lf_spmm_set_windows(lf_spmm_plan* plan, int32_t n_windows) {
    LF_REQUIRE(plan, LF_ERR_INVALID, "plan is null");
    LF_REQUIRE(n_windows >= 1 && (int64_t)n_windows * plan->window <= (1 << 20), LF_ERR_INVALID,
               "bad number of feature windows (%d)", n_windows);
    plan->windows = n_windows;
    return LF_OK;
}

int lf_spmm_time_ms(lf_spmm_plan* plan, const void* d_B, float* d_C, int32_t warmup, int32_t repeat,
                    void* d_flush, size_t flush_bytes, float* h_ms, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(plan && h_ms, LF_ERR_INVALID, "null argument");
    LF_REQUIRE(warmup >= 0 && repeat >= 1, LF_ERR_INVALID, "bad warmup/repeat");
    for (int i = 0; i < warmup; ++i)
        if (int rc = lf_spmm_run(plan, d_B, d_C, stream)) return rc;
    hipEvent_t t0, t1;
    LF_HIP(hipEventCreate(&t0));
    if (hipError_t e = hipEventCreate(&t1)) {
        (void)hipEventDestroy(t0);
        return lf::fail(LF_ERR_HIP, "hipEventCreate failed: %s", hipGetErrorString(e));
    }
    int rc = LF_OK;
    for (int i = 0; i < repeat && rc == LF_OK; ++i) {
        if (d_flush && flush_bytes >= 4) {
            const long long words = (long long)(flush_bytes / 4);
            fill_bytes_kernel<<<(int)std::min<long long>((words + 255) / 256, 8192), 256, 0, s>>>((uint32_t*)d_flush, words, (uint32_t)i);
        }
        hipError_t e = hipEventRecord(t0, s);
        if (e == hipSuccess) {
            rc = lf_spmm_run(plan, d_B, d_C, stream);
            if (rc != LF_OK) break;
            e = hipEventRecord(t1, s);
        }
        if (e == hipSuccess) e = hipEventSynchronize(t1);
        if (e == hipSuccess) e = hipEventElapsedTime(&h_ms[i], t0, t1);
        if (e != hipSuccess) rc = lf::fail(LF_ERR_HIP, "timing failed: %s", hipGetErrorString(e));
    }
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    return rc;
}

}  // extern "C"
