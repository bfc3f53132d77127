// Device-side building blocks shared by the SpMM kernels of liblfhip.so: launch arguments,
// dense-operand access (one 16-byte load per lane), per-lane accumulators, row stores.
// Everything lives in an anonymous namespace: each translation unit gets its own copy.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <utility>

#include "lf_internal.h"

namespace {

constexpr int kWG = 256;            // threads per workgroup (4 wavefronts)
#ifndef LF_TILE_SLOTS_PER_SUBWAVE
#define LF_TILE_SLOTS_PER_SUBWAVE 64
#endif
#ifndef LF_UNROLL
#define LF_UNROLL 8
#endif
#ifndef LF_TILE_MIN
#define LF_TILE_MIN 512
#endif
// (col, val) pairs staged in LDS per tile: a fixed amount of work per sub-wave, so narrow
// feature sizes (many sub-waves per workgroup) get larger tiles.  N = 128 -> 512 slots.
// `resident`: see spmm_partition_kernel.
constexpr int tile_slots(int lpr, bool resident) {
    const int n = LF_TILE_SLOTS_PER_SUBWAVE * (kWG / lpr);
    const int least = resident && lpr >= 32 ? 2 * LF_TILE_MIN : LF_TILE_MIN;
    return n < least ? least : n;
}
constexpr int kTileRows = 512;      // ELL rows per tile at most (<= tile_slots)
#ifndef LF_COOP_SLOTS
#define LF_COOP_SLOTS 256
#endif
#ifndef LF_CHUNK_SLOTS
#define LF_CHUNK_SLOTS 2048
#endif
constexpr int kCoopSlots = LF_COOP_SLOTS;    // a source row with more slab slots is reduced by a whole workgroup
constexpr int kChunkSlots = LF_CHUNK_SLOTS;  // ... in chunks of this many slots, or of a quarter to three quarters of it in
                                             // small matrices (lf_spmm_create); a chunk may end inside an ELL row
constexpr int kChunkSlotsLarge = 8192;       // ... or this many, in a matrix of at least kLargeMatrixSlots slots
constexpr long long kLargeMatrixSlots = 4ll << 20;
// Dense rows: a row holding at least 1/kDenseRowShare of its partition's columns.  Several of
// them read much the same rows of B, so they are cut into shorter chunks that are walked in
// column order: the chunks in flight then cover a window of B that the memory-side cache holds,
// and a row of B is fetched from HBM once for all of them.  500k x 2M matrix with 50 rows of
// 100,000 entries, bf16 N = 512, ms per product by chunk size (whole workgroup per chunk):
// 8192 unordered 1.46; ordered 8192 1.53, 4096 1.43, 2048 1.39, 1024 1.295, 512 1.30, 256 1.40,
// 128 1.70; a sub-wave per chunk: 512 1.40, 256 1.37, 128 1.34, 64 1.44.  (Short enough for
// the window to fit an XCD's L2 they would need far fewer chunks in flight than fill the GPU.)
constexpr int kDenseRowShare = 32;
constexpr int kDenseRowMinSlots = 4096;
constexpr long long kDenseMinBBytes = 128ll << 20;   // ... in a partition whose part of B is larger than this
constexpr int kDenseChunkSlots = 1024;
constexpr int kWideFinalPartials = 64;       // rows with more partial rows are added up by a kernel of their own
constexpr int kLgXcds = 3, kXcds = 1 << kLgXcds;
constexpr int kPartBytesMax = 16384;   // LDS for per-ELL-row sums of a balanced segment tile at most
constexpr int kUnroll = LF_UNROLL;  // B-row gathers in flight per sub-wave
static_assert(kUnroll == 8, "a batch of 8 or 16 entries is gathered eight at a time");
constexpr uint32_t kMetaLenMask = 0x7FFu;
constexpr int kMetaLenBits = 11;

enum GroupType : int { kEll = 0, kSeg = 1, kZero = 2, kChunk = 3, kEllSeg = 4 };

constexpr int kChunkDenseBit = 1 << 30;       // in Chunk::n_slots while the plan is built: a piece of a dense row

struct Chunk {
    long long slot_begin;   // first slot, relative to the bucket's slab
    int n_slots;
    int partial;            // index of the partial row this chunk produces; < 0: the chunk is the
                            // whole source row and goes straight to C
    int row;                // source row
    int first_col;          // column of the chunk's first slot (chunks of dense rows are ordered by it)
    int heavy;              // entry of the row in the heavy-row table (rows of several chunks)
    int pad_;
};

struct HeavyRow {
    int row;
    int partial_begin;
    int n_partials;
    int done;               // chunks of the row that have left their partial row in the present launch
};

struct Group {
    int type;
    int log_w;
    int rows_per_tile;
    int balanced;                 // kEllSeg: per-ELL-row sums through LDS (needs rows_per_tile * N floats); kSeg: log2 of the
                                  // sub-waves to a row, or more than a wavefront has
    long long n_items;            // ELL rows / rows to clear / chunks
    long long n_tiles;
    const int32_t* rows;          // kEll, kSeg: source rows; kZero: rows to clear
    const int32_t* meta;
    const int32_t* cols;
    const float* vals;
    const Chunk* chunks;          // kChunk
};

constexpr int kInlineGroups = 16;      // a row of lanes

struct LaunchArgs {
    const Group* groups;
    int n_groups;
    int accumulate;               // bit 0: C += result instead of C = result; bit 1 (kStreamC): no later
                                  // launch of the run reads these rows of C again; bit 2 (kStreamSlabs):
                                  // the slabs are too large to be worth caching
    int feat;                     // N: features computed by the launch, or of a slice of them (the last may have fewer)
    int all_feat;                 // features computed by the launch
    int ldb, ldc;                 // row strides of B and C in elements (N, or more for a feature window)
    int coop_slots;               // source rows of more slab slots are reduced by whole workgroups
    const void* B;
    float* C;
    unsigned long long b_bytes;   // from B to the end of the matrix
    int slice_heavy;              // heavy rows and partial values of a slice
    long long slice_partials;
    float* partials;
    HeavyRow* heavy;
    int n_tiles[kInlineGroups];   // of the first groups (0: none): a workgroup finds its group without reading the others
};

// ------------------------------------------------------------------------------------
// Dense-operand access: VEC features per lane as one 16-byte load.
template <typename BT> struct Dense;

template <> struct Dense<float> {
    static constexpr int kVec = 4;
    static constexpr int kElemBytes = 4;
    using Raw = float4;
    __device__ static __forceinline__ void unpack(const Raw& v, float (&x)[4]) {
        x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    }
};

struct bf16_t { uint16_t bits; };

template <> struct Dense<bf16_t> {
    static constexpr int kVec = 8;
    static constexpr int kElemBytes = 2;
    using Raw = uint4;
    __device__ static __forceinline__ void unpack(const Raw& v, float (&x)[8]) {
        x[0] = __uint_as_float(v.x << 16); x[1] = __uint_as_float(v.x & 0xFFFF0000u);
        x[2] = __uint_as_float(v.y << 16); x[3] = __uint_as_float(v.y & 0xFFFF0000u);
        x[4] = __uint_as_float(v.z << 16); x[5] = __uint_as_float(v.z & 0xFFFF0000u);
        x[6] = __uint_as_float(v.w << 16); x[7] = __uint_as_float(v.w & 0xFFFF0000u);
    }
};

// Accumulator of one sub-wave lane: CH chunks of VEC features.
template <int CH, int VEC> struct Acc {
    float v[CH][VEC];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
            for (int i = 0; i < VEC; ++i) v[c][i] = 0.f;
    }
};

// Position of a lane inside the feature dimension.
template <int LPR, int CH, int VEC> struct Lane {
    int sl;                 // lane inside the sub-wave
    int feat;               // N: features this launch computes
    int ldb, ldc;           // elements between consecutive rows of B and of C (>= N)
    int f[CH];              // first feature of each chunk (clamped to 0 when outside N)
    bool on[CH];
    __device__ __forceinline__ Lane(int sl_, int feat_, int ldb_, int ldc_)
        : sl(sl_), feat(feat_), ldb(ldb_), ldc(ldc_) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int f0 = (c * LPR + sl_) * VEC;
            on[c] = f0 < feat_;
            f[c] = on[c] ? f0 : 0;
        }
    }
};

// Where lane `ln` finds its 16 bytes of row `col` of B: the lane's own place in row 0 plus
// col * (bytes between rows) - one 32 x 32 -> 64-bit multiply-add per gather.  (Indexing in
// elements, with the row stride as a signed int, cost two 64-bit multiply-adds, two moves and a
// shift-add per gather: more vector instructions than the four FMAs the gather feeds.)
template <typename BT, int LPR, int CH>
__device__ __forceinline__ const char* dense_row(const void* B, const Lane<LPR, CH, Dense<BT>::kVec>& ln, int c,
                                                 int col) {
    const char* lane0 = reinterpret_cast<const char*>(B) + (size_t)ln.f[c] * Dense<BT>::kElemBytes;
    const uint32_t pitch = (uint32_t)ln.ldb * (uint32_t)Dense<BT>::kElemBytes;      // ldb <= 2^20
    return lane0 + (uint64_t)(uint32_t)col * pitch;
}

template <typename BT, int LPR, int CH>
__device__ __forceinline__ typename Dense<BT>::Raw load_dense(const void* B, const Lane<LPR, CH, Dense<BT>::kVec>& ln,
                                                              int c, int col) {
    return *reinterpret_cast<const typename Dense<BT>::Raw*>(dense_row<BT>(B, ln, c, col));
}

// acc += v * x.  The 16 bytes stay as they were loaded until here: unpacked while further loads are in
// flight, bf16 would hold twice the registers.
template <typename BT>
__device__ __forceinline__ void fma_dense(float v, const typename Dense<BT>::Raw& raw, float (&acc)[Dense<BT>::kVec]) {
    float x[Dense<BT>::kVec];
    Dense<BT>::unpack(raw, x);
#pragma unroll
    for (int i = 0; i < Dense<BT>::kVec; ++i) acc[i] = fmaf(v, x[i], acc[i]);
}

// Rows of B by key: the bytes to the row, from one 32-bit multiplication where the column is read.  Gathers go
// through a buffer resource over B, so a key and the lane's own offset are one addition away from the load, and
// kNone, past the end of B, reads zeros without touching memory: no traffic for padding, and nothing for an
// infinite element of B to turn into NaN.  Keys have 32 bits: where B is larger (WIDE) they are columns, and loads
// are predicated and take a 64-bit multiply-add each.
constexpr uint32_t kPastB = 0xFFFE0000u;       // (a lane's own offset is below 2^17)
typedef unsigned int lf_u32x4 __attribute__((ext_vector_type(4)));

template <int LPR, int CH, typename BT, bool WIDE> struct RowsOfB {
    using Raw = typename Dense<BT>::Raw;
    static constexpr int VEC = Dense<BT>::kVec;
    static constexpr uint32_t kNone = WIDE ? 0xFFFFFFFFu : kPastB;
    const char* base;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t pitch;                            // bytes between rows
    uint32_t lane_at[CH];                      // the lane's own bytes in a row
    // `bytes`: from B to the end of the matrix
    __device__ __forceinline__ RowsOfB(const void* B, unsigned long long bytes, const Lane<LPR, CH, VEC>& ln) {
        base = reinterpret_cast<const char*>(B);
        pitch = (uint32_t)ln.ldb * (uint32_t)Dense<BT>::kElemBytes;
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(B), 0, WIDE ? 0 : (int)(uint32_t)bytes, 0x00027000);
#pragma unroll
        for (int c = 0; c < CH; ++c) lane_at[c] = (uint32_t)(ln.f[c] * Dense<BT>::kElemBytes);
    }
    __device__ __forceinline__ uint32_t key(int col) const { return WIDE ? (uint32_t)col : (uint32_t)col * pitch; }
    __device__ __forceinline__ Raw load(int c, uint32_t k) const {
        Raw x{};
        if constexpr (WIDE) {
            if (k != kNone) x = *reinterpret_cast<const Raw*>(base + lane_at[c] + (uint64_t)k * pitch);
        } else {
            const lf_u32x4 raw = __builtin_amdgcn_raw_buffer_load_b128(rsrc, k + lane_at[c], 0, 0);
            __builtin_memcpy(&x, &raw, sizeof(Raw));
        }
        return x;
    }
};

template <int U, int LPR, int CH, typename BT, bool WIDE>
__device__ __forceinline__ void gather_fma(const RowsOfB<LPR, CH, BT, WIDE>& b, const uint32_t (&key)[U], const float (&val)[U],
                                           Acc<CH, Dense<BT>::kVec>& acc) {
    typename Dense<BT>::Raw x[U][CH];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < CH; ++c) x[u][c] = b.load(c, key[u]);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < CH; ++c) fma_dense<BT>(val[u], x[u][c], acc.v[c]);
}

// Entry I of a sub-wave's batch, from the lane that holds it, by a DPP broadcast: an operand modifier of the
// instruction that uses it, where a shuffle is an LDS instruction and its latency.  Lanes of other sub-waves need
// not be active.
template <int LPR, int I> __device__ __forceinline__ int batch_entry(int x) {
    constexpr int kRowBroadcast = 0x150;       // row_newbcast: a lane of each row of 16 to that row
    if constexpr (LPR >= 16) {
        return __builtin_amdgcn_update_dpp(0, x, kRowBroadcast + I, 0xF, 0xF, true);
    } else {                                   // two sub-waves to a row of 16 lanes
        const int first = __builtin_amdgcn_update_dpp(0, x, kRowBroadcast + I, 0xF, 0x3, false);
        return __builtin_amdgcn_update_dpp(first, x, kRowBroadcast + 8 + I, 0xF, 0xC, false);
    }
}

// Teams of 2^lg sub-waves of a wavefront, each on a stretch of entries (column, value) in memory: entry e goes to
// sub-wave e mod 2^lg.
template <int LPR, int CH, typename BT, bool WIDE> struct Teams {
    static constexpr int VEC = Dense<BT>::kVec;
    static constexpr int kLgSubs = LPR == 64 ? 0 : LPR == 32 ? 1 : LPR == 16 ? 2 : 3;       // log2 of a wavefront's sub-waves
    static constexpr int kBatch = LPR < 16 ? LPR : 16;      // entries of a sub-wave fetched at a time
    const RowsOfB<LPR, CH, BT, WIDE>& b;
    const int lg, sub;                         // size of the team; sub-wave in its team
    const int slot;                            // entry of a batch that the lane fetches (in every 16 lanes again)

    __device__ __forceinline__ Teams(const RowsOfB<LPR, CH, BT, WIDE>& b_, int lg_)
        : b(b_), lg(lg_), sub((int)(threadIdx.x & 63) / LPR & ((1 << lg_) - 1)), slot((int)threadIdx.x % kBatch) {}

    // The lane's entry of the batch at `base` of the `len` entries from `lo` on; no column (-1) past the end.  What is
    // made of the column waits for it: not here, where the entry is requested ahead.
    template <typename Pos>
    __device__ __forceinline__ void fetch(const int32_t* __restrict__ cols, const float* __restrict__ vals, Pos lo, int len,
                                          int base, int& col, float& val) const {
        const int e = base + (slot << lg) + sub;
        col = -1;
        val = 0.f;
        if (e < len) {
            col = cols[lo + e];
            val = vals ? vals[lo + e] : 1.f;
        }
    }

    // Entries FIRST + I... of the batch, summed on their own first: a stretch of n entries is then a chain of 8 + n / 8
    // additions instead of n, and a longer stretch to a sub-wave costs no precision.  Relative error (2-norm) against 64
    // bits of log-normal rows, one chain / this: 16000 x 128, N = 32 1.2e-7 / 8.8e-8; 8000 x 300, N = 256 2.0e-7 /
    // 1.4e-7; CSR, 1.2M x 9, N = 64 7.2e-8 / 5.8e-8.  The addition per eight entries: plans 0.999 of the time, CSR 1.003,
    // with bf16 0.96 to 1.04 (up to 8 registers more).
    template <int FIRST, size_t... I>
    __device__ __forceinline__ void gather(uint32_t key, float val, Acc<CH, VEC>& acc, std::index_sequence<I...>) const {
        typename Dense<BT>::Raw x[kUnroll][CH];
        auto load = [&](int u, uint32_t k) {
#pragma unroll
            for (int c = 0; c < CH; ++c) x[u][c] = b.load(c, k);
        };
        (load(I, (uint32_t)batch_entry<LPR, FIRST + I>((int)key)), ...);
        Acc<CH, VEC> batch;
        batch.clear();
        auto add = [&](int u, float v) {
#pragma unroll
            for (int c = 0; c < CH; ++c) fma_dense<BT>(v, x[u][c], batch.v[c]);
        };
        (add(I, __int_as_float(batch_entry<LPR, FIRST + I>(__float_as_int(val)))), ...);
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc.v[c][i] += batch.v[c][i];
    }

    // Adds the team's `len` entries (column, value; no values: ones) from `lo` on.  `most`: at least len, the same in a
    // team; teams with different ones diverge, and before combine() all of the wavefront have to be here again.
    template <typename Pos>
    __device__ __forceinline__ void sum(const int32_t* __restrict__ cols, const float* __restrict__ vals, Pos lo, int len,
                                        int most, Acc<CH, VEC>& acc) const {
        constexpr auto kEight = std::make_index_sequence<kUnroll>();
        int col;
        float val;
        fetch(cols, vals, lo, len, 0, col, val);
        for (int base = 0; base < most;) {
            const uint32_t k = col >= 0 ? b.key(col) : b.kNone;
            const float v = val;
            const int left = most - base;
            base += kBatch << lg;
            if (base < most) fetch(cols, vals, lo, len, base, col, val);   // ahead: a latency of its own
            gather<0>(k, v, acc, kEight);
            if constexpr (kBatch > kUnroll)
                if (left > (kUnroll << lg)) gather<kUnroll>(k, v, acc, kEight);
        }
    }

    // The team's sums, added pairwise: every lane of the team holds them afterwards.
    __device__ __forceinline__ void combine(Acc<CH, VEC>& acc) const {
        for (int d = LPR; d < (LPR << lg); d <<= 1)
#pragma unroll
            for (int c = 0; c < CH; ++c)
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc.v[c][i] += __shfl_xor(acc.v[c][i], d);
    }
};

// flags: LaunchArgs::accumulate.  Rows that nothing reads again in this run are stored
// non-temporally where that leaves the caches to B (lf_spmm_create decides); rows that a later column partition adds to stay cached
// (170k-row graph, two partitions: streaming them costs 7 %).
constexpr int kAccumulateC = 1, kStreamC = 2, kStreamSlabs = 4;
constexpr int kStreamMinWidth = 16;      // a launch of mostly wide rows: at least half of its ELL rows are this wide
constexpr long long kL2XcdBytes = 4ll << 20;
constexpr long long kL2Bytes = 8 * kL2XcdBytes;   // of the eight XCDs together
typedef float lf_f32x4 __attribute__((ext_vector_type(4)));

// 16 bytes to global memory, streamed or not by a run-time flag.  The streaming store goes
// through a global-memory pointer made from the address as an integer: with the same pointer in
// both branches the compiler folds the two stores into one ordinary store.
__device__ __forceinline__ void store_f32x4(float* dst, lf_f32x4 o, bool stream) {
    if (stream)
        __builtin_nontemporal_store(o, reinterpret_cast<lf_f32x4 __attribute__((address_space(1)))*>(reinterpret_cast<uintptr_t>(dst)));
    else
        *reinterpret_cast<lf_f32x4*>(dst) = o;
}

// 16 bytes of a slab, streamed or not (same construction as store_f32x4)
typedef int lf_i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ lf_i32x4 load_i32x4(const void* src, bool stream) {
    if (stream)
        return __builtin_nontemporal_load(
            reinterpret_cast<const lf_i32x4 __attribute__((address_space(1)))*>(reinterpret_cast<uintptr_t>(src)));
    return *reinterpret_cast<const lf_i32x4*>(src);
}

template <int LPR, int CH, int VEC>
__device__ __forceinline__ void store_row(float* C, int row, const Lane<LPR, CH, VEC>& ln,
                                          const Acc<CH, VEC>& acc, int flags) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        if (!ln.on[c]) continue;
        float* dst = C + (size_t)row * ln.ldc + ln.f[c];
#pragma unroll
        for (int i = 0; i < VEC; i += 4) {
            lf_f32x4 o = {acc.v[c][i], acc.v[c][i + 1], acc.v[c][i + 2], acc.v[c][i + 3]};
            if (flags & kAccumulateC) o += *reinterpret_cast<const lf_f32x4*>(dst + i);
            store_f32x4(dst + i, o, flags & kStreamC);
        }
    }
}

// goff[g] = exclusive prefix of m[g], goff[n_groups] = total, in three small launches:
// sums of blocks of 1024 groups, their exclusive scan by one workgroup (in place, total
// appended), then the scan inside every block.
__device__ __forceinline__ int block_inclusive_scan_1024(int x, int* s_wave) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int incl = x;
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(incl, d);
        if (lane >= d) incl += y;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    for (int w = 0; w < wave; ++w) incl += s_wave[w];
    __syncthreads();
    return incl;
}

__global__ void __launch_bounds__(1024)
scan_blocksum_kernel(const int32_t* __restrict__ m, long long n_groups, int32_t* __restrict__ partial) {
    __shared__ int s_wave[16];
    const long long i = (long long)blockIdx.x * 1024 + threadIdx.x;
    const int incl = block_inclusive_scan_1024(i < n_groups ? m[i] : 0, s_wave);
    if (threadIdx.x == 1023) partial[blockIdx.x] = incl;
}

__global__ void __launch_bounds__(1024)
scan_partials_kernel(int32_t* __restrict__ partial, int n_blocks) {
    __shared__ int s_wave[16];
    __shared__ int s_carry;
    if (threadIdx.x == 0) s_carry = 0;
    __syncthreads();
    for (int base = 0; base < n_blocks; base += 1024) {
        const int i = base + threadIdx.x;
        const int x = i < n_blocks ? partial[i] : 0;
        const int incl = block_inclusive_scan_1024(x, s_wave);
        const int carry = s_carry;
        if (i < n_blocks) partial[i] = carry + incl - x;
        __syncthreads();
        if (threadIdx.x == 1023) s_carry = carry + incl;
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[n_blocks] = s_carry;
}

__global__ void __launch_bounds__(1024)
scan_blocks_kernel(const int32_t* __restrict__ m, long long n_groups, const int32_t* __restrict__ partial,
                     int n_blocks, int32_t* __restrict__ goff) {
    __shared__ int s_wave[16];
    const long long i = (long long)blockIdx.x * 1024 + threadIdx.x;
    const int x = i < n_groups ? m[i] : 0;
    const int incl = block_inclusive_scan_1024(x, s_wave);
    if (i < n_groups) goff[i] = partial[blockIdx.x] + incl - x;
    if (blockIdx.x == 0 && threadIdx.x == 0) goff[n_groups] = partial[n_blocks];
}

// off[i] = exclusive prefix of m[i] for i < n, off[n] = total, enqueued on `s`.  `partial`
// needs ceil(n / 1024) + 1 ints.
inline hipError_t exclusive_scan_i32(const int32_t* m, long long n, int32_t* partial, int32_t* off, hipStream_t s) {
    const int n_blocks = (int)((n + 1023) / 1024);
    if (n_blocks == 0) return hipSuccess;
    scan_blocksum_kernel<<<n_blocks, 1024, 0, s>>>(m, n, partial);
    scan_partials_kernel<<<1, 1024, 0, s>>>(partial, n_blocks);
    scan_blocks_kernel<<<n_blocks, 1024, 0, s>>>(m, n, partial, n_blocks, off);
    return hipGetLastError();
}

// Lanes per row of B and 16-byte chunks per lane of a product of `feat` features.
inline int feature_shape(int feat, int dtype, int* lpr, int* ch) {
    const int vec = dtype == LF_DTYPE_BF16 ? 8 : 4;
    LF_REQUIRE(feat >= 32 && feat % 32 == 0, LF_ERR_UNSUPPORTED,
               "feat_size must be a positive multiple of 32 (got %d)", feat);
    LF_REQUIRE(feat <= 1024, LF_ERR_UNSUPPORTED, "feat_size above 1024 is not supported (got %d)", feat);
    const int lanes = feat / vec;
    int l = 8;
    while (l < lanes && l < 64) l <<= 1;
    int c = (lanes + l - 1) / l;
    if (c == 3) c = 4;
    LF_REQUIRE(c == 1 || c == 2 || c == 4, LF_ERR_UNSUPPORTED, "feat_size %d is not supported", feat);
    *lpr = l;
    *ch = c;
    return LF_OK;
}

// Feature slices: the features are cut into S slices, and the work - all tiles for the first slice, then all tiles for the
// second, .. - into a part for each XCD, so that an L2 has 1 / S of B to hold at a time instead of all of it, at the
// price of reading the entries S times.  A slice is 128 bytes or a multiple: a gather of 64 moves the line all the same
// (a table in the L2s is gathered from at 28 TB/s by rows of 128 bytes and more, 15.5 by rows of 64).  The last slice may
// be narrower, the parts weigh the same.
// A part is [from, upto) of the tiles of `slice` and [0, next) of those of the slice behind it, in 2^-32 of the tiles: an
// XCD has T / 8 of T pieces of 128 bytes, and only the last slice can be shorter than that.
struct XcdPart {
    int slice;
    unsigned from, upto, next;
};
constexpr unsigned kAllTiles = 0xFFFFFFFFu;

template <typename Int> __host__ __device__ inline Int tiles_before(Int n_tiles, unsigned fraction) {
    return fraction == kAllTiles ? n_tiles : (Int)((unsigned long long)n_tiles * fraction >> 32);
}

// What the parts are made from, in eighths of half a piece: a slice's length, the last slice's, and an XCD's.  (A table of
// the parts among a launch's arguments was 0.4 us of each product.)
struct XcdParts {
    int slice_len, last_len, weight, n_slices;
    int lg_near;                                           // log2 of the XCDs that take the same tiles at a time
    unsigned slice_inverse, last_inverse;                  // 2^32 / length, rounded up
};

// The part of XCD x.  XCDs that take the same tiles at a time are neighbours (32K rows of 32 entries, N = 192, S = 2: 78 us;
// with slice 0 on XCDs 0 .. 3 83).
__host__ __device__ __forceinline__ XcdPart xcd_part(const XcdParts& p, int x) {
    if (p.n_slices == 1) return XcdPart{0, (unsigned)x << 29, x + 1 == kXcds ? kAllTiles : (unsigned)(x + 1) << 29, 0u};
    const int place = ((x & ((1 << p.lg_near) - 1)) << (kLgXcds - p.lg_near)) + (x >> p.lg_near);
    const int begin = place * p.weight, end = begin + p.weight;
    const int slice = (int)((unsigned long long)begin * p.slice_inverse >> 32);
    auto fraction = [&](int at, int of_slice) {
        const bool last = of_slice == p.n_slices - 1;
        const int done = at - of_slice * p.slice_len;
        return done >= (last ? p.last_len : p.slice_len) ? kAllTiles : done * (last ? p.last_inverse : p.slice_inverse);
    };
    return XcdPart{slice, fraction(begin, slice), fraction(end, slice), end > (slice + 1) * p.slice_len ? fraction(end, slice + 1) : 0u};
}

struct Slices {
    int n = 1, feat = 0;                                   // slices, and features of each but the last
    double us = 0.0;                                       // their price
    XcdParts parts;
};

// Workgroups that a list of `n_tiles` tiles takes on an XCD
inline long long part_tiles(const XcdParts& parts, int x, long long n_tiles) {
    const XcdPart p = xcd_part(parts, x);
    return tiles_before(n_tiles, p.upto) - tiles_before(n_tiles, p.from) + tiles_before(n_tiles, p.next);
}

inline int slice_step(int dtype) { return dtype == LF_DTYPE_BF16 ? 64 : 32; }

// `pieces` of 128 bytes in slices of `wide` of them.  A row of a narrower last slice takes as many lanes as of the others,
// so it counts as half way between its width and theirs: by its width alone the XCD that has it was 2.3 times behind in
// products whose gathers hit (N = 224 in slices of 96, 96 and 32).
inline int slices_weight(int pieces, int wide) {
    const int n = (int)lf::ceil_div(pieces, wide);
    return 2 * wide * (n - 1) + wide + (pieces - (n - 1) * wide);        // in half pieces
}

inline XcdParts xcd_parts(int pieces, int wide) {
    XcdParts p;
    p.n_slices = (int)lf::ceil_div(pieces, wide);
    p.lg_near = lf::ilog2(p.n_slices);
    p.weight = slices_weight(pieces, wide);
    p.slice_len = 2 * kXcds * wide;
    p.last_len = kXcds * p.weight - (p.n_slices - 1) * p.slice_len;
    p.slice_inverse = (unsigned)lf::ceil_div(1ll << 32, p.slice_len);
    p.last_inverse = (unsigned)lf::ceil_div(1ll << 32, p.last_len);
    return p;
}

// The S of the least price in us: gathers that hit an L2 at 27 TB/s of what their lanes could take (5 % less for every
// doubling of the sub-waves to a wavefront, which wait for the longest of their rows), those that miss and the entries at
// 7.15 (misses of 128 bytes 6 % slower), the share that hits from the slice's size against 4.3 MB and from how often an XCD
// uses a row of B (the first use misses, unless it meets that of another XCD: 0.4 of one); `adjust` adds what else S and the
// sub-waves, 2^lg_subs to a wavefront, change.
// For the price that is compared with that of other partitions (us), a slice of about an L2 misses more: 20 % at 5 MB, and 10 %
// less for a doubling of the sub-waves (233K rows of 490, N = 128, slices of 3.7 MB in 8 partitions 3.81 ms, of 1.9 in 16
// 3.12).  Of slices chosen by that price, 5 % would be more than 3 % slower than S = 1, instead of 3 %.
//
// In a matrix whose neighbouring rows have near columns (stencils, bands; `span`: the columns of four such rows, on
// average) an XCD does not use all of B at a time but what its rows in flight span, four workgroups of
// group_rows(lanes of a row) each to a CU, and hardly a row of B that another XCD uses.  Stencils of 4K to 800K points, us,
// slices as if for a random matrix -> now, without any: plans, 27-point, 62K points, N = 416 124 -> 107, 107; 7-point, 21K, N = 256
// 14.9 -> 13.3, 13.3; 7-point, 160K, N = 352 138 -> 98, 138; CSR, 27-point, 62K, N = 416 167 -> 121, 121; 7-point, 21K, N = 256
// 18.1 -> 10.7, 10.7.  301 plans and 320 CSR products, every S timed: 4.5 and 7.1 % above the best S before,
// now 1.2 and 1.0; of 250 more plans 4 % are more than 3 % slower than with the slices of a random matrix, 17 % at worst.
constexpr int kNearGroupsPerCu = 4, kCusOfXcd = 32;
// Near columns hit an L1 as well as an L2, and by 15 TB/s; what does not fit is lost faster, by the 1.4th power.
constexpr double kNearHitRate = 15e6, kNearPower = 1.4;
struct Neighbours {
    double span = 0.0;                                     // 0: not known
    int64_t num_rows = 0;
    double per_sub = 0.0;                                  // what hits take longer for a doubling of the sub-waves to a wavefront
};
inline bool is_near(double span, int64_t num_cols) { return span > 0.0 && 2.0 * span < (double)num_cols; }

template <typename GroupRows, typename Adjust>
inline Slices feature_slices(int64_t num_cols, int64_t entries, int feat, int dtype, Neighbours neighbours, GroupRows group_rows, Adjust adjust) {
    constexpr double kL2 = 4.3e6, kHitRate = 27e6, kMissRate = 7.15e6, kMiss128 = 1.06, kFirstUse = 0.4, kPerSub = 0.05;
    constexpr double kSoftL2 = 5.0e6, kSoftPerSub = 0.1;
    const int elem = dtype == LF_DTYPE_BF16 ? 2 : 4, step = slice_step(dtype);
    const double gathered = (double)entries * feat * elem;
    const bool whole = feat % step == 0;
    const int pieces = whole ? feat / step : 1;
    int best = pieces;
    double least = 0.0;
    Slices slices;
    for (int n = 1; n <= kXcds && entries > 0; ++n) {
        const int wide = lf::ceil_div(pieces, n), width = whole ? wide * step : feat;
        if (lf::ceil_div(pieces, wide) != n) continue;
        int lpr, ch;
        if (width % 32 != 0 || feature_shape(width, dtype, &lpr, &ch) != LF_OK) {     // no product, but a price
            lpr = 64;
            ch = (int)lf::ceil_div((int64_t)width * elem, 1024);
        }
        // an XCD's part of a slice's tiles, of its bytes and of the lanes' (the last slice's, the longest, against the average)
        const double weight = slices_weight(pieces, wide);
        const double share = weight / (2.0 * wide * kXcds);
        const double bytes = gathered * weight / (2.0 * pieces);
        const double lanes = 16.0 * (double)entries * lpr * ch * weight / (wide + pieces - (n - 1) * wide);
        const bool near = is_near(neighbours.span, num_cols);
        double uses = (double)entries / (double)num_cols * share, in_use = (double)num_cols;
        if (near) {
            const double rows = (double)neighbours.num_rows;
            const double in_flight = std::min(rows * share, kNearGroupsPerCu * kCusOfXcd * group_rows(lpr));
            in_use = std::min(in_use, neighbours.span + in_flight * (double)num_cols / rows);
            uses = (double)entries / (double)num_cols;
        }
        const double again = std::max(0.0, 1.0 - kFirstUse / uses), slice_bytes = in_use * width * elem;
        const int lg_subs = lf::ilog2(64 / lpr);
        auto priced = [&](double hit, double per_sub) {
            return adjust(n, width, lg_subs, lanes * hit / (near ? kNearHitRate : kHitRate) * (1.0 + per_sub * lg_subs) +
                                             bytes * (1.0 - hit) / kMissRate * (width == step ? kMiss128 : 1.0) +
                                             8.0 * (double)entries * n / kMissRate);
        };
        const double held_share = std::min(1.0, kL2 / slice_bytes);
        const double price = near ? priced(std::pow(held_share, kNearPower) * again, neighbours.per_sub) : priced(held_share * again, kPerSub);
        if (n == 1 || price < least) {
            const double held = kSoftL2 / slice_bytes;
            least = price;
            slices.us = priced(held / std::cbrt(1.0 + held * held * held) * again, kSoftPerSub);
            best = wide;
            slices.n = n;
        }
    }
    slices.feat = whole ? best * step : feat;
    slices.parts = xcd_parts(pieces, best);
    return slices;
}

}  // namespace
