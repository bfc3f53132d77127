// CSR product without a plan for gfx950:  C[rows][N] = A_csr . B[cols][N], fp32 accumulate.
//
// The counterpart of bench_naive's kernel (playground_pipline/format_algos.py:1689-1755), which gives a row to a
// thread block.  Here the entries of a row are spread over a *team* of sub-waves: a sub-wave of LPR lanes covers a
// row of B with one 16-byte load per lane, and the 64 / LPR sub-waves of a wavefront work on one row, two rows, ...
// or a row each, as the lengths of the workgroup's rows ask for.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <utility>

#include "lf_internal.h"
#include "lf_spmm_device.h"

namespace {

// A workgroup of four wavefronts takes kCsrRowsFew or kCsrRowsMany consecutive rows; a wavefront takes the next rows
// off a counter whenever it is through with its own, so that nothing waits for the longest row but itself.
constexpr int kCsrThreads = 256;
constexpr int kCsrRowsFew = 8, kCsrRowsMany = 16;
constexpr long long kCsrManyRows = 24576;
constexpr int kCsrLongRow = 256;           // a row of more entries, and more than a wavefront's share, takes the whole workgroup
constexpr int kCsrUnroll = 8;              // gathers in flight per sub-wave

struct CsrArgs {
    const int32_t* indptr;
    const int32_t* indices;
    const float* values;                   // null: ones
    long long n_rows, n_groups;
    int rows_per_group;
    int slices;                            // feature slices, a power of two up to kXcds
    int feat, ld;                          // features of a slice; elements between rows of B and of C
    const void* B;
    float* C;
    unsigned long long b_bytes;
};

// Gathers go through a buffer resource over B: the lane that fetched an entry multiplies its column by the bytes of a
// row once, a gather then costs one addition (with the broadcast in it) for its address, and entries past the end of
// a row get an offset past the end of B, for which the hardware returns zeros without touching memory - no padding
// traffic, and nothing for an infinite element of B to turn into NaN.  Offsets have 32 bits: a larger B takes
// 64-bit addresses and predicated loads instead (WIDE; 57K rows of 28 entries, N = 64 .. 256: 1 - 7 % slower).
constexpr uint32_t kPastB = 0xFFFE0000u;   // (a lane's own offset is below 2^17)

// Entry I of the sub-wave's batch, from the lane that holds it, by a DPP broadcast: one operand modifier of the
// addition or move that uses it, where a shuffle is an LDS instruction and its latency.
template <int LPR, int I> __device__ __forceinline__ int batch_entry(int x) {
    constexpr int kRowBroadcast = 0x150;   // row_newbcast: a lane of each row of 16 to that row
    if constexpr (LPR >= 16) {
        return __builtin_amdgcn_update_dpp(0, x, kRowBroadcast + I, 0xF, 0xF, true);
    } else {                               // two sub-waves to a row of 16 lanes
        const int first = __builtin_amdgcn_update_dpp(0, x, kRowBroadcast + I, 0xF, 0x3, false);
        return __builtin_amdgcn_update_dpp(first, x, kRowBroadcast + 8 + I, 0xF, 0xC, false);
    }
}

typedef unsigned int lf_u32x4 __attribute__((ext_vector_type(4)));

// A wavefront's teams of 2^lg sub-waves.  Entry e of a row goes to sub-wave e mod 2^lg of its team.
template <int LPR, int CH, typename BT, bool WIDE> struct Teams {
    static constexpr int VEC = Dense<BT>::kVec;
    static constexpr int kBatch = LPR < 16 ? LPR : 16;      // entries of a sub-wave fetched at a time
    using Raw = typename Dense<BT>::Raw;
    const int32_t* indices;
    const float* values;
    const char* B;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t pitch;                        // bytes between rows of B
    uint32_t lane_at[CH];                  // the lane's own bytes in a row of B
    int lg;
    int sub;                               // sub-wave in its team
    int slot;                              // entry of a batch that the lane fetches (in every 16 lanes again)

    // The lane's entry of the batch at `base` of the row of `len` entries from `lo` on.
    __device__ __forceinline__ void fetch(int lo, int len, int base, int& col, float& val) const {
        const int e = base + (slot << lg) + sub;
        col = -1;
        val = 0.f;
        if (e < len) {
            col = indices[lo + e];
            val = values ? values[lo + e] : 1.f;
        }
    }

    template <int FIRST, size_t... I>
    __device__ __forceinline__ void gather(int at, float val, Acc<CH, VEC>& acc, std::index_sequence<I...>) const {
        Raw x[kCsrUnroll][CH];
        auto load = [&](int u, int from) {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                if constexpr (WIDE) {
                    x[u][c] = Raw{};
                    if (from >= 0) x[u][c] = *reinterpret_cast<const Raw*>(B + lane_at[c] + (uint64_t)(uint32_t)from * pitch);
                } else {
                    const lf_u32x4 raw = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (uint32_t)from + lane_at[c], 0, 0);
                    __builtin_memcpy(&x[u][c], &raw, sizeof(Raw));
                }
            }
        };
        (load(I, batch_entry<LPR, FIRST + I>(at)), ...);
        auto add = [&](int u, float v) {
#pragma unroll
            for (int c = 0; c < CH; ++c) fma_dense<BT>(v, x[u][c], acc.v[c]);
        };
        (add(I, __int_as_float(batch_entry<LPR, FIRST + I>(__float_as_int(val)))), ...);
    }

    // Adds the entries of the team's row; `most` is the length of the wavefront's longest row (uniform).
    __device__ __forceinline__ void sum(int lo, int len, int most, Acc<CH, VEC>& acc) const {
        constexpr auto kEight = std::make_index_sequence<kCsrUnroll>();
        int col;
        float val;
        fetch(lo, len, 0, col, val);
        for (int base = 0; base < most;) {
            const int at = WIDE ? col : col >= 0 ? (int)((uint32_t)col * pitch) : (int)kPastB;
            const float v = val;
            const int left = most - base;
            base += kBatch << lg;
            if (base < most) fetch(lo, len, base, col, val);
            gather<0>(at, v, acc, kEight);
            if constexpr (kBatch > kCsrUnroll)
                if (left > (kCsrUnroll << lg)) gather<kCsrUnroll>(at, v, acc, kEight);
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

// Bound by the gathers where rows are long; by the chain row pointer - entries - gathers and the number of
// wavefronts that hide it where they are short.  Requesting the next rows' entries ahead costs more registers than
// it hides (57K rows of 28, N = 64: 42 us, 40 so).
//
// What the lengths of a graph's rows cost is why a row belongs to a team, and why rows are handed out.  A sub-wave
// per row, and runs of rows to a sub-wave where a group holds longer ones, the form before, had every wavefront
// wait for its longest row or look for a row's end behind every gather.  Log-normal rows (sigma 0.8; 57K 0.9), us,
// before -> now:
//   rows x entries   N = 32        N = 64        N = 128       N = 256       bf16 N = 128
//   8000 x 32        22.3 -> 6.7                 23.8 -> 11.7
//   57000 x 28       49.3 -> 23.6  64.4 -> 40.1  113 -> 76     221 -> 158    71.2 -> 53.2
//   32000 x 128                                  235 -> 128
//   170K, power law                98 -> 72                    255 -> 172
// (from N = 64 on with feature slices, see csr_slices).
template <int LPR, int CH, typename BT, bool WIDE>
__global__ void __launch_bounds__(kCsrThreads)
csr_spmm_kernel(CsrArgs a) {
    constexpr int VEC = Dense<BT>::kVec;
    constexpr int kWaves = kCsrThreads / 64;
    constexpr int kLgSubs = LPR == 64 ? 0 : LPR == 32 ? 1 : LPR == 16 ? 2 : 3;      // log2 of the wavefront's sub-waves
    using T = Teams<LPR, CH, BT, WIDE>;
    __shared__ int s_next;
    extern __shared__ __align__(16) float s_red[];         // [kWaves][feat]: sums of a long row's parts
    // workgroup i runs on XCD i % 8; XCD x computes slice x mod slices of its rows
    const int xcd = blockIdx.x % kXcds, slice = xcd & (a.slices - 1);
    const long long group = (long long)(blockIdx.x / kXcds) * (kXcds / a.slices) + xcd / a.slices;
    if (group >= a.n_groups) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sl = lane % LPR, sub = lane / LPR;
    const Lane<LPR, CH, VEC> ln(sl, a.feat, a.ld, a.ld);
    const size_t skip = (size_t)slice * a.feat;
    float* C = a.C + skip;
    T t;
    t.indices = a.indices;
    t.values = a.values;
    t.B = (const char*)a.B + skip * Dense<BT>::kElemBytes;
    t.pitch = (uint32_t)a.ld * Dense<BT>::kElemBytes;
    t.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)t.B, 0, WIDE ? 0 : (int)(uint32_t)(a.b_bytes - skip * Dense<BT>::kElemBytes), 0x00027000);
#pragma unroll
    for (int c = 0; c < CH; ++c) t.lane_at[c] = ln.f[c] * Dense<BT>::kElemBytes;
    t.slot = sl % T::kBatch;

    const long long first_row = group * a.rows_per_group;
    const int n = (int)min((long long)a.rows_per_group, a.n_rows - first_row);       // at most 64
    const int start = a.indptr[first_row + min(lane, n)], end = a.indptr[first_row + min(lane + 1, n)];
    if (tid == 0) s_next = kWaves;
    __syncthreads();
    const int total = __builtin_amdgcn_readlane(end, 63) - __builtin_amdgcn_readfirstlane(start);
    const unsigned long long longs = __ballot(end - start > max(kCsrLongRow, total / kWaves));      // the same in every wavefront
    // as many sub-waves as give each one batch of gathers of an average row (half or twice as many: 1 - 7 % slower)
    int lg = 0;
    while (lg < kLgSubs && ((long long)(n * kCsrUnroll) << lg) < total) ++lg;
    t.lg = lg = __builtin_amdgcn_readfirstlane(lg);
    t.sub = sub & ((1 << lg) - 1);
    const int lg_rows = kLgSubs - lg, team = sub >> lg;
    const int sets = (n + (1 << lg_rows) - 1) >> lg_rows;
    for (int set = wave; set < sets;) {                      // 2^lg_rows rows at a time
        const int r = (set << lg_rows) + team, from = min(r, n - 1);
        const int lo = __shfl(start, from), hi = __shfl(end, from);        // (the lanes shuffled from are all active)
        const bool mine = r < n && ((longs >> from) & 1) == 0;
        const int len = mine ? hi - lo : 0;
        int most = len;
        for (int d = LPR << lg; d < 64; d <<= 1) most = max(most, __shfl_xor(most, d));
        Acc<CH, VEC> acc;
        acc.clear();
        t.sum(lo, len, __builtin_amdgcn_readfirstlane(most), acc);
        t.combine(acc);
        if (t.sub == 0 && mine) store_row<LPR, CH, VEC>(C, (int)(first_row + r), ln, acc, kStreamC);
        int next = 0;
        if (lane == 0) next = atomicAdd(&s_next, 1);
        set = __builtin_amdgcn_readfirstlane(next);
    }
    // Long rows: a part to each wavefront, the parts' sums added in their order.
    t.lg = kLgSubs;
    t.sub = sub;
    constexpr int kStep = T::kBatch << kLgSubs;
    for (unsigned long long todo = longs; todo; todo &= todo - 1) {                  // uniform
        const int r = __ffsll((long long)todo) - 1;
        const int lo = __builtin_amdgcn_readlane(start, r), len = __builtin_amdgcn_readlane(end, r) - lo;
        const int per = ((len - 1) / kWaves / kStep + 1) * kStep;
        const int from = (int)min((long long)wave * per, (long long)len), part = min(per, len - from);
        Acc<CH, VEC> acc;
        acc.clear();
        t.sum(lo + from, part, part, acc);
        t.combine(acc);
        if (sub == 0) {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                if (!ln.on[c]) continue;
#pragma unroll
                for (int i = 0; i < VEC; ++i) s_red[wave * a.feat + ln.f[c] + i] = acc.v[c][i];
            }
        }
        __syncthreads();
        for (int f = tid; f < a.feat; f += kCsrThreads) {
            float sum = 0.f;
            for (int w = 0; w < kWaves; ++w) sum += s_red[w * a.feat + f];
            C[(size_t)(first_row + r) * a.ld + f] = sum;
        }
        __syncthreads();                                     // before the next row's parts
    }
}

using CsrFn = void (*)(CsrArgs);

template <int LPR, int CH> CsrFn csr_kernel(int dtype, bool wide) {
    if (dtype == LF_DTYPE_BF16) return wide ? csr_spmm_kernel<LPR, CH, bf16_t, true> : csr_spmm_kernel<LPR, CH, bf16_t, false>;
    return wide ? csr_spmm_kernel<LPR, CH, float, true> : csr_spmm_kernel<LPR, CH, float, false>;
}

CsrFn csr_kernel(int lpr, int ch, int dtype, bool wide) {
    if (ch == 2) return csr_kernel<64, 2>(dtype, wide);
    if (ch == 4) return csr_kernel<64, 4>(dtype, wide);
    return lpr == 8 ? csr_kernel<8, 1>(dtype, wide) : lpr == 16 ? csr_kernel<16, 1>(dtype, wide)
         : lpr == 32 ? csr_kernel<32, 1>(dtype, wide) : csr_kernel<64, 1>(dtype, wide);
}

// Feature slices: XCD x computes slice x mod S of the features for every (8 / S)-th group of rows, so that its L2
// has 1 / S of B to hold instead of all of it, at the price of reading the entries S times.  A slice is
// 128 bytes or a multiple: a gather of 64 moves the line all the same (a table in the L2s is gathered from at 28 TB/s
// by rows of 128 bytes and more, 15.5 by rows of 64).  The S that a simple price puts first: gathers that miss at 7.3
// TB/s and those that hit at 28, the share that hits from the slice's size and from how often an XCD uses a row of B
// (from the second time on), and 10 % for every halving of the workgroups below 2048, which is what small matrices
// gain from the split.  130 matrices of 2K to 1.2M rows, log-normal and power-law, N = 64 .. 512, f32 and bf16, every
// S timed: the pick loses 2.1 % on average to the best, S = 1 24 %, S = 4 4.6 %.  Worst picks: 34 % (9K x 13K, 31K
// entries, bf16 N = 256: 8.5 us with 2, 11.4 with 4), and against S = 1 14 % (335K power-law rows, N = 128: 119 -> 135).
int csr_slices(int64_t num_rows, int64_t num_cols, int64_t nnz, int feat, int dtype) {
    constexpr double kL2 = 5.5e6, kMissRate = 7.3, kHitRate = 28.0, kGroups = 2048.0;
    const int elem = dtype == LF_DTYPE_BF16 ? 2 : 4, step = 128 / elem;
    const double b_bytes = (double)num_cols * feat * elem, gathered = (double)nnz * feat * elem;
    const double groups = (double)num_rows / (num_rows >= kCsrManyRows ? kCsrRowsMany : kCsrRowsFew) + 1.0;
    int best = 1;
    double least = 0.0;
    for (int s = 1; s <= kXcds && nnz > 0; s *= 2) {
        if (feat % (s * step) != 0) break;
        const double uses = (double)nnz / (double)num_cols * s / kXcds;
        const double hit = std::min(1.0, kL2 * s / b_bytes) * std::max(0.0, 1.0 - 1.0 / uses);
        double price = gathered * ((1.0 - hit) / kMissRate + hit / kHitRate) + 8.0 * (double)nnz * s / kMissRate;
        price *= 1.0 + 0.1 * std::max(0.0, std::log2(kGroups / (groups * s)));
        if (s == 1 || price < 0.98 * least) {
            least = price;
            best = s;
        }
    }
    return best;
}

}  // namespace

extern "C" {

int lf_csr_spmm_trusted_nnz(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values,
                            int64_t num_rows, int64_t num_cols, int64_t nnz, int32_t feat_size, int32_t b_dtype,
                            const void* d_B, float* d_C, lf_stream_t stream) {
    LF_REQUIRE(num_rows >= 0 && num_rows < (1ll << 31) && num_cols >= 1, LF_ERR_INVALID, "bad shape");
    if (num_rows == 0) return LF_OK;
    LF_REQUIRE(d_indptr && d_B && d_C, LF_ERR_INVALID, "null argument");
    LF_REQUIRE(b_dtype == LF_DTYPE_F32 || b_dtype == LF_DTYPE_BF16, LF_ERR_INVALID, "unknown B dtype %d", b_dtype);
    LF_REQUIRE((uintptr_t)d_B % 16 == 0 && (uintptr_t)d_C % 16 == 0, LF_ERR_INVALID, "B and C must be 16-byte aligned");
    int lpr, ch;
    if (int rc = feature_shape(feat_size, b_dtype, &lpr, &ch)) return rc;
    CsrArgs a{};
    a.slices = csr_slices(num_rows, num_cols, nnz, feat_size, b_dtype);
    a.feat = feat_size / a.slices;
    if (int rc = feature_shape(a.feat, b_dtype, &lpr, &ch)) return rc;
    a.indptr = d_indptr;
    a.indices = d_indices;
    a.values = d_values;
    a.n_rows = num_rows;
    a.rows_per_group = num_rows >= kCsrManyRows ? kCsrRowsMany : kCsrRowsFew;
    a.n_groups = lf::ceil_div(num_rows, (int64_t)a.rows_per_group);
    a.ld = feat_size;
    a.B = d_B;
    a.C = d_C;
    a.b_bytes = (unsigned long long)num_cols * feat_size * (b_dtype == LF_DTYPE_BF16 ? 2 : 4);
    const unsigned grid = (unsigned)(lf::ceil_div(a.n_groups, (int64_t)(kXcds / a.slices)) * kXcds);
    csr_kernel(lpr, ch, b_dtype, a.b_bytes > kPastB)<<<grid, kCsrThreads, (kCsrThreads / 64) * a.feat * sizeof(float), (hipStream_t)stream>>>(a);
    LF_HIP(hipGetLastError());
    return LF_OK;
}

int lf_csr_spmm_trusted(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values,
                        int64_t num_rows, int64_t num_cols, int32_t feat_size, int32_t b_dtype,
                        const void* d_B, float* d_C, lf_stream_t stream) {
    return lf_csr_spmm_trusted_nnz(d_indptr, d_indices, d_values, num_rows, num_cols, 0, feat_size, b_dtype, d_B, d_C, stream);
}

int lf_csr_spmm(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values,
                int64_t num_rows, int64_t num_cols, int64_t nnz, int32_t feat_size, int32_t b_dtype,
                const void* d_B, float* d_C, void* d_scratch, lf_stream_t stream) {
    // arguments first, so that a bad feature size or operand is reported without touching the GPU
    LF_REQUIRE(num_rows >= 0 && num_rows < (1ll << 31) && num_cols >= 1, LF_ERR_INVALID, "bad shape");
    if (num_rows > 0) {
        LF_REQUIRE(d_indptr && d_B && d_C, LF_ERR_INVALID, "null argument");
        LF_REQUIRE(b_dtype == LF_DTYPE_F32 || b_dtype == LF_DTYPE_BF16, LF_ERR_INVALID, "unknown B dtype %d", b_dtype);
        int lpr, ch;
        if (int rc = feature_shape(feat_size, b_dtype, &lpr, &ch)) return rc;
    }
    // no gather before the index arrays have passed
    if (int rc = lf::csr_check(d_indptr, d_indices, nullptr, num_rows, num_cols, nnz, d_scratch, nullptr, "lf_csr_spmm",
                               (hipStream_t)stream))
        return rc;
    return lf_csr_spmm_trusted_nnz(d_indptr, d_indices, d_values, num_rows, num_cols, nnz, feat_size, b_dtype, d_B, d_C, stream);
}

}  // extern "C"
