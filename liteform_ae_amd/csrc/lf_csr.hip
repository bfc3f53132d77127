// CSR product without a plan for gfx950:  C[rows][N] = A_csr . B[cols][N], fp32 accumulate.
//
// The counterpart of bench_naive's kernel (playground_pipline/format_algos.py:1689-1755), which gives a row to a
// thread block.  Here the entries of a row are spread over a *team* of sub-waves: a sub-wave of LPR lanes covers a
// row of B with one 16-byte load per lane, and the 64 / LPR sub-waves of a wavefront work on one row, two rows, ...
// or a row each, as the lengths of the workgroup's rows ask for.
#include <hip/hip_runtime.h>


#include "lf_internal.h"
#include "lf_spmm_device.h"

namespace {

// A workgroup of four wavefronts takes kCsrRowsFew or kCsrRowsMany consecutive rows; a wavefront takes the next rows
// off a counter whenever it is through with its own, so that nothing waits for the longest row but itself.
constexpr int kCsrThreads = 256;
constexpr int kCsrRowsFew = 8, kCsrRowsMany = 16;
constexpr long long kCsrManyRows = 24576;
constexpr int kCsrLongRow = 256;           // a row of more entries, and more than a wavefront's share, takes the whole workgroup

struct CsrArgs {
    const int32_t* indptr;
    const int32_t* indices;
    const float* values;                   // null: ones
    long long n_rows, n_groups;
    int rows_per_group;
    int share;                             // entries of a sub-wave, see csr_share
    int feat, ld;                          // features of a slice (the last may have fewer); elements between rows of B and of C
    XcdParts parts;
    const void* B;
    float* C;
    unsigned long long b_bytes;
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
    constexpr int kLgSubs = Teams<LPR, CH, BT, WIDE>::kLgSubs;
    __shared__ int s_next;
    extern __shared__ __align__(16) float s_red[];         // [kWaves][feat]: sums of a long row's parts
    // workgroup i runs on XCD i % 8 and takes entry i / 8 of that XCD's part
    const XcdPart part = xcd_part(a.parts, blockIdx.x % kXcds);
    const int n_groups = (int)a.n_groups;
    int slice = part.slice, group = tiles_before(n_groups, part.from) + blockIdx.x / kXcds;
    if (group >= tiles_before(n_groups, part.upto)) {
        group -= tiles_before(n_groups, part.upto);
        if (group >= tiles_before(n_groups, part.next)) return;
        ++slice;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sub = lane / LPR;
    const size_t skip = (size_t)slice * a.feat;
    const int feat = min(a.feat, a.ld - (int)skip);
    const Lane<LPR, CH, VEC> ln(lane % LPR, feat, a.ld, a.ld);
    const RowsOfB<LPR, CH, BT, WIDE> b((const char*)a.B + skip * Dense<BT>::kElemBytes, a.b_bytes - skip * Dense<BT>::kElemBytes, ln);
    float* C = a.C + skip;

    const long long first_row = (long long)group * a.rows_per_group;
    const int n = (int)min((long long)a.rows_per_group, a.n_rows - first_row);       // at most 64
    const int start = a.indptr[first_row + min(lane, n)], end = a.indptr[first_row + min(lane + 1, n)];
    if (tid == 0) s_next = kWaves;
    __syncthreads();
    const int total = __builtin_amdgcn_readlane(end, 63) - __builtin_amdgcn_readfirstlane(start);
    const unsigned long long longs = __ballot(end - start > max(kCsrLongRow, total / kWaves));      // the same in every wavefront
    // as many sub-waves as give each at most `share` entries of an average row
    int lg = 0;
    while (lg < kLgSubs && ((long long)(n * a.share) << lg) < total) ++lg;
    const Teams<LPR, CH, BT, WIDE> teams(b, __builtin_amdgcn_readfirstlane(lg));
    const int lg_rows = kLgSubs - teams.lg, team = sub >> teams.lg;
    const int sets = (n + (1 << lg_rows) - 1) >> lg_rows;
    for (int set = wave; set < sets;) {                      // 2^lg_rows rows at a time
        const int r = (set << lg_rows) + team, from = min(r, n - 1);
        const int lo = __shfl(start, from), hi = __shfl(end, from);        // (the lanes shuffled from are all active)
        const bool mine = r < n && ((longs >> from) & 1) == 0;
        const int len = mine ? hi - lo : 0;
        int most = len;
        for (int d = LPR << teams.lg; d < 64; d <<= 1) most = max(most, __shfl_xor(most, d));
        Acc<CH, VEC> acc;
        acc.clear();
        teams.sum(a.indices, a.values, lo, len, __builtin_amdgcn_readfirstlane(most), acc);
        teams.combine(acc);
        if (teams.sub == 0 && mine) store_row<LPR, CH, VEC>(C, (int)(first_row + r), ln, acc, kStreamC);
        int next = 0;
        if (lane == 0) next = atomicAdd(&s_next, 1);
        set = __builtin_amdgcn_readfirstlane(next);
    }
    // Long rows: a part to each wavefront, the parts' sums added in their order.
    const Teams<LPR, CH, BT, WIDE> all(b, kLgSubs);
    constexpr int kStep = Teams<LPR, CH, BT, WIDE>::kBatch << kLgSubs;
    for (unsigned long long todo = longs; todo; todo &= todo - 1) {                  // uniform
        const int r = __ffsll((long long)todo) - 1;
        const int lo = __builtin_amdgcn_readlane(start, r), len = __builtin_amdgcn_readlane(end, r) - lo;
        const int per = ((len - 1) / kWaves / kStep + 1) * kStep;
        const int from = (int)min((long long)wave * per, (long long)len), part = min(per, len - from);
        Acc<CH, VEC> acc;
        acc.clear();
        all.sum(a.indices, a.values, lo + from, part, part, acc);
        all.combine(acc);
        if (sub == 0) {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                if (!ln.on[c]) continue;
#pragma unroll
                for (int i = 0; i < VEC; ++i) s_red[wave * feat + ln.f[c] + i] = acc.v[c][i];
            }
        }
        __syncthreads();
        for (int f = tid; f < feat; f += kCsrThreads) {
            float sum = 0.f;
            for (int w = 0; w < kWaves; ++w) sum += s_red[w * feat + f];
            C[(size_t)(first_row + r) * a.ld + f] = sum;
        }
        __syncthreads();                                     // before the next row's parts
    }
}

// A sub-wave's entries of an average row at most.  One batch of gathers (half or twice as many: 1 - 7 % slower; 17K power-law
// rows of 3, N = 64 8.4 us, a batch and a half 9.7).  But where B is past the memory-side cache too, what counts is how
// many gathers are in flight, and two sub-waves on a row of nine leave half of theirs empty: a batch and a half.  1.8M rows of
// 9.6 and 8.8, N = 96: 1190 and 1162 us, 1250 and 1194 with one batch (1150 and 1128 with a sub-wave streaming over the ends of
// rows); 1.1M of 8.6, N = 192 1316, 1348, 1311.  (B of 53 to 210 MB: 500K rows of 9, N = 32 101 and 96; 147K of 11, N = 384 367
// and 354.)
constexpr unsigned long long kMallBytes = 256ull << 20;
int csr_share(unsigned long long b_bytes) { return b_bytes > kMallBytes ? kUnroll * 3 / 2 : kUnroll; }

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

// 16 % for every halving of the workgroups below 2048: what small matrices gain from the split besides; 2 % for every
// doubling of S and 7 us for a million rows' starts, for what its price does not hold; 0.3 us for every doubling of the
// sub-waves to a wavefront; and 4 % where a row takes a whole wavefront (rows of B over 512 bytes): nothing then fills the
// gathers that its last batch leaves empty (433K rows of 9 entries, N = 256: 647 us with S = 1, 604 with 2; 300K power-law
// rows of 5: 430, 346).  1000 matrices of 2K to 2M rows, log-normal and power-law, N = 64 .. 512, f32 and bf16, every S
// timed: the pick takes 0.89 of the time of S = 1 on average, 2.6 % more than the best; 3 % of them are more than 3 % slower
// than with S = 1, 21 % at worst (25K rows of 4, N = 160: 12.9 us, 15.6 with 5).  128K rows of 100, N = 96: 635 us with 1,
// 564 with 3.
Slices csr_slices(int64_t rows, int rows_per_group, int64_t groups, int64_t num_cols, int64_t nnz, int64_t span, int feat, int dtype) {
    return feature_slices(num_cols, nnz, feat, dtype, Neighbours{(double)span, rows, 0.05}, [&](int) { return (double)rows_per_group; }, [&](int s, int width, int lg_subs, double us) {
        return us * (1.0 + 0.16 * std::max(0.0, std::log2(2048.0 / ((double)groups * s))))
                  * (width * (dtype == LF_DTYPE_BF16 ? 2 : 4) > 512 ? 1.04 : 1.0) * (1.0 + 0.02 * std::log2((double)s))
               + 0.3 * lg_subs + 7e-6 * (double)rows * s;
    });
}

}  // namespace

extern "C" {

int lf_csr_spmm_trusted_span(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values,
                             int64_t num_rows, int64_t num_cols, int64_t nnz, int64_t span, int32_t feat_size,
                             int32_t b_dtype, const void* d_B, float* d_C, lf_stream_t stream) {
    LF_REQUIRE(num_rows >= 0 && num_rows < (1ll << 31) && num_cols >= 1, LF_ERR_INVALID, "bad shape");
    if (num_rows == 0) return LF_OK;
    LF_REQUIRE(d_indptr && d_B && d_C, LF_ERR_INVALID, "null argument");
    LF_REQUIRE(b_dtype == LF_DTYPE_F32 || b_dtype == LF_DTYPE_BF16, LF_ERR_INVALID, "unknown B dtype %d", b_dtype);
    LF_REQUIRE((uintptr_t)d_B % 16 == 0 && (uintptr_t)d_C % 16 == 0, LF_ERR_INVALID, "B and C must be 16-byte aligned");
    int lpr, ch;
    if (int rc = feature_shape(feat_size, b_dtype, &lpr, &ch)) return rc;
    CsrArgs a{};
    a.rows_per_group = num_rows >= kCsrManyRows ? kCsrRowsMany : kCsrRowsFew;
    a.n_groups = lf::ceil_div(num_rows, (int64_t)a.rows_per_group);
    const Slices slices = csr_slices(num_rows, a.rows_per_group, a.n_groups, num_cols, nnz, span, feat_size, b_dtype);
    a.feat = slices.feat;
    a.parts = slices.parts;
    if (int rc = feature_shape(a.feat, b_dtype, &lpr, &ch)) return rc;
    a.indptr = d_indptr;
    a.indices = d_indices;
    a.values = d_values;
    a.n_rows = num_rows;
    a.ld = feat_size;
    a.B = d_B;
    a.C = d_C;
    a.b_bytes = (unsigned long long)num_cols * feat_size * (b_dtype == LF_DTYPE_BF16 ? 2 : 4);
    a.share = csr_share(a.b_bytes);
    long long longest = 0;
    for (int x = 0; x < kXcds; ++x) longest = std::max(longest, part_tiles(a.parts, x, a.n_groups));
    const unsigned grid = (unsigned)(longest * kXcds);
    csr_kernel(lpr, ch, b_dtype, a.b_bytes > kPastB)<<<grid, kCsrThreads, (kCsrThreads / 64) * a.feat * sizeof(float), (hipStream_t)stream>>>(a);
    LF_HIP(hipGetLastError());
    return LF_OK;
}

int lf_csr_spmm_trusted_nnz(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values,
                            int64_t num_rows, int64_t num_cols, int64_t nnz, int32_t feat_size, int32_t b_dtype,
                            const void* d_B, float* d_C, lf_stream_t stream) {
    return lf_csr_spmm_trusted_span(d_indptr, d_indices, d_values, num_rows, num_cols, nnz, 0, feat_size, b_dtype, d_B, d_C, stream);
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
    int64_t span = 0;
    if (int rc = lf::csr_check(d_indptr, d_indices, nullptr, num_rows, num_cols, nnz, d_scratch, nullptr, &span, "lf_csr_spmm",
                               (hipStream_t)stream))
        return rc;
    return lf_csr_spmm_trusted_span(d_indptr, d_indices, d_values, num_rows, num_cols, nnz, span, feat_size, b_dtype, d_B, d_C, stream);
}

}  // extern "C"
