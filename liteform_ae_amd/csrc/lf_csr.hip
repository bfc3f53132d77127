// CSR product without a plan for gfx950:  C[rows][N] = A_csr . B[cols][N], fp32 accumulate.
//
// The counterpart of bench_naive's kernel (playground_pipline/format_algos.py:1689-1755), which gives a row to a
// thread block.  Here the entries of a row are spread over a *team* of sub-waves: a sub-wave of LPR lanes covers a
// row of B with one 16-byte load per lane, and the 64 / LPR sub-waves of a wavefront work on one row, two rows, ...
// or a row each, as the lengths of the workgroup's rows ask for.
#include <hip/hip_runtime.h>

#include "lf_index.h"
#include "lf_internal.h"
#include "lf_rules.h"
#include "lf_spmm_device.h"

namespace {

// A workgroup of four wavefronts takes 2, 4, 8 or 16 consecutive rows (csr_rows_of_group); a wavefront takes the next rows
// off a counter whenever it is through with its own, so that nothing waits for the longest row but itself.
constexpr int kCsrThreads = 256;
constexpr int kCsrChunkedRow = 512, kCsrChunk = 512;      // rows of more entries are cut into chunks, see csr_shape
constexpr double kSmallBatchUs = 0.35, kBatchUs = 0.6, kFinalUs = 10.0, kTail = 0.02, kPanelTail = 0.15, kFewOfACu = 4.0;
constexpr int kCsrLongRow = 256;           // a row of more entries, and more than a wavefront's share, takes the whole workgroup

struct CsrArgs {
    const int32_t* starts;                 // the row pointer, or (CsrMore) entries of row r in the launch's panel: [starts[r], ends[r])
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

// What a launch on one of several panels of columns, or with chunks of long rows, has besides.
struct CsrMore {
    const int32_t* ends;
    int flags;                             // kAccumulateC, kStreamC
    int long_row;                          // rows of more entries are in `chunks`
    int n_chunks;
    const int2* chunks;                    // (first entry, entries)
    float* partials;                       // [n_chunks][ld]
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
//
// MORE: panels and chunks.  An instantiation of its own: their arguments and tests cost every workgroup of the other launches (13.6K
// rows of 4, N = 480: 21.1 us, 24.7 with them).
//
// Three wavefronts to a SIMD at least for up to 1024 float features: left to itself the compiler took 174 registers, which are two, and
// products of more than 512 features 4 - 11 % more time (150K power-law rows, N = 544 / 1024 300 / 443 us, 335 / 472 so; 300K, N = 800 767, 833).
constexpr int csr_waves(int ch, bool floats, bool wide, bool more) { return ch == 4 && floats && !wide && !more ? 3 : 1; }
template <int LPR, int CH, typename BT, bool WIDE, bool MORE>
__global__ void __launch_bounds__(kCsrThreads, csr_waves(CH, sizeof(BT) == 4, WIDE, MORE))
csr_spmm_kernel(CsrArgs a, CsrMore more) {
    constexpr int VEC = Dense<BT>::kVec;
    constexpr int kWaves = kCsrThreads / 64;
    constexpr int kLgSubs = Teams<LPR, CH, BT, WIDE>::kLgSubs;
    __shared__ int s_next;
    extern __shared__ __align__(16) float s_red[];         // [kWaves][feat]: sums of a long row's parts
    // workgroup i runs on XCD i % 8 and takes entry i / 8 of that XCD's part
    const XcdPart part = xcd_part(a.parts, blockIdx.x % kXcds);
    const int n_groups = (int)a.n_groups;
    int slice = part.slice, group = blockIdx.x / kXcds, chunk = -1;
    if constexpr (MORE) {                                    // chunks first: they are the longest
        const int c0 = tiles_before(more.n_chunks, part.from), c = tiles_before(more.n_chunks, part.upto) - c0;
        const int g0 = tiles_before(n_groups, part.from), g = tiles_before(n_groups, part.upto) - g0;
        if (group < c) {
            chunk = c0 + group;
        } else if (group - c < g) {
            group += g0 - c;
        } else {
            group -= c + g;
            ++slice;
            const int c_next = tiles_before(more.n_chunks, part.next);
            if (group < c_next) chunk = group;
            else if ((group -= c_next) >= tiles_before(n_groups, part.next)) return;
        }
    } else {
        group += tiles_before(n_groups, part.from);
        if (group >= tiles_before(n_groups, part.upto)) {
            group -= tiles_before(n_groups, part.upto);
            if (group >= tiles_before(n_groups, part.next)) return;
            ++slice;
        }
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sub = lane / LPR;
    const size_t skip = (size_t)slice * a.feat;
    const int feat = min(a.feat, a.ld - (int)skip);
    const Lane<LPR, CH, VEC> ln(lane % LPR, feat, a.ld, a.ld);
    const RowsOfB<LPR, CH, BT, WIDE> b((const char*)a.B + skip * Dense<BT>::kElemBytes, a.b_bytes - skip * Dense<BT>::kElemBytes, ln);
    float* C = a.C + skip;

    // A chunk of a long row, or a long row: a part to each wavefront, the parts' sums added in their order.
    const Teams<LPR, CH, BT, WIDE> all(b, kLgSubs);
    constexpr int kStep = Teams<LPR, CH, BT, WIDE>::kBatch << kLgSubs;
    auto together = [&](int lo, int len, float* dst, bool add) {
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
            dst[f] = add ? dst[f] + sum : sum;
        }
        __syncthreads();                                     // before the next row's parts
    };
    if (MORE && chunk >= 0) {
        const int2 ck = more.chunks[chunk];
        together(__builtin_amdgcn_readfirstlane(ck.x), __builtin_amdgcn_readfirstlane(ck.y), more.partials + (size_t)chunk * a.ld + skip, false);
        return;
    }
    const int flags = MORE ? more.flags : kStreamC;
    const bool add = (flags & kAccumulateC) != 0;

    const long long first_row = (long long)group * a.rows_per_group;
    const int n = (int)min((long long)a.rows_per_group, a.n_rows - first_row);       // at most 64
    // (of the lanes past the last row: nothing, or the last row's once more)
    const int start = a.starts[first_row + (MORE ? min(lane, n - 1) : min(lane, n))];
    const int end = MORE ? more.ends[first_row + min(lane, n - 1)] : a.starts[first_row + min(lane + 1, n)];
    if (tid == 0) s_next = kWaves;
    __syncthreads();
    int total;
    unsigned long long longs = 0;                            // rows that are not summed with the others: the same in every wavefront
    if constexpr (MORE) {
        const bool whole = lane < n && end - start <= more.long_row;
        total = whole ? end - start : 0;
        for (int d = 1; d < 64; d <<= 1) total += __shfl_xor(total, d);
        total = __builtin_amdgcn_readfirstlane(total);
        longs = __ballot(whole && end - start > max(kCsrLongRow, total / kWaves));
    } else {
        total = __builtin_amdgcn_readlane(end, 63) - __builtin_amdgcn_readfirstlane(start);
        longs = __ballot(end - start > max(kCsrLongRow, total / kWaves));
    }
    const unsigned long long others = MORE ? longs | __ballot(end - start > more.long_row) : longs;
    // as many sub-waves as give each at most `share` entries of an average row
    int lg = 0;
    while (lg < kLgSubs && ((long long)(n * a.share) << lg) < total) ++lg;
    const Teams<LPR, CH, BT, WIDE> teams(b, __builtin_amdgcn_readfirstlane(lg));
    const int lg_rows = kLgSubs - teams.lg, team = sub >> teams.lg;
    const int sets = (n + (1 << lg_rows) - 1) >> lg_rows;
    for (int set = wave; set < sets;) {                      // 2^lg_rows rows at a time
        const int r = (set << lg_rows) + team, from = min(r, n - 1);
        const int lo = __shfl(start, from), hi = __shfl(end, from);        // (the lanes shuffled from are all active)
        const bool mine = r < n && ((others >> from) & 1) == 0;
        const int len = mine ? hi - lo : 0;
        int most = len;
        for (int d = LPR << teams.lg; d < 64; d <<= 1) most = max(most, __shfl_xor(most, d));
        Acc<CH, VEC> acc;
        acc.clear();
        teams.sum(a.indices, a.values, lo, len, __builtin_amdgcn_readfirstlane(most), acc);
        teams.combine(acc);
        if (teams.sub == 0 && mine && (len > 0 || !add)) store_row<LPR, CH, VEC>(C, (int)(first_row + r), ln, acc, flags);
        int next = 0;
        if (lane == 0) next = atomicAdd(&s_next, 1);
        set = __builtin_amdgcn_readfirstlane(next);
    }
    for (unsigned long long todo = longs; todo; todo &= todo - 1) {                  // uniform
        const int r = __ffsll((long long)todo) - 1;
        const int lo = __builtin_amdgcn_readlane(start, r);
        together(lo, __builtin_amdgcn_readlane(end, r) - lo, C + (size_t)(first_row + r) * a.ld, add);
    }
}

// bounds[p - 1][r]: first entry of row r at or past column p * width, p = 1 .. panels - 1.  The panels of a row that is left to the
// chunks are empty but for the last.
__global__ void __launch_bounds__(256)
csr_bounds_kernel(const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices, long long n_rows, int width, int long_row,
                  int32_t* __restrict__ bounds) {
    const long long r = (long long)blockIdx.x * 256 + threadIdx.x;
    if (r >= n_rows) return;
    const int start = indptr[r], end = indptr[r + 1];
    const int col = (int)(blockIdx.y + 1) * width;           // (below 2^31: a column of the matrix)
    int lo = start, hi = end - start > long_row ? start : end;
    while (lo < hi) {
        const int mid = lo + ((hi - lo) >> 1);
        if (indices[mid] < col) lo = mid + 1;
        else hi = mid;
    }
    bounds[(size_t)blockIdx.y * n_rows + r] = lo;
}

// Rows of more than kCsrChunkedRow entries, cut into chunks.  counters: chunks, rows, entries of the longest.
__global__ void __launch_bounds__(256)
csr_long_rows_kernel(const int32_t* __restrict__ indptr, long long n_rows, int2* __restrict__ chunks, int4* __restrict__ rows,
                     int* __restrict__ counters) {
    const long long r = (long long)blockIdx.x * 256 + threadIdx.x;
    if (r >= n_rows) return;
    const int start = indptr[r], len = indptr[r + 1] - start;
    if (len <= kCsrChunkedRow) return;
    const int n = lf::chunks_of(len, kCsrChunk);
    const int at = atomicAdd(&counters[0], n), row = atomicAdd(&counters[1], 1);
    atomicMax(&counters[2], len);
    rows[row] = make_int4((int)r, at, n, 0);
    for (int i = 0; i < n; ++i) chunks[at + i] = make_int2(start + i * kCsrChunk, min(kCsrChunk, len - i * kCsrChunk));
}

// Adds up the partial rows of a long row: blocks of threads over the features take partial rows k, k + blocks, ..., and their sums are
// added in block order.
constexpr int kFinalThreads = 256;
__global__ void __launch_bounds__(kFinalThreads)
csr_finalize_kernel(const int4* __restrict__ rows, const float* __restrict__ partials, float* __restrict__ C, int ld) {
    __shared__ float4 s_sum[kFinalThreads];
    const int4 row = rows[blockIdx.x];
    const int quads = ld / 4, blocks = kFinalThreads / quads;         // ld is a multiple of 32, 1024 at most
    const int block = threadIdx.x / quads, f = threadIdx.x % quads;
    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
    if (block < blocks) {
        const float4* from = reinterpret_cast<const float4*>(partials + (size_t)row.y * ld) + f;
#pragma unroll 4
        for (int k = block; k < row.z; k += blocks) {
            const float4 x = from[(size_t)k * quads];
            sum.x += x.x; sum.y += x.y; sum.z += x.z; sum.w += x.w;
        }
    }
    s_sum[threadIdx.x] = sum;
    __syncthreads();
    if (block != 0) return;
    for (int k = 1; k < blocks; ++k) {
        const float4 x = s_sum[k * quads + f];
        sum.x += x.x; sum.y += x.y; sum.z += x.z; sum.w += x.w;
    }
    reinterpret_cast<float4*>(C + (size_t)row.x * ld)[f] = sum;
}

// A sub-wave's entries of an average row at most.  One batch of gathers (half or twice as many: 1 - 7 % slower; 17K power-law
// rows of 3, N = 64 8.4 us, a batch and a half 9.7).  But where B is past the memory-side cache too, what counts is how
// many gathers are in flight, and two sub-waves on a row of nine leave half of theirs empty: a batch and a half.  1.8M rows of
// 9.6 and 8.8, N = 96: 1190 and 1162 us, 1250 and 1194 with one batch (1150 and 1128 with a sub-wave streaming over the ends of
// rows); 1.1M of 8.6, N = 192 1316, 1348, 1311.  (B of 53 to 210 MB: 500K rows of 9, N = 32 101 and 96; 147K of 11, N = 384 367
// and 354.)
constexpr unsigned long long kMallBytes = 256ull << 20;
int csr_share(unsigned long long b_bytes) { return b_bytes > kMallBytes ? kUnroll * 3 / 2 : kUnroll; }

using CsrFn = void (*)(CsrArgs, CsrMore);

template <int LPR, int CH, bool MORE> CsrFn csr_kernel(int dtype, bool wide) {
    if (dtype == LF_DTYPE_BF16) return wide ? csr_spmm_kernel<LPR, CH, bf16_t, true, MORE> : csr_spmm_kernel<LPR, CH, bf16_t, false, MORE>;
    return wide ? csr_spmm_kernel<LPR, CH, float, true, MORE> : csr_spmm_kernel<LPR, CH, float, false, MORE>;
}

template <bool MORE> CsrFn csr_kernel(int lpr, int ch, int dtype, bool wide) {
    if (ch == 2) return csr_kernel<64, 2, MORE>(dtype, wide);
    if (ch == 4) return csr_kernel<64, 4, MORE>(dtype, wide);
    return lpr == 8 ? csr_kernel<8, 1, MORE>(dtype, wide) : lpr == 16 ? csr_kernel<16, 1, MORE>(dtype, wide)
         : lpr == 32 ? csr_kernel<32, 1, MORE>(dtype, wide) : csr_kernel<64, 1, MORE>(dtype, wide);
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

// Panels.  Where a matrix uses a row of B often and a slice of B is far larger than an L2, the columns are cut into panels, a launch to
// each: the panel's part of a slice of B is about what an L2 holds.  A row's panels are looked up first (csr_bounds_kernel, 8 us), all
// but the first launch add to C.  The price of a panel is that of its slices, of the additions to C and of the rows' starts; panels
// are taken where they are 10 % cheaper.  us, without -> with: 82.9K rows of 91, N = 480 1682 -> 1140; 139K of 135, N = 224 1772 -> 1290;
// 154K of 144, N = 160 1930 -> 1290; 65.7K of 131, N = 384 1525 -> 898; 183K of 118, N = 384 4165 -> 3330.  Where they would lose: 333K
// of 13, N = 480 1210, in two 1350; 253K of 14, N = 160 326, 351.  (A hyb plan, whose partitions hold their rows by length, takes 850,
// 960, 930 and 820 for the first four.)  Rows share a sub-wave up to two batches here: 3 to 8 % better.
// Not below kPanelMinUs of price, where the launches cost what they save: 57K of 28, N = 64 41.4, in two 62.9; 57K of 60, N = 64 75.1, 90.9; 120K of
// 28, N = 64 111, 118; 24K of 60, N = 128 53.8, 63.2; beyond it 65K of 153, N = 64 320 -> 212, 200K of 60, N = 64 404 -> 377.
// Where few rows meet a B that the eight L2s nearly hold together (32 MB) they have to be 21 % cheaper: one launch is faster than its price there,
// and the tails of several count.  Price and us of one launch, in panels: 5790 rows of 170, N = 704, B of 26 MB 0.88, 153, 187; 6785 of 263, N =
// 960, 31 MB 0.81, 324, 383; 11,060 of 164, N = 480, 39 MB 0.84, 194, 207; but 18,984 of 256, N = 320, 37 MB 0.72, 443, 310; 11,316 of 133, N = 608, 36
// MB 0.77, 255, 203.  On the other side of both lines: 8834 of 127, N = 992, 49 MB 0.81, 258, 209; 52.7K of 239, N = 128, 33 MB 0.74, 572, 423; 125K of
// 290, N = 64, 24 MB 0.67, 955, 712.  92 products that are 10 % cheaper: 12 of them were slower, up to 22 %; of the 78 that remain none.
//
// Long rows.  A row is summed by the four wavefronts of a workgroup at most, a batch (8 entries where a wavefront has eight sub-waves, 16
// otherwise) to every sub-wave at a time, each 0.35 or 0.6 us behind the one before.  Where the longest row takes 10 us more than 0.02 of the
// product's price (0.15 in panels: 9000 rows of 184, longest 5018, N = 800 355 us, with chunks 399), rows of more than kCsrChunkedRow entries are cut into chunks, a workgroup to each, and a second kernel adds up their sums; the 10 us
// are that launch, the allocation of the work space and a larger kernel, 5 to 8 us together, and what a tail of that length hides behind
// anyway.  Up to kFewOfACu workgroups to a CU all start at once, and what counts is how many the fullest CU has: where chunks raise
// that the price goes up with it.  us, without -> with: 116K power-law rows, longest 6613, N = 352 212 -> 127; 150K, 13,000, N = 320 299 -> 149; 9K,
// 10,951, N = 672 90.3 -> 30.8; 2932 rows of 311, 5251, N = 128 38 -> 27.  On the other side of the lines: 16K power-law rows, 2636, N = 64 11.3, with
// chunks 15.9; 21K, 5468, N = 256 24.5, 32.7; 57K rows of 28, 1000, N = 64 40.9, 46; 2000 rows of 90, 1528, N = 800, two workgroups to a CU
// and with chunks three, 44.3, 54.1.  860 products of 2000 to 200,000 rows, N = 32 .. 1024, both ways: the 196 that take chunks take 0.74 of the time, four of
// them 1.01 to 1.05.
struct CsrShape {
    int rows_per_group = 0, panels = 1, width = 0;
    int64_t n_groups = 0, n_chunks = 0;
    Slices slices;
};
// longest: entries of the longest row (0: not known); counts: chunks, rows they are cut from, entries of the longest (null: no chunks)
CsrShape csr_shape(int64_t num_rows, int64_t num_cols, int64_t nnz, int64_t span, int feat, int dtype, int64_t longest, const int64_t* counts, bool may_panel) {
    constexpr double kPanelMinUs = 150.0, kPanelUs = 7.0, kBoundsUs = 8.0, kRowUs = 1e-4, kBytesOfC = 7e6, kWorth = 0.9, kWorthOfFew = 0.79;
    constexpr int kUsesOfB = 16;
    constexpr int64_t kPanelBytesOfB = 40'000'000;
    CsrShape shape;
    shape.width = (int)num_cols;
    const int price_rows = num_rows >= lf::kCsrManyRows ? lf::kCsrRowsMany : lf::kCsrRowsFew;
    auto priced = [&](int panels) {
        return csr_slices(num_rows, price_rows, lf::ceil_div(num_rows, (int64_t)price_rows), lf::ceil_div(num_cols, (int64_t)panels), nnz / panels, span, feat,
                          dtype);
    };
    shape.slices = priced(1);
    double least = shape.slices.us;
    const bool large = num_rows >= lf::kCsrManyRows || num_cols * feat * (dtype == LF_DTYPE_BF16 ? 2 : 4) >= kPanelBytesOfB;
    if (may_panel && least > kPanelMinUs && nnz > kUsesOfB * num_cols && !is_near((double)span, num_cols)) {
        const double one = least;
        for (int panels : {2, 3, 4, 6, 8}) {
            const Slices x = priced(panels);
            const double us = panels * x.us + kBoundsUs + (panels - 1) * ((double)num_rows * feat * 8.0 / kBytesOfC + kPanelUs + kRowUs * (double)num_rows * x.n);
            if (us < least && us < (large ? kWorth : kWorthOfFew) * one) {
                least = us;
                shape.slices = x;
                shape.panels = panels;
                shape.width = (int)lf::ceil_div(num_cols, (int64_t)panels);
            }
        }
    }
    shape.rows_per_group = lf::csr_rows_of_group(num_rows, nnz, longest, shape.panels);
    shape.n_groups = lf::ceil_div(num_rows, (int64_t)shape.rows_per_group);
    int lpr, ch;
    if (counts && counts[0] > 0 && feature_shape(shape.slices.feat, dtype, &lpr, &ch) == LF_OK) {
        const int batch = lpr < 16 ? lpr : 16;
        const double batches = (double)counts[2] * lpr / (kCsrThreads * batch);
        const double per_cu = (double)shape.slices.n / (kXcds * kCusOfXcd), of_a_cu = (double)shape.n_groups * per_cu;
        const double fuller = of_a_cu <= kFewOfACu ? std::ceil((double)(shape.n_groups + counts[0]) * per_cu) / std::ceil(of_a_cu) - 1.0 : 0.0;
        if ((lpr < 16 ? kSmallBatchUs : kBatchUs) * batches > kFinalUs + ((shape.panels > 1 ? kPanelTail : kTail) + fuller) * least) shape.n_chunks = counts[0];
    }
    return shape;
}

__global__ void csr_clear_kernel(int* counters) {
    if (threadIdx.x < 3) counters[threadIdx.x] = 0;
}

// The list of long rows: counters, rows (row, first chunk, chunks), chunks (first entry, entries).
struct ListLayout {
    int* counters;
    int4* rows;
    int2* chunks;
    size_t bytes;
    ListLayout(void* base, int64_t nnz) {
        const size_t most_rows = (size_t)(nnz / (kCsrChunkedRow + 1)) + 1, most_chunks = (size_t)(nnz / kCsrChunk) + most_rows;
        counters = (int*)base;
        rows = (int4*)((char*)base + 16);
        chunks = (int2*)((char*)base + 16 + most_rows * sizeof(int4));
        bytes = 16 + most_rows * sizeof(int4) + most_chunks * sizeof(int2);
    }
};

size_t work_bytes_of(const CsrShape& shape, int64_t num_rows, int feat) {
    return ((size_t)shape.n_chunks * feat + (size_t)(shape.panels - 1) * num_rows) * 4;       // partial rows, bounds of the panels
}

}  // namespace

extern "C" {

int lf_csr_long_rows(const int32_t* d_indptr, int64_t num_rows, int64_t nnz, void* d_list, size_t list_bytes, int64_t* h_counts, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(d_indptr && h_counts && d_list, LF_ERR_INVALID, "null argument");
    LF_REQUIRE(list_bytes >= lf_csr_long_rows_bytes(nnz), LF_ERR_INVALID, "the list needs %zu bytes", lf_csr_long_rows_bytes(nnz));
    const ListLayout l(d_list, nnz);
    csr_clear_kernel<<<1, 64, 0, s>>>(l.counters);
    LF_HIP(hipGetLastError());
    if (num_rows > 0) {
        csr_long_rows_kernel<<<(unsigned)lf::ceil_div(num_rows, 256), 256, 0, s>>>(d_indptr, num_rows, l.chunks, l.rows, l.counters);
        LF_HIP(hipGetLastError());
    }
    int h[3];
    LF_HIP(lf::read_back(h, l.counters, sizeof(h), s));
    for (int i = 0; i < 3; ++i) h_counts[i] = h[i];
    return LF_OK;
}

size_t lf_csr_long_rows_bytes(int64_t nnz) { return ListLayout(nullptr, nnz).bytes; }

int64_t lf_csr_spmm_work_bytes(int64_t num_rows, int64_t num_cols, int64_t nnz, int64_t span, const int64_t* h_counts, int64_t longest,
                               int32_t feat_size, int32_t b_dtype) {
    int lpr, ch;
    if (num_rows <= 0 || num_cols < 1 || feature_shape(feat_size, b_dtype, &lpr, &ch) != LF_OK) return 0;
    const int64_t guess[3] = {longest / kCsrChunk, 1, longest};                // (chunks at least)
    const bool unknown = !h_counts && longest > kCsrChunkedRow;
    const CsrShape shape = csr_shape(num_rows, num_cols, nnz, span, feat_size, b_dtype, h_counts ? h_counts[2] : longest, unknown ? guess : h_counts, true);
    if (unknown && shape.n_chunks > 0) return -1;
    return (int64_t)work_bytes_of(shape, num_rows, feat_size);
}

}  // extern "C"

namespace {

// (longest: see lf_csr_spmm_trusted_rows; negative: the product takes what it is given)
int csr_product(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values, int64_t num_rows, int64_t num_cols, int64_t nnz,
                int64_t span, int64_t longest, const void* d_list, const int64_t* h_counts, void* d_work, size_t work_bytes, int32_t feat_size,
                int32_t b_dtype, const void* d_B, float* d_C, hipStream_t s) {
    LF_REQUIRE(num_rows >= 0 && num_rows < (1ll << 31) && num_cols >= 1, LF_ERR_INVALID, "bad shape");
    if (num_rows == 0) return LF_OK;
    LF_REQUIRE(d_indptr && d_B && d_C, LF_ERR_INVALID, "null argument");
    LF_REQUIRE(b_dtype == LF_DTYPE_F32 || b_dtype == LF_DTYPE_BF16, LF_ERR_INVALID, "unknown B dtype %d", b_dtype);
    LF_REQUIRE((uintptr_t)d_B % 16 == 0 && (uintptr_t)d_C % 16 == 0 && (uintptr_t)d_work % 16 == 0, LF_ERR_INVALID,
               "B, C and the work space must be 16-byte aligned");
    int lpr, ch;
    if (int rc = feature_shape(feat_size, b_dtype, &lpr, &ch)) return rc;
    const bool ask = longest >= 0;
    const int64_t guess[3] = {longest > kCsrChunkedRow ? longest / kCsrChunk : 0, 1, longest};       // (chunks at least)
    const CsrShape shape = csr_shape(num_rows, num_cols, nnz, span, feat_size, b_dtype, ask ? longest : h_counts ? h_counts[2] : 0,
                                     ask ? guess : d_work && d_list ? h_counts : nullptr, ask || d_work != nullptr);
    if (ask && work_bytes_of(shape, num_rows, feat_size) > 0) return LF_WANTS_WORK;
    const int64_t n_chunks = shape.n_chunks;
    LF_REQUIRE(!d_work || work_bytes >= work_bytes_of(shape, num_rows, feat_size), LF_ERR_INVALID, "the product needs %zu bytes of work space",
               work_bytes_of(shape, num_rows, feat_size));
    CsrArgs a{};
    a.rows_per_group = shape.rows_per_group;
    a.n_groups = shape.n_groups;
    a.feat = shape.slices.feat;
    a.parts = shape.slices.parts;
    if (int rc = feature_shape(a.feat, b_dtype, &lpr, &ch)) return rc;
    a.indices = d_indices;
    a.values = d_values;
    a.n_rows = num_rows;
    a.ld = feat_size;
    a.B = d_B;
    a.C = d_C;
    a.b_bytes = (unsigned long long)num_cols * feat_size * (b_dtype == LF_DTYPE_BF16 ? 2 : 4);
    a.share = shape.panels > 1 ? 2 * kUnroll : csr_share(a.b_bytes);
    const bool wide = a.b_bytes > kPastB;
    CsrMore more{};
    more.long_row = n_chunks > 0 ? kCsrChunkedRow : 0x7FFFFFFF;
    more.n_chunks = (int)n_chunks;
    const ListLayout list(const_cast<void*>(d_list), nnz);
    more.chunks = list.chunks;
    more.partials = (float*)d_work;
    int32_t* bounds = (int32_t*)((float*)d_work + (size_t)n_chunks * feat_size);
    if (shape.panels > 1) {
        csr_bounds_kernel<<<dim3((unsigned)lf::ceil_div(num_rows, 256), (unsigned)(shape.panels - 1)), 256, 0, s>>>(
            d_indptr, d_indices, num_rows, shape.width, more.long_row, bounds);
        LF_HIP(hipGetLastError());
    }
    const CsrFn kernel = shape.panels > 1 || n_chunks > 0 ? csr_kernel<true>(lpr, ch, b_dtype, wide) : csr_kernel<false>(lpr, ch, b_dtype, wide);
    for (int p = 0; p < shape.panels; ++p) {
        const bool last = p + 1 == shape.panels;
        a.starts = p == 0 ? d_indptr : bounds + (size_t)(p - 1) * num_rows;
        more.ends = last ? d_indptr + 1 : bounds + (size_t)p * num_rows;
        more.flags = (p > 0 ? kAccumulateC : 0) | (last ? kStreamC : 0);
        if (p > 0) more.n_chunks = 0;
        long long longest = 0;
        for (int x = 0; x < kXcds; ++x) longest = std::max(longest, part_tiles(a.parts, x, a.n_groups) + part_tiles(a.parts, x, more.n_chunks));
        LF_REQUIRE(longest * kXcds < (1ll << 31), LF_ERR_UNSUPPORTED, "too many rows");
        kernel<<<(unsigned)(longest * kXcds), kCsrThreads, (kCsrThreads / 64) * a.feat * sizeof(float), s>>>(a, more);
        LF_HIP(hipGetLastError());
    }
    if (n_chunks > 0) {
        csr_finalize_kernel<<<(unsigned)h_counts[1], kFinalThreads, 0, s>>>(list.rows, more.partials, d_C, feat_size);
        LF_HIP(hipGetLastError());
    }
    return LF_OK;
}

}  // namespace

extern "C" {

int lf_csr_spmm_trusted_work(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values,
                             int64_t num_rows, int64_t num_cols, int64_t nnz, int64_t span, const void* d_list, const int64_t* h_counts,
                             void* d_work, size_t work_bytes, int32_t feat_size,
                             int32_t b_dtype, const void* d_B, float* d_C, lf_stream_t stream) {
    return csr_product(d_indptr, d_indices, d_values, num_rows, num_cols, nnz, span, -1, d_list, h_counts, d_work, work_bytes, feat_size, b_dtype,
                       d_B, d_C, (hipStream_t)stream);
}

int lf_csr_spmm_trusted_rows(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values,
                             int64_t num_rows, int64_t num_cols, int64_t nnz, int64_t span, int64_t longest, int32_t feat_size,
                             int32_t b_dtype, const void* d_B, float* d_C, lf_stream_t stream) {
    LF_REQUIRE(longest >= 0, LF_ERR_INVALID, "bad length of the longest row");
    return csr_product(d_indptr, d_indices, d_values, num_rows, num_cols, nnz, span, longest, nullptr, nullptr, nullptr, 0, feat_size, b_dtype, d_B, d_C,
                       (hipStream_t)stream);
}

int lf_csr_spmm_trusted_span(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values,
                             int64_t num_rows, int64_t num_cols, int64_t nnz, int64_t span, int32_t feat_size,
                             int32_t b_dtype, const void* d_B, float* d_C, lf_stream_t stream) {
    return csr_product(d_indptr, d_indices, d_values, num_rows, num_cols, nnz, span, -1, nullptr, nullptr, nullptr, 0, feat_size, b_dtype, d_B, d_C,
                       (hipStream_t)stream);
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
    if (int rc = lf::csr_check(d_indptr, d_indices, nullptr, num_rows, num_cols, nnz, d_scratch, nullptr, &span, nullptr, "lf_csr_spmm",
                               (hipStream_t)stream))
        return rc;
    return lf_csr_spmm_trusted_span(d_indptr, d_indices, d_values, num_rows, num_cols, nnz, span, feat_size, b_dtype, d_B, d_C, stream);
}

}  // extern "C"
