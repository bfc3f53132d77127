// Block-sparse (BSR, square blocks of 16, 32 or 64) fp16 SpMM on the gfx950 matrix cores:
//     Y[mb*BS][F] (fp16) = A_bsr (fp16 blocks) . X[nb*BS][F] (fp16),  fp32 accumulation.
//
// Takes over the kernel that bench_bsrmm builds through SparseTIR/TVM with fp16 WMMA
// 16x16x16 fragments (playground_pipline/format_algos.py:1182-1643; any block size that is a
// multiple of 16 there, format_algos.py:1581-1582; 32 is what the driver passes,
// proc05.spmm.end-to-end.py:205).  This is the one place of the library where dense-block
// matrix-core work is the right shape; it is still bound by memory (2 KiB of A and 32 rows of X
// per 32x32xF block product: ~26 flop/byte at F = 128), so the kernel is organised around
// keeping wide, coalesced loads in flight.
//
// A wavefront owns one block row and 16 VF features (VF = 8, 4 or 2) and needs neither LDS nor barriers.  It uses
// v_mfma_f32_16x16x32_f16, whose B operand is eight k (rows of X) of one column per lane:
//   * lane (kq = lane / 16, li = lane % 16) loads the rows k = 8 kq .. 8 kq + 7 of X at the
//     features VF li .. VF li + VF - 1, 16 bytes each with VF = 8: every load instruction reads four whole
//     256-byte pieces of rows of X;
//   * which column of the instruction a feature takes is free, so instruction f = 0 .. VF - 1 is
//     given the features VF li + f: the eight k of one of a lane's features are the same
//     half of the same word of its eight loads, put together by four v_perm_b32;
//   * the results of the instructions are then VF consecutive features of a row in
//     one lane, which stores them together.
// A operands are 16 bytes of a row of the block (8 kq ..), read in memory order.  Blocks of 16 are
// taken in pairs - the upper half of the wavefront (kq >= 2) works on the second one -, blocks of 64 in two
// steps of 32 columns.  The loads of the next step are under way during the products of this one.
// The kernel before this transposed X through LDS in 2-byte stores, with a barrier and one block's
// loads in flight per workgroup.  Both in turn on one GPU: 1M x 1M, 8 blocks per block row, N = 128, blocks
// of 16 / 32 / 64: 0.514 / 0.397 / 0.519 -> 0.360 / 0.393 / 0.497 ms, N = 256, blocks of 32: 0.842 -> 0.712
// (all at 7 TB/s of A blocks and rows of X, what a gather that misses the L2s reaches); 40K x 40K, blocks of 16,
// N = 200: 44 -> 19.5 us, blocks of 32, N = 128: 18.8 -> 14.0.  It loses where block rows are very short:
// 800K x 800K, 2 blocks of 32 a row, N = 128: 102 -> 106.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <algorithm>

#include "lf_internal.h"
#include "lf_rules.h"

namespace {

constexpr int kFeatTile = 128;     // features per wavefront at most

// Wavefronts per workgroup; they are independent of each other.  Up to kFewUnits of them go out one by one, which
// spreads them over the CUs (40K x 40K, blocks of 32, N = 128: 15.9 -> 14.5 us, N = 24 10.5 -> 9.5);
// otherwise four, so that the feature tiles of a block row share its blocks in the L1.  Where a
// product is bound by memory throughout - large, whole tiles of features, long block rows - eight that
// start together move more.  Four against eight in turn on one GPU, 15 shapes of 262K to 1M rows, 6 to 24
// blocks a row, N = 128 .. 512: 0.9 to 7.4 % faster each (1M x 1M, 8 blocks a row, N = 128, blocks of 32 / 16: 405.8 /
// 372.5 -> 395.4 / 364.9 us; 800K x 800K, 7 blocks of 16, N = 384: 709.5 -> 660.7); with short block rows
// the CU waits for the last of eight (800K x 800K, 2 blocks a row, N = 128: 105 -> 110).  Two such workgroups
// of blocks of 64 would not have the registers.
constexpr long long kFewUnits = 4096;
constexpr int kLongBlockRow = 6;       // blocks
constexpr int most_threads(int block) { return block == 64 ? 256 : 512; }

// A Y of this size or more is stored past the caches, which leaves them to X (128K x 128K, blocks of 32,
// N = 512: 104 -> 96 us; 1M x 1M, N = 256: 759 -> 734); a smaller one the next operation may find there.
constexpr int64_t kStreamYBytes = 64ll << 20;

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// A block row of 64 is two steps a block, one after the other, and few block rows leave CUs idle: two wavefronts share each
// then, and the second one's sums go through LDS.  us, alone -> by two: 100 block rows of 10, F = 32 6.9 -> 6.4, F = 64 9.6 ->
// 8.1; 400 of 10, F = 16 / 48 10.3 / 14.3 -> 9.3 / 12.1, F = 128 18.9 -> 17.0; 800 of 10, F = 48 19.5 -> 22.0.
// Up to 256 block rows, features in tiles of 64 as well: 200 of 10, F = 128 12.2 -> 12.0, 100 10.7 -> 8.2 (400: 17.0, 22.1).
constexpr long long kPairedRows = 512, kPairedNarrowRows = 256;
constexpr int kPairedBlocks = 4;

// VF consecutive features of a row, as they are loaded and stored.
template <int VF> struct Feats;
template <> struct Feats<8> { typedef uint32_t vec __attribute__((ext_vector_type(4))); };
template <> struct Feats<4> { typedef uint32_t vec __attribute__((ext_vector_type(2))); };
template <> struct Feats<2> { typedef uint32_t vec __attribute__((ext_vector_type(1))); };

// What a wavefront loads for one step of 32 columns of A: eight rows of X and a row of each of A's
// row tiles per lane.
template <int BS, int VF> struct BsrStep {
    static constexpr int kTiles = BS / 16;
    typename Feats<VF>::vec x[8];
    uint4 a[kTiles];
};

// TWO: both wavefronts of a workgroup share a block row (blocks of 64; an argument instead cost the others 1 %).
template <int BS, int VF, bool TWO>
__global__ void __launch_bounds__(TWO ? 128 : most_threads(BS))
bsr_spmm_kernel(const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices,
                const _Float16* __restrict__ data, const _Float16* __restrict__ X,
                _Float16* __restrict__ Y, int feat, int n_tiles, long long n_units, int stream_y) {
    constexpr int RT = BS / 16;                          // row tiles of a block row
    constexpr int SPB = BS == 64 ? 2 : 1;                // steps per block
    constexpr int BPS = BS == 16 ? 2 : 1;                // blocks per step
    using Vec = typename Feats<VF>::vec;
    __shared__ float4_t s_part[TWO ? RT * VF * 64 : 1];  // sums of the second wavefront
    const int lane = threadIdx.x & 63, li = lane & 15, kq = lane >> 4;
    // the feature tiles of a block row go to neighbouring wavefronts, which read the same blocks of A
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long unit = TWO ? (long long)blockIdx.x : (long long)blockIdx.x * (blockDim.x / 64) + wave;
    if (unit >= n_units) return;
    const int brow = (int)(unit / n_tiles);
    const int f = (int)(unit % n_tiles) * (16 * VF) + VF * li;
    const bool on = f < feat;                            // feat is a multiple of 8: a vector is inside or outside
    int jb = indptr[brow], je = indptr[brow + 1];
    if constexpr (TWO) {
        const int mid = jb + (je - jb + 1) / 2;
        jb = wave ? mid : jb;
        je = wave ? je : mid;
    }

    float4_t acc[RT][VF];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int i = 0; i < VF; ++i) acc[t][i] = float4_t{0.f, 0.f, 0.f, 0.f};

    const int n_steps = BPS == 2 ? (je - jb + 1) / 2 : (je - jb) * SPB;
    // Every load below is unconditional - lanes past the last feature read what the tile's first lane
    // reads, steps past the end the last block - so that the wait for one step's loads need not
    // allow for a path on which the next step's were not issued.
    const int f_in = on ? f : f - VF * li;
    // step s: block jb + s / SPB, columns 32 * (s % SPB) ..; or blocks jb + 2 s and jb + 2 s + 1
    auto block_of = [&](int s, int half) { return min(BPS == 2 ? jb + 2 * s + half : jb + s / SPB, je - 1); };
    struct Cols { int c0, c1; };
    auto cols_of = [&](int s) { return Cols{indices[block_of(s, 0)], BPS == 2 ? indices[block_of(s, 1)] : 0}; };
    auto load = [&](int s, Cols c, BsrStep<BS, VF>& st) {
        const bool second = BPS == 2 && kq >= 2;
        const int k0 = BPS == 2 ? 8 * (kq & 1) : 32 * (s % SPB) + 8 * kq;
        const _Float16* src = X + ((size_t)(second ? c.c1 : c.c0) * BS + k0) * feat + f_in;
#pragma unroll
        for (int r = 0; r < 8; ++r) st.x[r] = *reinterpret_cast<const Vec*>(src + (size_t)r * feat);
        const int j = second ? block_of(s, 1) : block_of(s, 0);
        const _Float16* blk = data + (size_t)j * BS * BS + li * BS + k0;
#pragma unroll
        for (int t = 0; t < RT; ++t) st.a[t] = *reinterpret_cast<const uint4*>(blk + 16 * t * BS);
    };
    // An odd last block of 16 has no partner: the half of the wavefront that read the block once more adds
    // nothing.  Both operands are cleared: 0 * Inf is NaN whichever of them is infinite.
    auto drop_missing = [&](BsrStep<BS, VF>& st) {
        if (BPS == 2 && kq >= 2 && ((je - jb) & 1)) {
            st.a[0] = make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 8; ++r) st.x[r] = Vec{};
        }
    };
    auto multiply = [&](const BsrStep<BS, VF>& st) {
#pragma unroll
        for (int i = 0; i < VF; ++i) {                   // feature f + i
            union { uint32_t w[4]; half8_t h; } b;
            const uint32_t sel = i & 1 ? 0x07060302u : 0x05040100u;
#pragma unroll
            for (int q = 0; q < 4; ++q) b.w[q] = __builtin_amdgcn_perm(st.x[2 * q + 1][i >> 1], st.x[2 * q][i >> 1], sel);
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                union { uint4 w; half8_t h; } a;
                a.w = st.a[t];
                acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.h, b.h, acc[t][i], 0, 0, 0);
            }
        }
    };
    if (n_steps > 0) {
        BsrStep<BS, VF> s0, s1;
        Cols even = cols_of(0), odd = cols_of(1);
        load(0, even, s0);
        int s = 0;
        for (; s + 2 < n_steps; s += 2) {
            load(s + 1, odd, s1);
            even = cols_of(s + 2);
            multiply(s0);
            load(s + 2, even, s0);
            odd = cols_of(s + 3);
            multiply(s1);
        }
        if (s + 1 < n_steps) {
            load(s + 1, odd, s1);
            multiply(s0);
            drop_missing(s1);
            multiply(s1);
        } else {
            drop_missing(s0);
            multiply(s0);
        }
    }
    if constexpr (TWO) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int i = 0; i < VF; ++i)
                if (wave) s_part[(t * VF + i) * 64 + lane] = acc[t][i];
        __syncthreads();
        if (wave) return;
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int i = 0; i < VF; ++i) acc[t][i] += s_part[(t * VF + i) * 64 + lane];
    }

    // D layout of the instruction: lane holds column li, rows 4 kq + v
    if (!on) return;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            union { _Float16 h[VF]; Vec w; } o;
#pragma unroll
            for (int i = 0; i < VF; ++i) o.h[i] = (_Float16)acc[t][i][v];
            Vec* dst = reinterpret_cast<Vec*>(Y + ((size_t)brow * BS + 16 * t + 4 * kq + v) * feat + f);
            // (through an integer, or the compiler folds the two stores into one ordinary store)
            if (stream_y)
                __builtin_nontemporal_store(o.w, reinterpret_cast<Vec __attribute__((address_space(1)))*>(reinterpret_cast<uintptr_t>(dst)));
            else
                *dst = o.w;
        }
}

using BsrFn = void (*)(const int32_t*, const int32_t*, const _Float16*, const _Float16*, _Float16*, int, int, long long, int);
template <int BS, bool TWO> BsrFn bsr_kernel(int vf) {
    return vf == 8 ? bsr_spmm_kernel<BS, 8, TWO> : vf == 4 ? bsr_spmm_kernel<BS, 4, TWO> : bsr_spmm_kernel<BS, 2, TWO>;
}

}  // namespace

extern "C" {

int lf_bsr_spmm_trusted_nnz(const int32_t* d_indptr, const int32_t* d_indices, const void* d_data,
                            int64_t num_block_rows, int64_t num_block_cols, int64_t nnz_blocks, int32_t block_size,
                            int32_t feat_size, const void* d_X, void* d_Y, lf_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    LF_REQUIRE(block_size == 16 || block_size == 32 || block_size == 64, LF_ERR_UNSUPPORTED,
               "blocks of 16, 32 or 64 rows and columns are supported (got %d)", block_size);
    LF_REQUIRE(num_block_rows >= 0 && num_block_rows < (1ll << 26) && num_block_cols >= 1 &&
                   num_block_cols < (1ll << 26), LF_ERR_INVALID, "bad block shape");
    LF_REQUIRE(feat_size >= 8 && feat_size % 8 == 0, LF_ERR_UNSUPPORTED,
               "feat_size must be a positive multiple of 8 (got %d)", feat_size);
    if (num_block_rows == 0) return LF_OK;
    LF_REQUIRE(d_indptr && d_X && d_Y, LF_ERR_INVALID, "null argument");
    LF_REQUIRE((uintptr_t)d_X % 16 == 0 && (uintptr_t)d_Y % 16 == 0 && (uintptr_t)d_data % 16 == 0, LF_ERR_INVALID,
               "X, Y and the block data must be 16-byte aligned");
    const bool few_blocks = nnz_blocks < kPairedBlocks * num_block_rows;      // (also where their number is not known)
    const long long tiles_of_128 = lf::ceil_div(feat_size, kFeatTile);
    const bool paired = block_size == 64 && num_block_rows * tiles_of_128 <= kPairedRows && !few_blocks;
    const int vf = paired && feat_size > 64 && num_block_rows * tiles_of_128 <= kPairedNarrowRows ? 4 : lf::bsr_lane_features(feat_size, block_size, num_block_rows, nnz_blocks);
    const int n_tiles = (int)lf::ceil_div(feat_size, 16 * vf);
    const long long units = (long long)num_block_rows * n_tiles;
    const bool stream_y = (int64_t)num_block_rows * block_size * feat_size * 2 >= kStreamYBytes;
    const bool eight = block_size != 64 && stream_y && feat_size % kFeatTile == 0 && nnz_blocks >= kLongBlockRow * num_block_rows;
    const int threads = paired ? 128 : n_tiles == 1 && units <= kFewUnits ? 64 : eight ? 512 : 256;
    const long long groups = paired ? units : lf::ceil_div(units, threads / 64);
    LF_REQUIRE(groups < (1ll << 31), LF_ERR_UNSUPPORTED, "too many block rows and features");
    const _Float16* data = (const _Float16*)d_data;
    const _Float16* X = (const _Float16*)d_X;
    _Float16* Y = (_Float16*)d_Y;
    const BsrFn kernel = block_size == 16 ? bsr_kernel<16, false>(vf) : block_size == 32 ? bsr_kernel<32, false>(vf)
                         : paired ? bsr_kernel<64, true>(vf) : bsr_kernel<64, false>(vf);
    kernel<<<(unsigned)groups, threads, 0, s>>>(d_indptr, d_indices, data, X, Y, feat_size, n_tiles, units, stream_y);
    LF_HIP(hipGetLastError());
    return LF_OK;
}

int lf_bsr_spmm_trusted(const int32_t* d_indptr, const int32_t* d_indices, const void* d_data,
                        int64_t num_block_rows, int64_t num_block_cols, int32_t block_size,
                        int32_t feat_size, const void* d_X, void* d_Y, lf_stream_t stream) {
    return lf_bsr_spmm_trusted_nnz(d_indptr, d_indices, d_data, num_block_rows, num_block_cols, 0, block_size, feat_size,
                                   d_X, d_Y, stream);
}

int lf_bsr_spmm(const int32_t* d_indptr, const int32_t* d_indices, const void* d_data,
                int64_t num_block_rows, int64_t num_block_cols, int64_t nnz_blocks, int32_t block_size,
                int32_t feat_size, const void* d_X, void* d_Y, void* d_scratch, lf_stream_t stream) {
    LF_REQUIRE(block_size == 16 || block_size == 32 || block_size == 64, LF_ERR_UNSUPPORTED,
               "blocks of 16, 32 or 64 rows and columns are supported (got %d)", block_size);
    LF_REQUIRE(num_block_rows >= 0 && num_block_rows < (1ll << 26) && num_block_cols >= 1 &&
                   num_block_cols < (1ll << 26), LF_ERR_INVALID, "bad block shape");
    // no gather before the block index arrays have passed
    if (int rc = lf::csr_check(d_indptr, d_indices, nullptr, num_block_rows, num_block_cols, nnz_blocks, d_scratch, nullptr, nullptr, nullptr,
                               "lf_bsr_spmm", (hipStream_t)stream))
        return rc;
    return lf_bsr_spmm_trusted_nnz(d_indptr, d_indices, d_data, num_block_rows, num_block_cols, nnz_blocks, block_size,
                                   feat_size, d_X, d_Y, stream);
}

}  // extern "C"
