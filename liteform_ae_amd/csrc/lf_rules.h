// Rules of dispatch that need nothing but sizes.  Plain constexpr functions, which a host program may call as well.
#ifndef LF_RULES_H
#define LF_RULES_H

namespace lf {

// ---- rows to a workgroup of the CSR product
constexpr int kCsrRowsFew = 8, kCsrRowsMany = 16;
constexpr long long kCsrManyRows = 24576;
// Few long rows, some much longer than others: 2 to a workgroup, or 4 where they are more, as the last workgroups of 8 are left alone with
// their longest rows for a part of the product that counts.  8 -> 2 rows, us: 2461 rows of 367, longest 2301, N = 64 34.7 -> 21.3; 4972 of 271, 4533,
// N = 64 29.6 -> 22.7; 3025 of 227, 888, N = 192 32.5 -> 26.3; 2975 of 162, 751, N = 128 16.8 -> 15.9 (4 rows: 18.0); 12,890 of 212, 2179, N = 128, 4
// rows 71.5 -> 66.5; of one length, 4137 of 377, 703, N = 32 16.0 -> 13.5.  Beyond the lines: rows of one length, 10,026 of 276, longest 502, N = 64
// 34.4, with 2 35.3, 2840 of 214, 287, N = 160 21.4, 22.3, 4705 of 235, 530, N = 96 24.4, 25.6; more rows of less than kCsrVeryLong, 9140 of
// 107, 1051, N = 160 39.5, 40.3; 24,000 of 250, N = 96 with 2 6 % more, with 4 1; shorter ones, 2000 of 60, N = 96 as long.  295 products of
// 2000 to 17,000 rows, N = 32 .. 512: the 179 by this rule take 0.90 of the time, 5 of them 1.01 to 1.07 (6714 of 352, N = 96 1.04 with one set
// of columns, 0.81 with another).
constexpr long long kCsrFewRows = 5120, kCsrFewEvenRows = 6144, kCsrFewVeryLongRows = 12288;
constexpr int kCsrLong = 96, kCsrVeryLong = 208, kCsrEvenLong = 300;
// entries: of the rows; longest: of all their entries (0: unknown); panels: that the entries are spread over, one of which the launch is for
constexpr int csr_rows_of_group(long long rows, long long entries, long long longest, int panels) {
    if (rows >= kCsrManyRows) return kCsrRowsMany;
    const long long of_panel = entries / panels;
    if (rows <= kCsrFewEvenRows && of_panel >= kCsrEvenLong * rows) return 2;
    if (2 * longest * rows < 5 * entries) return kCsrRowsFew;                  // (no row of two and a half times the average)
    if (of_panel >= kCsrVeryLong * rows) return rows <= kCsrFewVeryLongRows ? 2 : 4;
    return rows <= kCsrFewRows && of_panel >= kCsrLong * rows ? 2 : kCsrRowsFew;
}

// ---- features to a lane of the BSR product
// Rows of X of up to 64 features fill half of the 128 that a wavefront takes with 8 to a lane, or a quarter: lanes past the last feature
// would load and multiply for nothing, in registers that other wavefronts could use (blocks of 32: 198 with 8 features,
// 102 with 4, 65 with 2).  8 features a lane -> 4 or 2, us: blocks of 32, 20,000 block rows of 4, F = 16 / 32 / 48 52.1 / 60.1 / 74.4 ->
// 37.9 / 52.7 / 64.3; of 10, F = 16 126.7 -> 90.0; blocks of 16, 22,282 block rows of 8, F = 16 34.4 -> 25.3; blocks of 64, 1500 of 10,
// F = 40 39.8 -> 29.8.  From 49 features on (57 with blocks of 32) half of the lanes or fewer are idle, and where many blocks keep the
// memory busy 4 features a lane lose to the wider loads of 8.  Inside the lines: blocks of 64, 1397 block rows of 7, F = 56 30.3 -> 24.8, of 32,
// 7757 of 8, F = 64 54.6 -> 53.5, of 16, 10,176 of 6, F = 64 24.5 -> 24.2; beyond: of 64, 1948 of 8, F = 56 37.8, 40.1; of 32, 18,331 of 5, F = 64
// 85.7, 87.9; of 16, 10,169 of 10, F = 64 34.2, 35.0.  177 products of 32,000 to 800,000 rows, F = 16 .. 64: the 155 with 4 or 2 take 0.90 of
// the time, and no more than with 8 where the kernel is longer than a call (7.5 us).  Above 64 features two tiles of 4 a lane lose up to 20 % or
// gain 4, by the sizes.
constexpr int bsr_lane_features(int feat, int block, long long block_rows, long long blocks) {       // blocks == 0: not known
    if (feat <= 32) return 2;
    if (feat > 64) return 8;
    if (feat <= 48 || (block == 32 && feat <= 56)) return 4;
    const long long most_rows = block == 16 ? 16384 : block == 32 ? (1ll << 62) : 2048, most_blocks = block == 64 ? 12288 : 65536;
    return blocks > 0 && blocks <= most_blocks && block_rows <= most_rows ? 4 : 8;
}

}  // namespace lf
#endif
