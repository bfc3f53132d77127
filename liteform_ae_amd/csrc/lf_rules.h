// Rules of dispatch that need nothing but sizes.  Plain constexpr functions, which a host program may call as well.
#ifndef LF_RULES_H
#define LF_RULES_H

namespace lf {

// ---- rows to a workgroup of the CSR product
constexpr int kCsrRowsFew = 8, kCsrRowsMany = 16;
constexpr long long kCsrManyRows = 24576;
// Few long rows, some much longer than others: 2 to a workgroup, as the last workgroups of 8 are left alone with their longest rows for a part
// of the product that counts.  8 -> 2 rows, us: 2461 rows of 367, longest 2301, N = 64 34.7 -> 21.3; 4972 of 271, 4533, N = 64 29.6 -> 22.7; 3025 of
// 227, 888, N = 192 32.5 -> 26.3; 2975 of 162, 751, N = 128 16.8 -> 15.9.  Beyond the lines: rows of one length, 10,026 of 276, longest 502,
// N = 64 34.4, with 2 35.3, 2840 of 214, 287, N = 160 21.4, 22.3; more rows, 5817 of 266, 4201, N = 32 18.5, 19.8, 9140 of 107, 1051, N = 160
// 39.5, 40.3; shorter ones, 2000 of 60, N = 96 as long.  295 products of 2000 to 17,000 rows, N = 32 .. 512: the 117 by this rule take 0.89 of the
// time, 1.01 at most.  4 rows lie between 8 and 2, but where 2 are better than 4 they can be worse than 8: 2975 rows as above 18.0.
constexpr long long kCsrFewRows = 5120;
constexpr int kCsrLongAverage = 96, kCsrUneven = 3;
// entries: of the rows; longest: of all their entries (0: unknown); panels: that the entries are spread over, one of which the launch is for
constexpr int csr_rows_of_group(long long rows, long long entries, long long longest, int panels) {
    if (rows >= kCsrManyRows) return kCsrRowsMany;
    const bool uneven = longest * rows >= kCsrUneven * entries;
    return rows <= kCsrFewRows && uneven && entries / panels >= kCsrLongAverage * rows ? 2 : kCsrRowsFew;
}

}  // namespace lf
#endif
