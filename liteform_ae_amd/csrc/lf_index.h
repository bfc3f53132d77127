// Index arithmetic that has to stay inside 32 bits for arrays of up to 2^31 - 1 entries.  Plain constexpr functions, which a
// kernel and a host program may both call.
#ifndef LF_INDEX_H
#define LF_INDEX_H

namespace lf {

// Source of the group of four slots that starts at slot q of a segment (first entry `start`, `fill` entries): the group's first
// entry, or the segment's last one where the group is padding, which is loaded and dropped.  (start + q itself passes 2^31 in
// the padding of the last rows of a matrix of nearly 2^31 entries.)
constexpr int group_source(int start, int fill, int q) {
    const int last = fill > 0 ? fill - 1 : 0;
    return start + (q < last ? q : last);
}

// A segment of `fill` >= 4 entries is walked from its entry j, a lane's four entries `ahead` (below 2^16) from there: whether they
// start inside the segment, and where they are loaded, which is back from its end where they pass it.  (j + ahead may pass
// 2^31 at the end of a segment of nearly that many entries.)
constexpr bool fours_inside(int j, int ahead, int fill) { return (unsigned)j + (unsigned)ahead < (unsigned)fill; }
constexpr int fours_source(int j, int ahead, int fill) {
    const unsigned at = (unsigned)j + (unsigned)ahead, most = (unsigned)(fill - 4);
    return (int)(at < most ? at : most);
}

}  // namespace lf
#endif
