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

// Chunks of at most `chunk` entries that a row of `len` > 0 entries is cut into.
constexpr int chunks_of(int len, int chunk) { return (len - 1) / chunk + 1; }

}  // namespace lf
#endif
