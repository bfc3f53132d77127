// Index arithmetic that has to stay inside 32 bits for arrays of up to 2^31 - 1 entries.  Plain constexpr functions, which a
// kernel and a host program may both call.
#ifndef LF_INDEX_H
#define LF_INDEX_H

namespace lf {

// Where the group of four slots that starts at slot q of a segment (first entry `start`) is loaded from arrays of n >= 4 entries: its
// first entry, or back from the arrays' end where it passes that.  (q runs on into the segment's padding, whose groups are loaded and
// dropped: up to 1023 past its last entry, and so past 2^31 in the last rows of a matrix of nearly that many entries.)
constexpr int group_source(int start, int q, int n) {
    const unsigned at = (unsigned)start + (unsigned)q, most = (unsigned)(n - 4);
    return (int)(at < most ? at : most);
}

// Chunks of at most `chunk` entries that a row of `len` > 0 entries is cut into.
constexpr int chunks_of(int len, int chunk) { return (len - 1) / chunk + 1; }

}  // namespace lf
#endif
