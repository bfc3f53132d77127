// Shared helpers for liblfhip.so: error reporting and small integer utilities.
#pragma once
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>

#include "liteform_hip.h"

namespace lf {

// Thread-local message behind lf_last_error().
std::string& last_error();

int fail(int status, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

inline bool is_pow2(int64_t x) { return x > 0 && (x & (x - 1)) == 0; }
inline int ilog2(int64_t x) { return 63 - __builtin_clzll((unsigned long long)x); }
inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace lf

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
namespace lf {
// Page-locked host memory for what a call reads back from (or hands to) the GPU, on loan from a pool
// shared by all threads: a read-back of some hundred bytes and the wait for it take 14 us this way
// and 23 from pageable memory.  The pool keeps at most kPooledBuffers buffers of kPooledBytes (1 MB
// in all); a loan beyond that is allocated and freed, and a larger one uses pageable memory.  Usable
// on every device (allocated portable).  Give the loan back only when the stream has been waited for.
class PinnedLoan {
public:
    static constexpr size_t kPooledBytes = 128 << 10;
    static constexpr size_t kPooledBuffers = 8;
    explicit PinnedLoan(size_t bytes);
    ~PinnedLoan();
    PinnedLoan(const PinnedLoan&) = delete;
    PinnedLoan& operator=(const PinnedLoan&) = delete;
    template <typename T> T* as(size_t byte_offset = 0) const { return reinterpret_cast<T*>((char*)p_ + byte_offset); }
    bool ok() const { return p_ != nullptr; }
    bool pinned() const { return pinned_; }            // a kernel may read and write it

private:
    void* p_ = nullptr;
    bool pinned_ = false;
};

// Words from `up` to the GPU, `n_clear` cleared there, words from there to `down`, in one launch where the loans are pinned: a copy, a
// fill and a copy are three, 5 us each of a call that waits for them.  (A few KB of either: the kernel's loads and stores cross PCIe.)
struct Words {
    const void* from = nullptr;
    void* to = nullptr;
    size_t bytes = 0;              // a multiple of 4
};
hipError_t move_words(Words up, bool up_pinned, void* clear, size_t clear_bytes, Words down, bool down_pinned, hipStream_t s);

// A few words from the GPU, and the wait for them.
inline hipError_t read_back(void* h_dst, const void* d_src, size_t bytes, hipStream_t s) {
    PinnedLoan loan(bytes);
    if (!loan.ok()) return hipErrorOutOfMemory;
    hipError_t e = hipMemcpyAsync(loan.as<char>(), d_src, bytes, hipMemcpyDeviceToHost, s);
    const hipError_t w = hipStreamSynchronize(s);
    if (e == hipSuccess) e = w;
    if (e == hipSuccess) std::memcpy(h_dst, loan.as<char>(), bytes);
    return e;
}

// Structural check of caller-supplied CSR (or BSR block) index arrays on the GPU, behind
// lf_csr_check and in front of lf_csr_spmm / lf_bsr_spmm; `what` names the arrays in the
// error message.  h_span, h_longest (optional): see lf_csr_check_span, lf_csr_check_rows.  Synchronises `s`.
int csr_check(const int32_t* d_indptr, const int32_t* d_indices, const float* d_values, int64_t num_rows,
              int64_t num_cols, int64_t nnz, void* d_scratch, int32_t* h_flags, int64_t* h_span, int64_t* h_longest, const char* what,
              hipStream_t s);
}  // namespace lf
#endif

#define LF_REQUIRE(cond, status, ...)                  \
    do {                                               \
        if (!(cond)) return lf::fail(status, __VA_ARGS__); \
    } while (0)

#define LF_HIP(call)                                                                     \
    do {                                                                                 \
        hipError_t _e = (call);                                                          \
        if (_e != hipSuccess)                                                            \
            return lf::fail(LF_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(_e), \
                            __FILE__, __LINE__);                                         \
    } while (0)
