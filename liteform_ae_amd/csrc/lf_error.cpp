// Error state and status strings of the C ABI, and the pool of page-locked read-back buffers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <vector>

#include "lf_internal.h"

namespace lf {

std::string& last_error() {
    static thread_local std::string msg;
    return msg;
}

int fail(int status, const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    last_error() = buf;
    return status;
}

namespace {
std::mutex g_pinned_lock;
// (never destroyed: a plan may still be released while the process ends)
std::vector<void*>& pinned_pool() {
    static std::vector<void*>* pool = new std::vector<void*>();
    return *pool;
}
}  // namespace

PinnedLoan::PinnedLoan(size_t bytes) {
    if (bytes <= kPooledBytes) {
        {
            std::lock_guard<std::mutex> hold(g_pinned_lock);
            auto& pool = pinned_pool();
            if (!pool.empty()) {
                p_ = pool.back();
                pool.pop_back();
                pinned_ = true;
                return;
            }
        }
        if (hipHostMalloc(&p_, kPooledBytes, hipHostMallocPortable) == hipSuccess) {
            pinned_ = true;
            return;
        }
        (void)hipGetLastError();
        p_ = nullptr;
    }
    p_ = std::malloc(bytes ? bytes : 1);
}

PinnedLoan::~PinnedLoan() {
    if (!pinned_) {
        std::free(p_);
        return;
    }
    {
        std::lock_guard<std::mutex> hold(g_pinned_lock);
        auto& pool = pinned_pool();
        if (pool.size() < kPooledBuffers) {
            pool.push_back(p_);
            return;
        }
    }
    (void)hipHostFree(p_);
}

namespace {
__global__ void __launch_bounds__(256)
move_words_kernel(const uint32_t* up_from, uint32_t* up_to, long long up, uint32_t* clear, long long n_clear, const uint32_t* down_from,
                  uint32_t* down_to, long long down) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x, stride = (long long)gridDim.x * 256;
    for (long long i = t; i < up; i += stride) up_to[i] = up_from[i];
    for (long long i = t; i < n_clear; i += stride) clear[i] = 0;
    for (long long i = t; i < down; i += stride) down_to[i] = down_from[i];
}
}  // namespace

hipError_t move_words(Words up, bool up_pinned, void* clear, size_t clear_bytes, Words down, bool down_pinned, hipStream_t s) {
    hipError_t e = hipSuccess;
    if (up.bytes && !up_pinned) {
        e = hipMemcpyAsync(up.to, up.from, up.bytes, hipMemcpyHostToDevice, s);
        up.bytes = 0;
    }
    const size_t down_bytes = down_pinned ? down.bytes : 0, most = std::max(std::max(up.bytes, down_bytes), clear_bytes) / 4;
    if (e == hipSuccess && most > 0) {
        move_words_kernel<<<(unsigned)std::min<size_t>((most + 255) / 256, 4096), 256, 0, s>>>(
            (const uint32_t*)up.from, (uint32_t*)up.to, (long long)(up.bytes / 4), (uint32_t*)clear, (long long)(clear_bytes / 4),
            (const uint32_t*)down.from, (uint32_t*)down.to, (long long)(down_bytes / 4));
        e = hipGetLastError();
    }
    if (e == hipSuccess && down.bytes && !down_pinned) e = hipMemcpyAsync(down.to, down.from, down.bytes, hipMemcpyDeviceToHost, s);
    return e;
}

}  // namespace lf

extern "C" {

int lf_version(void) { return LF_VERSION; }

const char* lf_last_error(void) { return lf::last_error().c_str(); }

const char* lf_status_string(int status) {
    switch (status) {
        case LF_OK: return "ok";
        case LF_ERR_INVALID: return "invalid argument";
        case LF_ERR_TOO_SMALL: return "partition holds a single nonzero";
        case LF_ERR_HIP: return "HIP runtime error";
        case LF_ERR_CONFIG: return "bucket widths do not fit the matrix";
        case LF_ERR_UNSUPPORTED: return "unsupported size or type";
        case LF_ERR_WORKSPACE: return "workspace too small";
        default: return "unknown status";
    }
}

}  // extern "C"
