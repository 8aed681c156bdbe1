// Host side of the engine's memory: error messages, device buffers, page-locked buffers.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstddef>
#include <cstdio>
#include <string>

#include "../../include/emc_hip.h"

namespace emc {

inline thread_local std::string g_last_error;

// Message and code of a failed call. A HIP call's failure stays behind as the thread's last error until
// it is read, whatever succeeds after it: it is read here, so that a caller that goes on without the
// memory it asked for (or is called again) does not find it after its next launch.
inline int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_last_error = buf;
    if (code == EMC_E_HIP || code == EMC_E_NOMEM) (void)hipGetLastError();
    return code;
}

// Counts device allocations and frees of the engine buffers (every engine): a captured graph
// holds buffer addresses, so it is captured again once any buffer may have moved.
inline std::atomic<unsigned long> g_alloc_gen{0};

#define HIP_TRY(expr)                                                                        \
    do {                                                                                     \
        hipError_t err_ = (expr);                                                            \
        if (err_ != hipSuccess)                                                              \
            return emc::fail(EMC_E_HIP, "%s failed: %s", #expr, hipGetErrorString(err_));   \
    } while (0)

// Device buffer with an element count.
template <typename T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;    // elements in use
    size_t cap = 0;  // elements allocated: a smaller request reuses the allocation
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    DevBuf(DevBuf &&o) noexcept : p(o.p), n(o.n), cap(o.cap) {
        o.p = nullptr;
        o.n = o.cap = 0;
    }
    DevBuf &operator=(DevBuf &&o) noexcept {
        if (this != &o) {
            release();
            p = o.p;
            n = o.n;
            cap = o.cap;
            o.p = nullptr;
            o.n = o.cap = 0;
        }
        return *this;
    }
    ~DevBuf() { release(); }
    int alloc(size_t count) {
        if (p && count <= cap && count > 0) {
            n = count;
            return 0;
        }
        release();
        if (count == 0) return 0;
        ++g_alloc_gen;
        hipError_t err = hipMalloc((void **)&p, count * sizeof(T));
        if (err != hipSuccess) {
            p = nullptr;
            return fail(EMC_E_NOMEM, "hipMalloc of %zu bytes failed: %s", count * sizeof(T),
                        hipGetErrorString(err));
        }
        n = cap = count;
        return 0;
    }
    // Memory that only serves speed: count elements if the device keeps `leave` bytes free beside them (the
    // iteration and the calls after it allocate as well), else none and false.
    bool alloc_spare(size_t count, size_t leave) {
        if (p && count <= cap && count > 0) {
            n = count;
            return true;
        }
        release();
        size_t freeb = 0, totalb = 0;
        if (hipMemGetInfo(&freeb, &totalb) != hipSuccess) return (void)hipGetLastError(), false;
        return freeb >= leave && count <= (freeb - leave) / sizeof(T) && alloc(count) == 0;
    }
    int upload(const T *src, size_t count, hipStream_t s) {
        int rc = alloc(count);
        if (rc) return rc;
        if (count) HIP_TRY(hipMemcpyAsync(p, src, count * sizeof(T), hipMemcpyHostToDevice, s));
        return 0;
    }
    void release() {
        if (p) {
            ++g_alloc_gen;
            (void)hipFree(p);
        }
        p = nullptr;
        n = cap = 0;
    }
};

// Page-locked host memory (grow only) that the per-iteration lists are built in, so that
// their uploads run at the host link's speed without a staging copy.
template <typename T>
struct PinnedBuf {
    T *p = nullptr;
    size_t cap = 0;
    PinnedBuf() = default;
    PinnedBuf(const PinnedBuf &) = delete;
    PinnedBuf &operator=(const PinnedBuf &) = delete;
    ~PinnedBuf() { release(); }
    int reserve(size_t count) {
        count = std::max<size_t>(count, 1);
        if (p && count <= cap) return 0;
        release();
        const size_t want = count + count / 4;  // room for lists that grow a little
        if (hipHostMalloc((void **)&p, want * sizeof(T), hipHostMallocDefault) != hipSuccess) {
            p = nullptr;
            return fail(EMC_E_NOMEM, "hipHostMalloc of %zu bytes failed", want * sizeof(T));
        }
        cap = want;
        return 0;
    }
    void release() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        cap = 0;
    }
};

}  // namespace emc
