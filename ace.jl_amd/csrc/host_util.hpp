// Host helpers shared by the translation units of libacehip.so: the
// thread-local error message behind ace_last_error(), the HIP_TRY macro and
// the grow-only buffer on device memory.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "grow_buf.hpp"

// last error message of the calling thread (one instance per process)
inline thread_local std::string g_err;

inline int set_err(const std::string& s) {
    g_err = s;
    return -1;
}

#define HIP_TRY(expr)                                                              \
    do {                                                                           \
        hipError_t e_ = (expr);                                                    \
        if (e_ != hipSuccess)                                                      \
            return set_err(std::string(#expr) + ": " + hipGetErrorString(e_));    \
    } while (0)

struct HipMemory {
    static int alloc(void** p, size_t bytes) {
        HIP_TRY(hipMalloc(p, bytes));
        return 0;
    }
    static void release(void* p) { (void)hipFree(p); }
    static int copy(void* p, const void* host, size_t bytes) {
        HIP_TRY(hipMemcpy(p, host, bytes, hipMemcpyHostToDevice));
        return 0;
    }
};

template <typename T>
using DevBuf = acehost::GrowBuf<T, HipMemory>;
