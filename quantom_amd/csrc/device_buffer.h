// device_buffer.h — device memory owned by the engine, and HIP errors as exceptions of the C entry points.
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <string>
#include <utility>
#include <vector>

#include "../../include/lima.h"

namespace lima {

struct LimaError {
    int code;
    std::string msg;
    LimaError(int c, std::string m) : code(c), msg(std::move(m)) {}
};

#define HIP_TRY(expr)                                                                         \
    do {                                                                                      \
        hipError_t e_ = (expr);                                                               \
        if (e_ != hipSuccess) {                                                               \
            throw LimaError(LIMA_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));   \
        }                                                                                     \
    } while (0)

// `n` elements at `p`.  A failed allocation throws and leaves a size that the memory has (callers
// compare `n` with what they need and launch kernels on `p`), and no error for a later launch's check.
template <typename T> struct DBuf {
    T* p = nullptr;
    size_t n = 0;
    DBuf() = default;
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    ~DBuf() { free(); }
    // exactly `count` elements; the contents are not kept
    void alloc(size_t count) {
        free();
        if (count) p = request(count);
        n = count;
    }
    // at least `count` elements; the contents are not kept.  If there is no memory for that, the
    // buffer has its former size again.
    void grow(size_t count) {
        if (n >= count) return;
        const size_t before = n;
        try {
            alloc(count);
        } catch (const LimaError&) {
            if (before) alloc(before);
            throw;
        }
    }
    void upload(const std::vector<T>& v) {
        const size_t count = std::max<size_t>(v.size(), 1);
        if (n != count) alloc(count);
        if (!v.empty()) HIP_TRY(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    }
    void zero() {
        if (p) HIP_TRY(hipMemset(p, 0, n * sizeof(T)));
    }
    void free() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }

private:
    static T* request(size_t count) {
        void* q = nullptr;
        const hipError_t e = hipMalloc(&q, count * sizeof(T));
        if (e == hipSuccess) return static_cast<T*>(q);
        (void)hipGetLastError();
        throw LimaError(LIMA_E_HIP, "hipMalloc of " + std::to_string(count * sizeof(T)) + " bytes: " + hipGetErrorString(e));
    }
};

}  // namespace lima
