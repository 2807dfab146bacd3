// common.hpp -- error plumbing, device buffers and launch helpers shared by the
// EROT HIP kernels and the host drivers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <stdexcept>
#include <string>
#include <vector>

namespace regot {

// Errors cross the C-ABI as a negative status plus a thread-local message.
struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string& msg) : std::runtime_error(msg), code(c) {}
};

enum Status : int {
    OK = 0,
    E_INVALID = -1,   // bad argument (sizes, dtype, null pointer)
    E_HIP = -2,       // HIP runtime failure
    E_NOMEM = -3,     // device allocation failed
    E_STATE = -4,     // operation needs state that is not there (e.g. no Hessian yet)
    E_INTERNAL = -5,
    E_SOLVER = -6,    // a solver stopped with an error (e.g. a failed line search)
};

[[noreturn]] inline void fail(int code, const char* fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    throw Error(code, buf);
}

#define HIP_CHECK(expr)                                                               \
    do {                                                                              \
        hipError_t _e = (expr);                                                       \
        if (_e != hipSuccess)                                                         \
            ::regot::fail(::regot::E_HIP, "%s failed: %s (%s:%d)", #expr,             \
                          hipGetErrorString(_e), __FILE__, __LINE__);                 \
    } while (0)

#define KERNEL_CHECK() HIP_CHECK(hipGetLastError())

// What a failed device allocation may have back before it is tried once more:
// memory that the handle whose call runs on this thread keeps for later calls.
struct Spare {
    void* owner = nullptr;
    void (*give_back)(void*) = nullptr;
};
inline thread_local Spare spare_memory;
struct SpareScope {
    Spare was;
    SpareScope(void* owner, void (*give_back)(void*)) : was(spare_memory)
    {
        spare_memory = Spare{owner, give_back};
    }
    SpareScope(const SpareScope&) = delete;
    SpareScope& operator=(const SpareScope&) = delete;
    ~SpareScope() { spare_memory = was; }
};

inline hipError_t device_malloc(void** p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess && spare_memory.give_back) {
        (void)hipGetLastError();
        spare_memory.give_back(spare_memory.owner);
        e = hipMalloc(p, bytes);
    }
    return e;
}

// Device allocation (hipMalloc), released on destruction, or a part of a Slab.
template <typename T>
struct DBuf {
    T* p = nullptr;
    size_t n = 0;
    bool owned = true;
    DBuf() = default;
    explicit DBuf(size_t count) { alloc(count); }
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    DBuf(DBuf&& o) noexcept : p(o.p), n(o.n), owned(o.owned) { o.p = nullptr; o.n = 0; }
    DBuf& operator=(DBuf&& o) noexcept
    {
        if (this != &o) {
            release();
            p = o.p; n = o.n; owned = o.owned;
            o.p = nullptr; o.n = 0;
        }
        return *this;
    }
    ~DBuf() { release(); }
    void alloc(size_t count)
    {
        release();
        if (count == 0) count = 1;
        hipError_t e = device_malloc(reinterpret_cast<void**>(&p), count * sizeof(T));
        if (e != hipSuccess) {
            p = nullptr;
            fail(E_NOMEM, "hipMalloc of %zu bytes failed: %s", count * sizeof(T),
                 hipGetErrorString(e));
        }
        n = count;
    }
    // Grow-only reallocation; contents are not preserved.
    void ensure(size_t count)
    {
        if (count > n || p == nullptr) alloc(count);
    }
    void release()
    {
        if (p && owned) (void)hipFree(p);
        p = nullptr;
        n = 0;
        owned = true;
    }
    // count elements at ptr, which someone else frees.
    void view(void* ptr, size_t count)
    {
        release();
        p = static_cast<T*>(ptr);
        n = count;
        owned = false;
    }
    operator T*() const { return p; }
};

// Several device buffers in one allocation: a handle's vectors cost one
// hipMalloc and one hipFree (20 to 40 us each, the bulk of a small handle's
// life) instead of a dozen.  add() every buffer, then make().
struct Slab {
    DBuf<unsigned char> mem;
    struct Part {
        void* buf;
        void (*set)(void*, void*, size_t);
        size_t at, count;
    };
    std::vector<Part> parts;
    size_t bytes = 0;
    template <typename T>
    void add(DBuf<T>& b, size_t count)
    {
        if (count == 0) count = 1;
        parts.push_back({&b,
                         [](void* buf, void* ptr, size_t c) {
                             static_cast<DBuf<T>*>(buf)->view(ptr, c);
                         },
                         bytes, count});
        bytes += (count * sizeof(T) + 255) / 256 * 256;
    }
    void make()
    {
        std::vector<Part> ps;
        ps.swap(parts);
        const size_t total = bytes;
        bytes = 0;
        mem.alloc(total);
        for (const Part& q : ps) q.set(q.buf, mem.p + q.at, q.count);
    }
};

// Pinned host staging memory (hipHostMalloc), released on destruction.
template <typename T>
struct HBuf {
    T* p = nullptr;
    size_t n = 0;
    HBuf() = default;
    HBuf(const HBuf&) = delete;
    HBuf& operator=(const HBuf&) = delete;
    ~HBuf() { release(); }
    void ensure(size_t count)
    {
        if (count <= n && p) return;
        release();
        if (count == 0) count = 1;
        HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&p), count * sizeof(T),
                                hipHostMallocDefault));
        n = count;
    }
    void release()
    {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        n = 0;
    }
};

// Pinned, device-mapped host array: kernels write it, the host reads it after
// the writing work has completed (stream order + event).
template <typename T>
struct MappedRing {
    T* h = nullptr;
    T* d = nullptr;
    size_t cap = 0;
    MappedRing() = default;
    MappedRing(const MappedRing&) = delete;
    MappedRing& operator=(const MappedRing&) = delete;
    ~MappedRing() { release(); }
    void ensure(size_t c)
    {
        if (h && c <= cap) return;
        release();
        if (c < 1) c = 1;
        HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&h), sizeof(T) * c, hipHostMallocMapped));
        HIP_CHECK(hipHostGetDevicePointer(reinterpret_cast<void**>(&d), h, 0));
        cap = c;
    }
    void release()
    {
        if (h) (void)hipHostFree(h);
        h = nullptr;
        d = nullptr;
        cap = 0;
    }
};

inline int ceil_div(long a, long b) { return static_cast<int>((a + b - 1) / b); }

// Grid of `blocks` workgroups of 256 threads.  A launch holds fewer than 2^32
// threads along x, so wider ones continue along y; the kernel's block is
// blockIdx.y gridDim.x + blockIdx.x, and the last few may lie past the end.
inline dim3 wide_grid(long blocks)
{
    constexpr long kX = 1L << 23;
    if (blocks <= kX) return dim3(static_cast<unsigned>(blocks));
    return dim3(static_cast<unsigned>(kX), static_cast<unsigned>((blocks + kX - 1) / kX));
}

}  // namespace regot
