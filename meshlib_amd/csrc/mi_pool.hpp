// mi_pool.hpp -- device buffers and streams of the host side: owned buffers, pooled temporaries, pooled streams.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstddef>
#include <mutex>

namespace mi {

// Device memory for the temporaries of one call or of a mesh's creation, and streams, kept for reuse: a hipMalloc and
// its hipFree cost about 57 and 83 us, a stream 150 and 55, and opening a 328 k-triangle mesh and checking it took
// ten of the former and two of the latter, 1.4 of its 4.3 ms.  Both pools are bounded (at most kTempKeep buffers
// of together kTempKeepBytes, kStreamKeep streams), are used under a lock, and take back only what no queued work
// uses any more.  They allocate no host memory (nothing here throws) and free nothing when the process ends, so no
// HIP call runs from a static destructor.
constexpr size_t kTempKeep = 8, kTempKeepBytes = size_t(64) << 20, kStreamKeep = 8;

struct TempPool {
    struct Idle { void* p; size_t bytes; int device; };
    std::mutex mu;
    Idle idle[kTempKeep];      // oldest first
    size_t count = 0, held = 0;

    Idle remove(size_t i)
    {
        const Idle d = idle[i];
        std::copy(idle + i + 1, idle + count, idle + i);
        --count;
        held -= d.bytes;
        return d;
    }
    // a buffer of at least `bytes` on the current device, the smallest idle one that is not far too large
    hipError_t take(size_t bytes, void** p, size_t* got, int* device)
    {
        hipError_t e = hipGetDevice(device);
        if (e != hipSuccess) return e;
        {
            std::lock_guard<std::mutex> lk(mu);
            size_t best = count;
            for (size_t i = 0; i < count; ++i)
                if (idle[i].device == *device && idle[i].bytes >= bytes && idle[i].bytes / 4 <= bytes + (size_t(1) << 18) &&
                    (best == count || idle[i].bytes < idle[best].bytes))
                    best = i;
            if (best < count) {
                const Idle d = remove(best);
                *p = d.p;
                *got = d.bytes;
                return hipSuccess;
            }
        }
        *got = bytes;
        return allocate(p, bytes);
    }
    // hipMalloc that gives the idle buffers back where memory is short.  HIP keeps a failed call's error until
    // hipGetLastError reads it, which the check after the next launch would; an error handled or returned here is read.
    hipError_t allocate(void** p, size_t bytes)
    {
        hipError_t e = hipMalloc(p, bytes);
        if (e != hipErrorOutOfMemory) return e;
        (void)hipGetLastError();
        if (!release()) return e;
        e = hipMalloc(p, bytes);
        if (e == hipErrorOutOfMemory) (void)hipGetLastError();
        return e;
    }
    // bytes that the next calls on the device find or can get back
    size_t idleBytes(int device)
    {
        std::lock_guard<std::mutex> lk(mu);
        size_t sum = 0;
        for (size_t i = 0; i < count; ++i)
            if (idle[i].device == device) sum += idle[i].bytes;
        return sum;
    }
    // nothing queued may use the buffer any more
    void give(void* p, size_t bytes, int device)
    {
        Idle drop[kTempKeep + 1];
        size_t dropped = 0;
        if (bytes > kTempKeepBytes) {
            drop[dropped++] = { p, bytes, device };
        } else {
            std::lock_guard<std::mutex> lk(mu);
            while (count && (count == kTempKeep || held + bytes > kTempKeepBytes)) drop[dropped++] = remove(0);
            idle[count++] = { p, bytes, device };
            held += bytes;
        }
        for (size_t i = 0; i < dropped; ++i) (void)hipFree(drop[i].p);
    }
    // frees every idle buffer; false if there was none
    bool release()
    {
        Idle drop[kTempKeep];
        size_t dropped = 0;
        {
            std::lock_guard<std::mutex> lk(mu);
            while (count) drop[dropped++] = remove(count - 1);
        }
        for (size_t i = 0; i < dropped; ++i) (void)hipFree(drop[i].p);
        return dropped > 0;
    }
};

inline TempPool& tempPool()
{
    static TempPool pool;
    return pool;
}

struct StreamPool {
    struct Idle { hipStream_t s; int device; };
    std::mutex mu;
    Idle idle[kStreamKeep];
    size_t count = 0;

    // a non-blocking stream of the device, which must be the current one
    hipError_t take(int device, hipStream_t* s)
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            for (size_t i = count; i-- > 0;)
                if (idle[i].device == device) {
                    *s = idle[i].s;
                    idle[i] = idle[--count];
                    return hipSuccess;
                }
        }
        return hipStreamCreateWithFlags(s, hipStreamNonBlocking);
    }
    void give(hipStream_t s, int device)
    {
        if (!s) return;
        if (hipStreamSynchronize(s) == hipSuccess) {
            std::lock_guard<std::mutex> lk(mu);
            if (count < kStreamKeep) {
                idle[count++] = { s, device };
                return;
            }
        }
        (void)hipStreamDestroy(s);
    }
};

inline StreamPool& streamPool()
{
    static StreamPool pool;
    return pool;
}

// RAII device buffer
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf() { if (p) (void)hipFree(p); }
    hipError_t alloc(size_t b)
    {
        if (p) { (void)hipFree(p); p = nullptr; bytes = 0; }
        if (b == 0) return hipSuccess;
        const hipError_t e = tempPool().allocate(&p, b);
        if (e == hipSuccess) bytes = b;
        else p = nullptr;
        return e;
    }
    template <class T> T* as() const { return static_cast<T*>(p); }
};

// RAII lease of a pooled device buffer that only work queued on `s` uses
struct TempBuf {
    void* p = nullptr;
    size_t bytes = 0;
    int device = 0;
    hipStream_t stream = nullptr;
    TempBuf() = default;
    TempBuf(const TempBuf&) = delete;
    TempBuf& operator=(const TempBuf&) = delete;
    ~TempBuf()
    {
        if (!p) return;
        if (hipStreamSynchronize(stream) == hipSuccess) tempPool().give(p, bytes, device);
        else (void)hipFree(p);
    }
    hipError_t take(size_t b, hipStream_t s)
    {
        stream = s;
        if (b == 0) return hipSuccess;
        const hipError_t e = tempPool().take(b, &p, &bytes, &device);
        if (e != hipSuccess) p = nullptr;
        return e;
    }
    template <class T> T* as() const { return static_cast<T*>(p); }
};

} // namespace mi
