// The host side's pools (meshlib_amd/csrc/mi_pool.hpp) against a stand-in runtime with a few bytes of memory that
// keeps a failed call's error until hipGetLastError reads it, as HIP does: an allocation that succeeds once the idle
// buffers are given back leaves no error behind for the check after the next launch, nor does one that fails.
// exit 0 when everything holds
#include "../../meshlib_amd/csrc/mi_pool.hpp"

#include <cstdio>
#include <cstdlib>
#include <map>

namespace {
size_t g_free = 0;
hipError_t g_last = hipSuccess;
std::map<void*, size_t> g_live;
int g_bad = 0;
void check(bool ok, const char* what)
{
    if (!ok) { ++g_bad; std::printf("FAILED: %s\n", what); }
}
} // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
    if (n > g_free) return g_last = hipErrorOutOfMemory;
    *p = std::malloc(1);
    g_free -= n;
    g_live[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    if (!p) return hipSuccess;
    g_free += g_live.at(p);
    g_live.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetLastError(void) { const hipError_t e = g_last; g_last = hipSuccess; return e; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
}

int main()
{
    const size_t MiB = size_t(1) << 20;
    g_free = 100 * MiB;
    { mi::TempBuf t; check(t.take(60 * MiB, nullptr) == hipSuccess, "first temporary"); }
    check(mi::tempPool().held == 60 * MiB && g_free == 40 * MiB, "the temporary is kept");
    {   // fits only without the idle temporary
        mi::DevBuf b;
        check(b.alloc(80 * MiB) == hipSuccess && b.bytes == 80 * MiB, "owned buffer after the idle ones went back");
        check(hipGetLastError() == hipSuccess, "owned buffer: no error left for the check after a launch");
    }
    { mi::TempBuf t; check(t.take(30 * MiB, nullptr) == hipSuccess, "second temporary"); }
    {
        mi::TempBuf t;
        check(t.take(90 * MiB, nullptr) == hipSuccess, "temporary after the idle ones went back");
        check(hipGetLastError() == hipSuccess, "temporary: no error left");
    }
    {   // does not fit at all: an error now, none for the next call
        mi::DevBuf b;
        check(b.alloc(200 * MiB) == hipErrorOutOfMemory && !b.p, "too large");
        check(hipGetLastError() == hipSuccess, "too large: no error left");
        mi::TempBuf t;
        check(t.take(200 * MiB, nullptr) == hipErrorOutOfMemory && !t.p, "too large a temporary");
        check(hipGetLastError() == hipSuccess, "too large a temporary: no error left");
    }
    { mi::TempBuf t; check(t.take(50 * MiB, nullptr) == hipSuccess, "third temporary"); }
    check(mi::tempPool().idleBytes(0) == 50 * MiB && mi::tempPool().idleBytes(1) == 0, "idle bytes by device");
    mi::tempPool().release();
    check(g_free == 100 * MiB && g_live.empty(), "everything given back");
    std::printf("bad %d\n", g_bad);
    return g_bad != 0;
}
