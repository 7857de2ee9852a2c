// Device checks of the winding number's square root and quotient (midSqrt, midDipole in mi_walk.hpp) against the
// correctly rounded operations.  Built into tests/cpp/libmid_math.so, called by tests/test_gpu_mid_math.py.
#include "mi_walk.hpp"

#include <cmath>

using namespace mi;

namespace {

__device__ unsigned long long g_wrong;

// every float of the range: the square root
__global__ void kRoots()
{
    unsigned long long bad = 0;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < kMidSpan; i += gridDim.x * 256) {
        const float x = __uint_as_float(kMidLow + i);
        float half;
        if (midSqrt(x, half) != sqrtf(x)) ++bad;
    }
    if (bad) atomicAdd(&g_wrong, bad);
}

// every float of [1, 4) and each of its multiples by powers of 4 in the range: root, half and quotient scale exactly
__global__ void kScales()
{
    unsigned long long bad = 0;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < (1u << 24); i += gridDim.x * 256) {
        const float x = __uint_as_float(0x3f800000u + i);
        float half, h;
        const float root = midSqrt(x, half), q = midDipole(1.f, x);
        for (int k = -30; k < 30; ++k) {
            const float y = ldexpf(x, 2 * k);
            if (!midRange(y)) continue;
            if (midSqrt(y, h) != ldexpf(root, k) || h != ldexpf(half, -k) || midDipole(1.f, y) != ldexpf(q, -3 * k)) ++bad;
        }
    }
    if (bad) atomicAdd(&g_wrong, bad);
}

// quotients over squared lengths first, first + stride, .. of [1, 4) and every numerator of [1, 2)
__global__ void kQuotients(uint32_t first, uint32_t stride)
{
    const float dd = __uint_as_float(0x3f800000u + ((first + blockIdx.x * stride) & 0xffffffu));
    const float den = sqrtf(dd) * dd;
    unsigned long long bad = 0;
    for (uint32_t n = threadIdx.x; n < (1u << 23); n += blockDim.x) {
        const float num = __uint_as_float(0x3f800000u + n);
        if (midDipole(num, dd) != num / den) ++bad;
    }
    if (bad) atomicAdd(&g_wrong, bad);
}

long long finish()
{
    unsigned long long h = 0, *p = nullptr;
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) return -1;
    if (hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(g_wrong)) != hipSuccess) return -1;
    if (hipMemcpy(&h, p, sizeof h, hipMemcpyDeviceToHost) != hipSuccess) return -1;
    const unsigned long long zero = 0;
    if (hipMemcpy(p, &zero, sizeof zero, hipMemcpyHostToDevice) != hipSuccess) return -1;
    return (long long)h;
}

} // namespace

// how many results differ, or -1 after an error
extern "C" long long mid_roots() { kRoots<<<4096, 256>>>(); return finish(); }
extern "C" long long mid_scales() { kScales<<<4096, 256>>>(); return finish(); }
extern "C" long long mid_quotients(uint32_t first, uint32_t count, uint32_t stride)
{
    kQuotients<<<count, 256>>>(first, stride);
    return finish();
}
