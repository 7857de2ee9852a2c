// mi_volume.hip -- bounding cylinders of the tree's nodes (MeshDev::cyl, read by the lane walks).
//
// A node's cylinder: axis n = its dipole's direction area, normalised; centre c = the centre of its box,
// moved along n to the middle of its vertices' range; t = half that range, r = the largest distance of a
// vertex from the axis.  Every vertex lies inside, hence every triangle.
//
// The record of internal node j is 64 bytes, 32 per child: (c, n.x), (n.y, n.z, t and r as two halves, ref).  The
// halves count in units of MeshDev::cylUnit, a 2^15th of the mesh's diagonal rounded up to a power of two: 11 bits
// instead of bf16's 8, and a mixed-precision fma reads them as they are.
// t and r are widened by the rounding of the moved centre and by kWidenCoord and kWidenSize (mi_bound.hpp) before they are
// rounded up.
#include "mi_bound.hpp"
#include "mi_walk.hpp"

#include <algorithm>
#include <cfloat>
#include <cmath>

namespace mi {
namespace {

// Slivers -- strips and fans of long narrow triangles -- are long along an edge, not flat: a node whose triangles
// cover less than kRodArea of its box's squared diagonal while its middle leaf's longest edge spans half of the
// diagonal takes that edge as its axis (a rod), and so does a triangle with less than kRodArea of its longest
// edge's square (a regular triangle has 0.43, a regular patch about 0.5).  50 k points with discs alone, with rods
// and with rods and halves: a tube of 60 k strips of 1 : 10,000 10.9 / 1.5 / 0.82 ms, 40 k separate triangles
// of 1 : 250 0.91 / 0.09 / 0.08.  What rods do not help: 50,000 triangles around one vertex 51 / 38 / 35 ms, where
// the points nearest to that vertex are equally far from all of them.
constexpr float kRodArea = 0.1f;

struct Frame { float c[3], n[3]; };

// axis and provisional centre of a node with the box [mn, mx] and the direction area (nx, ny, nz)
__device__ __forceinline__ Frame nodeFrame(const float mn[3], const float mx[3], float nx, float ny, float nz)
{
    Frame f;
    for (int i = 0; i < 3; ++i) f.c[i] = 0.5f * mn[i] + 0.5f * mx[i];
    const float big = fmaxf(fabsf(nx), fmaxf(fabsf(ny), fabsf(nz)));
    f.n[0] = 1.f; f.n[1] = 0.f; f.n[2] = 0.f;
    if (big > 0 && big < INFINITY) {
        const float x = nx / big, y = ny / big, z = nz / big;
        const float len = sqrtf(x * x + y * y + z * z);
        f.n[0] = x / len; f.n[1] = y / len; f.n[2] = z / len;
    }
    return f;
}

// the longest edge of a triangle and its squared length
__device__ __forceinline__ float longestEdge(const Leaf& L, float e[3])
{
    const float* v[3] = { L.a, L.b, L.c };
    float best = -1.f;
    for (int i = 0; i < 3; ++i) {
        const float* p = v[i];
        const float* q = v[(i + 1) % 3];
        const float x = q[0] - p[0], y = q[1] - p[1], z = q[2] - p[2], l = x * x + y * y + z * z;
        if (l > best) { best = l; e[0] = x; e[1] = y; e[2] = z; }
    }
    return best;
}

// the frame of an internal node with the dipole (dirArea, area) d and the middle leaf `slot`
__device__ __forceinline__ Frame innerFrame(const MeshDev& m, const float mn[3], const float mx[3], const float4& d, int slot)
{
    const float x = mx[0] - mn[0], y = mx[1] - mn[1], z = mx[2] - mn[2], dd = x * x + y * y + z * z;
    if (d.w < kRodArea * dd) {
        float e[3];
        const float l = longestEdge(loadLeafLanes(m.tri, slot), e);
        if (l >= 0.25f * dd && l < INFINITY) return nodeFrame(mn, mx, e[0], e[1], e[2]);
    }
    return nodeFrame(mn, mx, d.x, d.y, d.z);
}

// offset of a vertex along the axis and its squared distance from it
__device__ __forceinline__ void along(const Frame& f, const float* v, float& h, float& rr)
{
    const float x = v[0] - f.c[0], y = v[1] - f.c[1], z = v[2] - f.c[2];
    h = x * f.n[0] + y * f.n[1] + z * f.n[2];
    const float a = x - h * f.n[0], b = y - h * f.n[1], c = z - h * f.n[2];
    rr = a * a + b * b + c * c;
}

// floats as unsigned integers of the same order (NaN above everything)
__device__ __forceinline__ uint32_t ordered(float x)
{
    const uint32_t b = __float_as_uint(x);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float unordered(uint32_t u)
{
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// per internal node: ordered(max h), ordered(max -h), bits of max rr, its middle leaf
struct Range { uint32_t hi, lo, rr, middle; };

// Every leaf goes down its own path and adds its corners to each node on it: neighbours share most of the path,
// so equal nodes are reduced within the wave, and a node that holds the whole block within the block, before
// the atomics (waves alone met in the top nodes' counters: 1.3 M faces 1.15 ms, now 0.30 ms).
constexpr int kRangeThreads = 1024;
__global__ __launch_bounds__(kRangeThreads) void kCylinderRanges(MeshDev m, Range* __restrict__ range)
{
    __shared__ float part[3][kRangeThreads / 64];
    __shared__ int whole[kRangeThreads / 64];       // the wave's only node, or -1
    const int slot = blockIdx.x * kRangeThreads + threadIdx.x;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const bool valid = slot < m.numFaces;
    Leaf L = loadLeafLanes(m.tri, valid ? slot : 0);
    int first = 0, num = m.numFaces, node = valid ? m.rootRef : -1;
    for (int level = 0; level < m.depth; ++level) {
        float hi = -INFINITY, lo = -INFINITY, rr = 0.f;
        int child = -1;
        if (node >= 0) {
            const float4 n0 = m.dnode[4 * (size_t)node], n1 = m.dnode[4 * (size_t)node + 1];
            const float4 n2 = m.dnode[4 * (size_t)node + 2], n3 = m.dnode[4 * (size_t)node + 3];
            const int h = num >> 1;
            const bool right = slot >= first + h;
            const float mn[3] = { right ? n1.z : n0.x, right ? n1.w : n0.y, right ? n2.x : n0.z };
            const float mx[3] = { right ? n2.y : n0.w, right ? n2.z : n1.x, right ? n2.w : n1.y };
            child = __float_as_int(right ? n3.y : n3.x);
            if (right) first += h;
            num = right ? num - h : h;
            if (child >= 0) {
                const float4 d = m.dint[2 * (size_t)child + 1];
                const int middle = first + (num >> 1);
                if (slot == middle) range[child].middle = (uint32_t)middle;
                const Frame f = innerFrame(m, mn, mx, d, middle);
                const float* v[3] = { L.a, L.b, L.c };
                for (int i = 0; i < 3; ++i) {
                    float a, b;
                    along(f, v[i], a, b);
                    // a vertex without finite offsets makes the node's cylinder unbounded
                    if (!(a - a == 0) || !(b < INFINITY)) { a = INFINITY; b = INFINITY; }
                    hi = fmaxf(hi, a); lo = fmaxf(lo, -a); rr = fmaxf(rr, b);
                }
            }
        }
        node = child;
        for (int d = 1; d < 64; d <<= 1) {
            const int on = __shfl_up(child, d);
            const float oh = __shfl_up(hi, d), ol = __shfl_up(lo, d), orr = __shfl_up(rr, d);
            if (lane >= d && on == child) { hi = fmaxf(hi, oh); lo = fmaxf(lo, ol); rr = fmaxf(rr, orr); }
        }
        const int next = __shfl_down(child, 1);
        const int end = __shfl(child, 63);
        const bool one = waveBallot(child == end) == ~0ull;
        if (lane == 63) {
            whole[w] = one ? child : -1;
            part[0][w] = hi; part[1][w] = lo; part[2][w] = rr;
        }
        __syncthreads();
        bool all = whole[0] >= 0;
        for (int k = 1; k < kRangeThreads / 64; ++k) all = all && whole[k] == whole[0];
        if (all) {
            if (threadIdx.x < 3) {
                float x = part[threadIdx.x][0];
                for (int k = 1; k < kRangeThreads / 64; ++k) x = fmaxf(x, part[threadIdx.x][k]);
                Range& r = range[whole[0]];
                uint32_t* const to = threadIdx.x == 0 ? &r.hi : threadIdx.x == 1 ? &r.lo : &r.rr;
                atomicMax(to, threadIdx.x == 2 ? __float_as_uint(x) : ordered(x));
            }
        } else if (child >= 0 && (lane == 63 || next != child)) {
            atomicMax(&range[child].hi, ordered(hi));
            atomicMax(&range[child].lo, ordered(lo));
            atomicMax(&range[child].rr, __float_as_uint(rr));
        }
        __syncthreads();
    }
}

// the smallest half not below x (x >= 0; infinity and NaN give infinity)
__device__ __forceinline__ uint32_t halfUp(float x)
{
    if (!(x <= 65504.f)) return 0x7c00u;
    const _Float16 h = (_Float16)x;
    const uint32_t b = __builtin_bit_cast(uint16_t, h);
    return (float)h < x ? b + 1u : b;
}

__device__ __forceinline__ void putCylinder(float4* out, const float c[3], const float n[3], float t, float r, float big,
                                            float unit, int ref)
{
    const float wide = big * kWidenCoord + (t + r) * kWidenSize;
    bool ok = big < INFINITY && t < INFINITY && r < INFINITY;
    for (int i = 0; i < 3; ++i) ok = ok && fabsf(c[i]) < INFINITY && fabsf(n[i]) < 2.f;
    // a quotient below the normal range is rounded to a multiple of 2^-149, far below the widening
    const uint32_t tr = ok ? (halfUp((t + wide) / unit) << 16) | halfUp((r + wide) / unit) : 0x7c007c00u;
    out[0] = make_float4(ok ? c[0] : 0.f, ok ? c[1] : 0.f, ok ? c[2] : 0.f, ok ? n[0] : 1.f);
    out[1] = make_float4(ok ? n[1] : 0.f, ok ? n[2] : 0.f, __uint_as_float(tr), __int_as_float(ref));
}

// a leaf's cylinder: the triangle's normal and smallest enclosing circle, or a sliver's longest edge
__device__ __forceinline__ void leafCylinder(const MeshDev& m, int slot, float4* out)
{
    const Leaf L = loadLeafLanes(m.tri, slot);
    const float* v[3] = { L.a, L.b, L.c };
    double e[3][3], len[3];       // edges v[i] -> v[i + 1]
    for (int i = 0; i < 3; ++i) {
        len[i] = 0;
        for (int k = 0; k < 3; ++k) {
            e[i][k] = (double)v[(i + 1) % 3][k] - v[i][k];
            len[i] += e[i][k] * e[i][k];
        }
    }
    const float nx = (float)(e[0][1] * e[1][2] - e[0][2] * e[1][1]);
    const float ny = (float)(e[0][2] * e[1][0] - e[0][0] * e[1][2]);
    const float nz = (float)(e[0][0] * e[1][1] - e[0][1] * e[1][0]);
    int longest = 0;
    if (len[1] > len[longest]) longest = 1;
    if (len[2] > len[longest]) longest = 2;
    const int i1 = (longest + 1) % 3, i2 = (longest + 2) % 3;
    // weights of the corners: the circumcentre of an acute triangle, else the longest edge's middle
    double w[3] = { 0, 0, 0 };
    const double wa = len[1] * (len[0] + len[2] - len[1]), wb = len[2] * (len[0] + len[1] - len[2]);
    const double wc = len[0] * (len[1] + len[2] - len[0]), sum = wa + wb + wc;
    if (len[longest] < len[i1] + len[i2] && sum > 0) { w[0] = wa / sum; w[1] = wb / sum; w[2] = wc / sum; }
    else { w[longest] = 0.5; w[i1] = 0.5; }
    float c[3], big = 0.f;
    for (int k = 0; k < 3; ++k) {
        c[k] = (float)(w[0] * v[0][k] + w[1] * v[1][k] + w[2] * v[2][k]);
        for (int i = 0; i < 3; ++i) big = fmaxf(big, fabsf(v[i][k]));
        if (!(v[0][k] - v[0][k] == 0) || !(v[1][k] - v[1][k] == 0) || !(v[2][k] - v[2][k] == 0)) big = INFINITY;
    }
    Frame f = nodeFrame(c, c, nx, ny, nz);
    float edge[3];
    const float l = longestEdge(L, edge);
    if (0.5f * sqrtf(nx * nx + ny * ny + nz * nz) < kRodArea * l) f = nodeFrame(c, c, edge[0], edge[1], edge[2]);
    for (int k = 0; k < 3; ++k) f.c[k] = c[k];
    float t = 0.f, rr = 0.f;
    for (int i = 0; i < 3; ++i) {
        float h, q;
        along(f, v[i], h, q);
        t = fmaxf(t, fabsf(h));
        rr = fmaxf(rr, q);
    }
    putCylinder(out, f.c, f.n, t, sqrtf(rr), big, m.cylUnit, ~slot);
}

__global__ __launch_bounds__(kBlock) void kCylinderRecords(MeshDev m, const Range* __restrict__ range, float4* __restrict__ cyl)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;      // child i & 1 of internal node i >> 1
    if (i >= 2 * ((int64_t)m.numFaces - 1)) return;
    const int j = (int)(i >> 1);
    const float4 n0 = m.dnode[4 * (size_t)j], n1 = m.dnode[4 * (size_t)j + 1];
    const float4 n2 = m.dnode[4 * (size_t)j + 2], n3 = m.dnode[4 * (size_t)j + 3];
    const bool right = i & 1;
    const int ref = __float_as_int(right ? n3.y : n3.x);
    float4* out = cyl + 2 * (size_t)i;
    if (ref < 0) {
        leafCylinder(m, ~ref, out);
        return;
    }
    const float mn[3] = { right ? n1.z : n0.x, right ? n1.w : n0.y, right ? n2.x : n0.z };
    const float mx[3] = { right ? n2.y : n0.w, right ? n2.z : n1.x, right ? n2.w : n1.y };
    const float4 d = m.dint[2 * (size_t)ref + 1];
    Frame f = innerFrame(m, mn, mx, d, (int)range[ref].middle);
    const float hi = unordered(range[ref].hi), lo = -unordered(range[ref].lo);
    const float mid = 0.5f * hi + 0.5f * lo;
    float big = 0.f;
    double off = 0, offSq = 0;      // what the rounding of the moved centre shifts it by: along the axis, and squared
    for (int k = 0; k < 3; ++k) {
        const float c = f.c[k] + mid * f.n[k];
        const double e = c - ((double)f.c[k] + (double)mid * f.n[k]);
        off += e * f.n[k];
        offSq += e * e;
        f.c[k] = c;
        big = fmaxf(big, fmaxf(fabsf(mn[k]), fabsf(mx[k])));
    }
    const float shiftT = 1.001f * (float)fabs(off), shiftR = 1.001f * sqrtf((float)fmax(offSq - off * off, 0.0));
    putCylinder(out, f.c, f.n, 0.5f * hi - 0.5f * lo + shiftT, sqrtf(__uint_as_float(range[ref].rr)) + shiftR, big, m.cylUnit,
                ref);
}

__global__ void kRangeInit(Range* r, int n)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) r[i] = Range{ 0u, 0u, 0u, 0u };
}

} // namespace

// Distances from which a lane walks over boxes, in diagonals of the mesh times the root of its number of faces: there the
// limit's slack is some 17 edges deep.  10,000 points, cylinders / boxes: 1.3 M faces 3,000 diagonals away 2.6 / 13.2 ms,
// 29,000 24 / 3.4, 290,000 263 / 0.33; 20 k faces 29,000 away 0.41 / 1.05, 290,000 2.5 / 0.34.
constexpr double kFarSizes = 1.2e7;

static double diagonal(const float rootMin[3], const float rootMax[3])
{
    double dd = 0;
    for (int i = 0; i < 3; ++i) dd += ((double)rootMax[i] - rootMin[i]) * ((double)rootMax[i] - rootMin[i]);
    return std::sqrt(dd);
}

float cylinderUnit(const float rootMin[3], const float rootMax[3])
{
    const double diag = diagonal(rootMin, rootMax);
    if (!(diag > 0) || !(diag < 1e308)) return 1.f;
    return (float)std::ldexp(1.0, std::max(std::ilogb(diag) + 1 - 15, -126));
}

float farDistSq(const float rootMin[3], const float rootMax[3], int32_t numFaces)
{
    const double far = kFarSizes / std::sqrt((double)numFaces) * diagonal(rootMin, rootMax);
    return far * far < (double)FLT_MAX ? (float)(far * far) : INFINITY;      // not a number: infinity
}

size_t cylinderScratchBytes(int32_t numFaces) { return numFaces > 1 ? (size_t)(numFaces - 1) * sizeof(Range) : 0; }

hipError_t buildCylinders(const MeshDev& m, float4* cyl, void* scratch, hipStream_t s)
{
    const int ni = m.numFaces - 1;
    if (ni < 1) return hipSuccess;
    Range* r = static_cast<Range*>(scratch);
    hipLaunchKernelGGL(kRangeInit, dim3((ni + kBlock - 1) / kBlock), dim3(kBlock), 0, s, r, ni);
    hipLaunchKernelGGL(kCylinderRanges, dim3((m.numFaces + kRangeThreads - 1) / kRangeThreads), dim3(kRangeThreads), 0, s, m,
                       r);
    hipLaunchKernelGGL(kCylinderRecords, dim3((unsigned)((2 * (int64_t)ni + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, m, r,
                       cyl);
    return hipGetLastError();
}

} // namespace mi
