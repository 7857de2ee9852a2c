// mi_tree_gpu.hip -- AABB tree + dipoles + flattened layout built on the GPU.
//
// Tree (source/MRMesh/MRAABBTreeMaker.hpp:50-165): every internal node splits its leaves at the
// median (left gets num/2) under a total order -- key (min+max) along the node box's dims sorted by
// extent, largest first, ties to the next dim, last to the face id.  Because the order is total,
// the left set of each node is unique, however it is found; and because every node gives num/2 of its
// leaves to its left child, the shape of the tree, all node numbers (children root+1 and root+2*half)
// and all leaf ranges follow from the number of faces alone (nodeAt) -- no level waits for the host.
//   * nodes of more than kSub leaves are split level by level, several blocks a node: three rounds of radix
//     selection on the first key (histograms of 11, 11 and 10 bits), a block per node that settles equal
//     first keys by the other keys, partition of the leaves into the two halves with their boxes;
//   * nodes of at most kSub leaves are finished by one block each in LDS, all their levels in one launch
//     (a bitonic sort of each node's leaves per level), dipoles included.
// Four library radix sorts per level were 1,800 launches for a mesh of 328 k faces, bound by the launches; now 60
// launches, and creating that mesh from host arrays went from 13.0 to 1.35 ms (0.9 ms of it kernels).
// Leaf boxes, dipoles (source/MRMesh/MRDipole.cpp:23-71) and the flattened arrays repeat the host
// builder's float expressions in the same order (the library is compiled with -ffp-contract=off and
// correctly rounded division and square root), so every record equals the host build bit-for-bit.
#include "mi_tree_gpu.hpp"

#include <algorithm>
#include <cfloat>

namespace mi {
namespace {

constexpr int kB = 256;
// leaves of a subtree built in LDS, two a thread: three blocks of 48 KB a CU (2048 leaves in one 96-KB block a CU:
// 1.3 M faces 1.08 ms against 0.64 ms, one level fewer above)
constexpr int kSub = 1024;
constexpr int kSubThreads = 512;
constexpr int kChunk = 4096;        // leaves of a block of the level kernels
constexpr int kBins = 2048;         // histogram of one selection round

// leaf record while building: {min.xyz, max.x} {max.y, max.z, face, 0}
struct Elem { float4 a, b; };

__device__ __forceinline__ uint32_t ordU(float x)
{
    const uint32_t b = __float_as_uint(x);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float unordU(uint32_t u)
{
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}
// sort key of a float under '<' (-0 and +0 compare equal)
__device__ __forceinline__ uint32_t keyU(float x) { return ordU(x + 0.0f); }

// std::nextafter(x, -FLT_MAX) / (x, FLT_MAX) for finite x
__device__ __forceinline__ float nextDown(float x)
{
    if (x == -FLT_MAX) return x;
    if (x == 0.0f) return __uint_as_float(0x80000001u);
    const uint32_t b = __float_as_uint(x);
    return __uint_as_float(x > 0.0f ? b - 1u : b + 1u);
}
__device__ __forceinline__ float nextUp(float x)
{
    if (x == FLT_MAX) return x;
    if (x == 0.0f) return __uint_as_float(0x00000001u);
    const uint32_t b = __float_as_uint(x);
    return __uint_as_float(x > 0.0f ? b + 1u : b - 1u);
}

// a node: its pre-order number, the first of its leaves in left-to-right order and their number
struct Node { int32_t v, first, num; };

// node i (from the left) of a level all of whose parents have two leaves or more
__device__ __forceinline__ Node child(const Node& p, bool right)
{
    const int32_t h = p.num >> 1;
    return right ? Node{ p.v + 2 * h, p.first + h, p.num - h } : Node{ p.v + 1, p.first, h };
}
__device__ __forceinline__ Node nodeAt(int32_t n, int level, uint32_t i)
{
    Node d{ 0, 0, n };
    for (int l = level - 1; l >= 0; --l) d = child(d, (i >> l) & 1u);
    return d;
}

// computeFaceBox + insignificantlyExpanded (source/MRMesh/MRAABBTree.cpp:15-29, MRBox.h:260-270)
__global__ void kLeafBoxes(const float* __restrict__ verts, const int32_t* __restrict__ tris, int32_t n,
                           Elem* __restrict__ el)
{
    const int32_t f = blockIdx.x * kB + threadIdx.x;
    if (f >= n) return;
    float mn[3] = { FLT_MAX, FLT_MAX, FLT_MAX }, mx[3] = { -FLT_MAX, -FLT_MAX, -FLT_MAX };
    for (int k = 0; k < 3; ++k) {
        const float* p = verts + 3 * (int64_t)tris[3 * (int64_t)f + k];
        for (int i = 0; i < 3; ++i) {
            if (p[i] < mn[i]) mn[i] = p[i];
            if (p[i] > mx[i]) mx[i] = p[i];
        }
    }
    for (int i = 0; i < 3; ++i) { mn[i] = nextDown(mn[i]); mx[i] = nextUp(mx[i]); }
    el[f].a = make_float4(mn[0], mn[1], mn[2], mx[0]);
    el[f].b = make_float4(mx[1], mx[2], __int_as_float(f), 0.f);
}

// dims by (extent, index), smallest first -- findSortedBoxDims (source/MRMesh/MRBox.h:378-396)
__device__ __forceinline__ void sortedDims(const float mn[3], const float mx[3], int sd[3])
{
    const float e[3] = { mx[0] - mn[0], mx[1] - mn[1], mx[2] - mn[2] };
    sd[0] = 0; sd[1] = 1; sd[2] = 2;
    auto lessP = [&](int a, int b) { return e[a] < e[b] || (!(e[b] < e[a]) && a < b); };
    int t;
    if (lessP(sd[1], sd[0])) { t = sd[0]; sd[0] = sd[1]; sd[1] = t; }
    if (lessP(sd[2], sd[1])) { t = sd[1]; sd[1] = sd[2]; sd[2] = t; }
    if (lessP(sd[1], sd[0])) { t = sd[0]; sd[0] = sd[1]; sd[1] = t; }
}

// the four keys of a leaf in its node's order, k = 0 (first) to 3 (the face); sd = sortedDims of the node
__device__ __forceinline__ uint32_t leafKey(const Elem& e, const int sd[3], int k)
{
    if (k == 3) return (uint32_t)__float_as_int(e.b.z);
    const float c[3] = { e.a.x + e.a.w, e.a.y + e.b.x, e.a.z + e.b.y };
    const int d = sd[2 - k];
    return keyU(d == 0 ? c[0] : d == 1 ? c[1] : c[2]);
}

// ---------------------------------------------------------------- levels of large nodes
//
// Per node of the level: its box, the histograms of the three rounds, the pivot (the leaf of rank num/2: the
// leaves before it in the order go left) and the write positions of both halves.
struct LevelNode {
    uint32_t box[6];        // ordered encoding: min xyz, max xyz
    uint32_t pivot[4];      // its keys; those behind the first that no other leaf shares are 0
    uint32_t left, right;   // leaves written so far
    uint32_t listed;        // leaves in `list`
};

struct Level {
    int32_t n;              // faces
    int32_t level;
    int32_t blocksPerNode;
    Elem* src;
    Elem* dst;
    uint32_t* k0;           // first key of the leaf at each position
    uint32_t* list;         // positions of the leaves left after two rounds, per node from its first
    LevelNode* nodes;
    LevelNode* next;        // of the next level; null at the last one
    uint32_t* hist;         // 3 * kBins per node
};

// this block's node and its chunk of leaves
__device__ __forceinline__ Node blockNode(const Level& L, uint32_t& i, int32_t& begin, int32_t& end)
{
    i = blockIdx.x / (uint32_t)L.blocksPerNode;
    const Node d = nodeAt(L.n, L.level, i);
    begin = d.first + (int32_t)(blockIdx.x % (uint32_t)L.blocksPerNode) * kChunk;
    end = min(begin + kChunk, d.first + d.num);
    return d;
}

__device__ __forceinline__ void nodeDims(const LevelNode& nd, int sd[3])
{
    float mn[3], mx[3];
    for (int k = 0; k < 3; ++k) { mn[k] = unordU(nd.box[k]); mx[k] = unordU(nd.box[3 + k]); }
    sortedDims(mn, mx, sd);
}

__device__ __forceinline__ void clearNode(LevelNode& nd)
{
    for (int k = 0; k < 3; ++k) { nd.box[k] = 0xffffffffu; nd.box[3 + k] = 0u; }
    nd.left = nd.right = nd.listed = 0u;
}

// what the first level starts from; the later ones are prepared by the level before
__global__ void kLevelInit(Level L)
{
    const int t = blockIdx.x * kB + threadIdx.x;
    if (t < 3 * kBins) L.hist[t] = 0u;
    if (t == 0) clearNode(L.nodes[0]);
}

// the block's sum of every thread's value before its own, and of all
__device__ __forceinline__ uint32_t scanBlock(uint32_t own, uint32_t& total)
{
    __shared__ uint32_t sums[kB / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t s = own;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(s, d);
        if (lane >= d) s += o;
    }
    __syncthreads();      // the last call's sums have been read
    if (lane == 63) sums[w] = s;
    __syncthreads();
    uint32_t before = s - own;
    total = 0;
    for (int k = 0; k < kB / 64; ++k) {
        if (k < w) before += sums[k];
        total += sums[k];
    }
    return before;
}

// the box of the first level's node (the others' come with the partition above them)
__global__ __launch_bounds__(kB) void kLevelBox(Level L)
{
    uint32_t i;
    int32_t begin, end;
    blockNode(L, i, begin, end);
    float b[6] = { FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX };
    for (int32_t p = begin + (int32_t)threadIdx.x; p < end; p += kB) {
        const Elem e = L.src[p];
        const float o[6] = { e.a.x, e.a.y, e.a.z, e.a.w, e.b.x, e.b.y };
        for (int k = 0; k < 3; ++k) { b[k] = fminf(b[k], o[k]); b[k + 3] = fmaxf(b[k + 3], o[k + 3]); }
    }
    for (int d = 32; d; d >>= 1)
        for (int k = 0; k < 3; ++k) {
            b[k] = fminf(b[k], __shfl_xor(b[k], d));
            b[k + 3] = fmaxf(b[k + 3], __shfl_xor(b[k + 3], d));
        }
    __shared__ float part[kB / 64][6];
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 6; ++k) part[threadIdx.x >> 6][k] = b[k];
    __syncthreads();
    if (threadIdx.x >= 6 || begin >= end) return;
    const int k = threadIdx.x;
    float x = part[0][k];
    for (int w = 1; w < kB / 64; ++w) x = k < 3 ? fminf(x, part[w][k]) : fmaxf(x, part[w][k]);
    if (k < 3) atomicMin(&L.nodes[i].box[k], ordU(x));
    else atomicMax(&L.nodes[i].box[k], ordU(x));
}

// the bin of a histogram that holds rank `rank` (block-wide): rank becomes the rank inside the bin, count the
// bin's size
__device__ __forceinline__ uint32_t pickBin(const uint32_t* hist, uint32_t& rank, uint32_t& count)
{
    __shared__ uint32_t found[3];
    constexpr int per = kBins / kB;
    static_assert(per == 8, "two vector loads");
    const uint4 v0 = reinterpret_cast<const uint4*>(hist)[2 * threadIdx.x], v1 = reinterpret_cast<const uint4*>(hist)[2 * threadIdx.x + 1];
    const uint32_t h[per] = { v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w };
    uint32_t own = 0, all;
    for (int k = 0; k < per; ++k) own += h[k];
    uint32_t before = scanBlock(own, all);
    if (rank >= before && rank < before + own) {
        int k = 0;
        while (rank >= before + h[k]) { before += h[k]; ++k; }
        found[0] = (uint32_t)(per * threadIdx.x + k);
        found[1] = rank - before;
        found[2] = h[k];
    }
    __syncthreads();
    const uint32_t bin = found[0];
    rank = found[1];
    count = found[2];
    __syncthreads();
    return bin;
}

// the bits of a 32-bit key in selection round r
__device__ __forceinline__ uint32_t roundBits(uint32_t key, int r)
{
    return r == 0 ? key >> 21 : r == 1 ? (key >> 10) & 2047u : key & 1023u;
}

// Selection round ROUND on the first key: the histogram of the leaves whose bits of the earlier rounds are
// the picked ones.  Round 0 also stores the keys, the last round lists its leaves.
template <int ROUND>
__global__ __launch_bounds__(kB) void kLevelHist(Level L)
{
    __shared__ uint32_t h[kBins];
    __shared__ uint32_t mine[ROUND == 2 ? kChunk : 1];
    __shared__ uint32_t count2, base2;
    uint32_t i;
    int32_t begin, end;
    const Node d = blockNode(L, i, begin, end);
    for (int k = threadIdx.x; k < kBins; k += kB) h[k] = 0u;
    if (threadIdx.x == 0) count2 = 0u;
    uint32_t* const hist = L.hist + (size_t)i * 3 * kBins;
    uint32_t prefix = 0, rank = (uint32_t)(d.num >> 1), count;
    if (ROUND >= 1) prefix = pickBin(hist, rank, count);
    if (ROUND >= 2) prefix = (prefix << 11) | pickBin(hist + kBins, rank, count);
    int sd[3];
    if (ROUND == 0) nodeDims(L.nodes[i], sd);
    __syncthreads();
    for (int32_t p = begin + (int32_t)threadIdx.x; p < end; p += kB) {
        uint32_t key;
        if (ROUND == 0) {
            key = leafKey(L.src[p], sd, 0);
            L.k0[p] = key;
        } else {
            key = L.k0[p];
            if ((ROUND == 1 ? key >> 21 : key >> 10) != prefix) continue;
        }
        atomicAdd(&h[roundBits(key, ROUND)], 1u);
        if (ROUND == 2) mine[atomicAdd(&count2, 1u)] = (uint32_t)p;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kBins; k += kB)
        if (h[k]) atomicAdd(&hist[ROUND * kBins + k], h[k]);
    if (ROUND == 2) {
        if (threadIdx.x == 0) base2 = atomicAdd(&L.nodes[i].listed, count2);
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < count2; k += kB) L.list[(uint32_t)d.first + base2 + k] = mine[k];
    }
}

// One block per node: the pivot's first key, and where several leaves share it the other keys, by the same
// selection over those leaves.
__global__ __launch_bounds__(kB) void kLevelPivot(Level L)
{
    __shared__ __align__(16) uint32_t h[kBins];
    __shared__ uint32_t shared;
    const uint32_t i = blockIdx.x;
    const Node d = nodeAt(L.n, L.level, i);
    if (L.next && threadIdx.x < 2) clearNode(L.next[2 * i + threadIdx.x]);
    const uint32_t* const hist = L.hist + (size_t)i * 3 * kBins;
    uint32_t rank = (uint32_t)(d.num >> 1), count;
    uint32_t k0 = pickBin(hist, rank, count);
    k0 = (k0 << 11) | pickBin(hist + kBins, rank, count);
    k0 = (k0 << 10) | pickBin(hist + 2 * kBins, rank, count);
    uint32_t piv[4] = { k0, 0u, 0u, 0u };
    if (count > 1) {
        int sd[3];
        nodeDims(L.nodes[i], sd);
        const int32_t ties = (int32_t)L.nodes[i].listed;
        for (int w = 1; w < 4 && count > 1; ++w) {
            uint32_t prefix = 0;
            for (int r = 0; r < 3 && count > 1; ++r) {
                __syncthreads();
                for (int k = threadIdx.x; k < kBins; k += kB) h[k] = 0u;
                __syncthreads();
                for (int32_t q = (int32_t)threadIdx.x; q < ties; q += kB) {
                    const uint32_t p = L.list[d.first + q];
                    bool in = L.k0[p] == k0;
                    if (!in) continue;
                    const Elem e = L.src[p];
                    for (int u = 1; u < w; ++u) in = in && leafKey(e, sd, u) == piv[u];
                    const uint32_t key = leafKey(e, sd, w);
                    if (r == 1) in = in && (key >> 21) == prefix;
                    if (r == 2) in = in && (key >> 10) == prefix;
                    if (in) atomicAdd(&h[roundBits(key, r)], 1u);
                }
                __syncthreads();
                prefix = (prefix << (r == 2 ? 10 : 11)) | pickBin(h, rank, count);
                // a bin of one leaf is the pivot: its remaining bits are its own
                if (count == 1 && r < 2) {
                    __syncthreads();
                    for (int32_t q = (int32_t)threadIdx.x; q < ties; q += kB) {
                        const uint32_t p = L.list[d.first + q];
                        bool in = L.k0[p] == k0;
                        if (!in) continue;
                        const Elem e = L.src[p];
                        for (int u = 1; u < w; ++u) in = in && leafKey(e, sd, u) == piv[u];
                        const uint32_t key = leafKey(e, sd, w);
                        if (in && (key >> (r == 0 ? 21 : 10)) == prefix) shared = key;
                    }
                    __syncthreads();
                    prefix = shared;
                }
            }
            piv[w] = prefix;
        }
    }
    if (threadIdx.x < 4) {
        const int t = threadIdx.x;
        L.nodes[i].pivot[t] = t == 0 ? piv[0] : t == 1 ? piv[1] : t == 2 ? piv[2] : piv[3];
    }
}

// Writes the level's nodes and moves every leaf to its half of the node's range (in any order); on the way the
// boxes of both halves, and the histograms are cleared for the next level (a box pass and a clearing launch per
// level more: 12 and 4 us of 79 a level at 328 k faces).
__global__ __launch_bounds__(kB) void kLevelPartition(Level L, TreeNode* __restrict__ tree, int32_t* __restrict__ firstOf)
{
    __shared__ uint32_t base[2];
    __shared__ float part[kB / 64][12];
    uint32_t i;
    int32_t begin, end;
    const Node d = blockNode(L, i, begin, end);
    LevelNode& nd = L.nodes[i];
    const int32_t h = d.num >> 1;
    if (begin == d.first && threadIdx.x == 0) {
        TreeNode t;
        for (int k = 0; k < 3; ++k) { t.box.min[k] = unordU(nd.box[k]); t.box.max[k] = unordU(nd.box[3 + k]); }
        t.l = d.v + 1;
        t.r = d.v + 2 * h;
        tree[d.v] = t;
        firstOf[d.v] = d.first;
    }
    int sd[3];
    nodeDims(nd, sd);
    const uint32_t piv[4] = { nd.pivot[0], nd.pivot[1], nd.pivot[2], nd.pivot[3] };
    constexpr int per = kChunk / kB;
    uint32_t goLeft = 0, mine = 0;
    for (int k = 0; k < per; ++k) {
        const int32_t p = begin + k * kB + (int32_t)threadIdx.x;
        if (p >= end) break;
        ++mine;
        const uint32_t key = L.k0[p];
        bool left = key < piv[0];
        if (key == piv[0]) {
            const Elem e = L.src[p];
            for (int w = 1; w < 4; ++w) {
                const uint32_t kw = leafKey(e, sd, w);
                if (kw != piv[w]) { left = kw < piv[w]; break; }
            }
        }
        if (left) goLeft |= 1u << k;
    }
    const uint32_t nl = (uint32_t)__popc(goLeft);
    // both counts in one scan: 16 bits each (at most kChunk)
    uint32_t total;
    const uint32_t before = scanBlock(nl | ((mine - nl) << 16), total);
    if (threadIdx.x == 0) {
        base[0] = atomicAdd(&nd.left, total & 0xffffu);
        base[1] = atomicAdd(&nd.right, total >> 16);
    }
    __syncthreads();
    int32_t l = d.first + (int32_t)(base[0] + (before & 0xffffu));
    int32_t r = d.first + h + (int32_t)(base[1] + (before >> 16));
    float box[12];      // of the left and of the right half
    for (int k = 0; k < 12; ++k) box[k] = k % 6 < 3 ? FLT_MAX : -FLT_MAX;
    for (int k = 0; k < (int)mine; ++k) {
        const Elem e = L.src[begin + k * kB + (int32_t)threadIdx.x];
        const bool left = (goLeft >> k) & 1u;
        L.dst[left ? l++ : r++] = e;
        const float o[6] = { e.a.x, e.a.y, e.a.z, e.a.w, e.b.x, e.b.y };
        for (int c = 0; c < 3; ++c) {
            const float lo = o[c], hi = o[3 + c];
            if (left) { box[c] = fminf(box[c], lo); box[3 + c] = fmaxf(box[3 + c], hi); }
            else { box[6 + c] = fminf(box[6 + c], lo); box[9 + c] = fmaxf(box[9 + c], hi); }
        }
    }
    if (!L.next) return;
    for (int k = 0; k < 12; ++k)
        for (int x = 32; x; x >>= 1) box[k] = k % 6 < 3 ? fminf(box[k], __shfl_xor(box[k], x)) : fmaxf(box[k], __shfl_xor(box[k], x));
    const int lane = threadIdx.x & 63;
    if (lane == 0)
        for (int k = 0; k < 12; ++k) part[threadIdx.x >> 6][k] = box[k];
    __syncthreads();
    if (threadIdx.x < 12) {
        const int k = threadIdx.x % 6;
        const bool least = k < 3;
        float x = part[0][threadIdx.x];
        for (int w = 1; w < kB / 64; ++w) x = least ? fminf(x, part[w][threadIdx.x]) : fmaxf(x, part[w][threadIdx.x]);
        uint32_t* const to = &L.next[2 * i + threadIdx.x / 6].box[k];
        const uint32_t moved = threadIdx.x < 6 ? total & 0xffffu : total >> 16;
        if (moved) { if (least) atomicMin(to, ordU(x)); else atomicMax(to, ordU(x)); }
    }
    const size_t words = (size_t)3 * kBins << (L.level + 1);
    for (size_t t = (size_t)blockIdx.x * kB + threadIdx.x; t < words; t += (size_t)gridDim.x * kB) L.hist[t] = 0u;
}

// leaf dipole: dirArea = cross(b-a, c-a)/2, area = |dirArea|, pos = area * centroid
// (source/MRMesh/MRDipole.cpp:28-45, triCenter / leftDirDblArea in MRMeshMath.cpp:119-149)
__device__ __forceinline__ Dipole leafDipole(const float* __restrict__ verts, const int32_t* __restrict__ tris,
                                             int32_t face)
{
    const int32_t* t = tris + 3 * (int64_t)face;
    const float* a = verts + 3 * (int64_t)t[0];
    const float* b = verts + 3 * (int64_t)t[1];
    const float* c = verts + 3 * (int64_t)t[2];
    const float ab[3] = { b[0] - a[0], b[1] - a[1], b[2] - a[2] };
    const float ac[3] = { c[0] - a[0], c[1] - a[1], c[2] - a[2] };
    const float cr[3] = { ab[1] * ac[2] - ab[2] * ac[1], ab[2] * ac[0] - ab[0] * ac[2], ab[0] * ac[1] - ab[1] * ac[0] };
    const float third = 1 / 3.0f;
    Dipole d;
    for (int k = 0; k < 3; ++k) d.dirArea[k] = 0.5f * cr[k];
    d.area = sqrtf(d.dirArea[0] * d.dirArea[0] + d.dirArea[1] * d.dirArea[1] + d.dirArea[2] * d.dirArea[2]);
    for (int k = 0; k < 3; ++k) d.pos[k] = d.area * (third * ((a[k] + b[k]) + c[k]));
    d.rr = 0;
    return d;
}

// sum of the children's dipoles (source/MRMesh/MRDipole.cpp:47-60)
__device__ __forceinline__ void addDipoles(Dipole* __restrict__ dip, const Node& d)
{
    const Dipole dl = dip[d.v + 1], dr = dip[d.v + 2 * (d.num >> 1)];
    Dipole o;
    for (int k = 0; k < 3; ++k) {
        o.pos[k] = dl.pos[k] + dr.pos[k];
        o.dirArea[k] = dl.dirArea[k] + dr.dirArea[k];
    }
    o.area = dl.area + dr.area;
    o.rr = 0;
    dip[d.v] = o;
}

// ---------------------------------------------------------------- subtrees of at most kSub leaves

struct SubShared {
    uint64_t key[kSub];            // leaf at each position: first key << 32 | leaf
    float box[6][kSub];            // by leaf
    int32_t face[kSub];
    uint32_t acc[6][kSub / 2];     // node boxes, by half the node's first position (nodes of two leaves or more)
};

// One block per node of level `level`: all levels below it.  A thread keeps the nodes that cover its two
// positions; leaves move between positions of one node only.
__global__ __launch_bounds__(kSubThreads) void kSubtrees(int32_t n, int level, const Elem* __restrict__ el,
                                                         const float* __restrict__ verts, const int32_t* __restrict__ tris,
                                                         TreeNode* __restrict__ tree, Dipole* __restrict__ dip,
                                                         int32_t* __restrict__ firstOf)
{
    extern __shared__ __align__(16) unsigned char subMem[];
    SubShared& S = *reinterpret_cast<SubShared*>(subMem);
    const Node root = nodeAt(n, level, blockIdx.x);
    const int s0 = root.num, tid = threadIdx.x, lane = tid & 63;
    Node nd[2];            // first relative to the root's
    int leaf[2];
    for (int q = 0; q < 2; ++q) {
        const int p = tid + q * kSubThreads;
        nd[q] = Node{ root.v, 0, p < s0 ? s0 : 0 };
        leaf[q] = p;
        if (p < s0) {
            const Elem e = el[root.first + p];
            S.box[0][p] = e.a.x; S.box[1][p] = e.a.y; S.box[2][p] = e.a.z;
            S.box[3][p] = e.a.w; S.box[4][p] = e.b.x; S.box[5][p] = e.b.y;
            S.face[p] = __float_as_int(e.b.z);
        }
    }
    int levels = 0;
    for (int maxNum = s0; maxNum > 1; maxNum = (maxNum + 1) >> 1, ++levels) {
        for (int k = 0; k < 6; ++k) S.acc[k][tid] = k < 3 ? 0xffffffffu : 0u;
        __syncthreads();
        // node boxes: runs of equal nodes within the wave, then one atomic per run
        for (int q = 0; q < 2; ++q) {
            const bool in = nd[q].num > 1;
            const int f = in ? nd[q].first : -1;
            float b[6] = { FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX };
            if (in)
                for (int k = 0; k < 6; ++k) b[k] = S.box[k][leaf[q]];
            for (int d = 1; d < 64; d <<= 1) {
                const int of = __shfl_up(f, d);
                float o[6];
                for (int k = 0; k < 6; ++k) o[k] = __shfl_up(b[k], d);
                if (lane >= d && of == f)
                    for (int k = 0; k < 3; ++k) {
                        b[k] = fminf(b[k], o[k]);
                        b[k + 3] = fmaxf(b[k + 3], o[k + 3]);
                    }
            }
            const int nf = __shfl_down(f, 1);
            if (in && (lane == 63 || nf != f))
                for (int k = 0; k < 3; ++k) {
                    atomicMin(&S.acc[k][f >> 1], ordU(b[k]));
                    atomicMax(&S.acc[3 + k][f >> 1], ordU(b[k + 3]));
                }
        }
        __syncthreads();
        const auto dims = [&](int f, int sd[3]) {
            float mn[3], mx[3];
            for (int k = 0; k < 3; ++k) { mn[k] = unordU(S.acc[k][f >> 1]); mx[k] = unordU(S.acc[3 + k][f >> 1]); }
            sortedDims(mn, mx, sd);
        };
        const auto element = [&](int e) {
            Elem x;
            x.a = make_float4(S.box[0][e], S.box[1][e], S.box[2][e], S.box[3][e]);
            x.b = make_float4(S.box[4][e], S.box[5][e], __int_as_float(S.face[e]), 0.f);
            return x;
        };
        for (int q = 0; q < 2; ++q) {
            const int p = tid + q * kSubThreads;
            if (p >= s0) continue;
            uint64_t key = (uint32_t)leaf[q];
            if (nd[q].num > 1) {
                int sd[3];
                dims(nd[q].first, sd);
                key |= (uint64_t)leafKey(element(leaf[q]), sd, 0) << 32;
                if (p == nd[q].first) {
                    TreeNode t;
                    for (int k = 0; k < 3; ++k) {
                        t.box.min[k] = unordU(S.acc[k][p >> 1]);
                        t.box.max[k] = unordU(S.acc[3 + k][p >> 1]);
                    }
                    t.l = nd[q].v + 1;
                    t.r = nd[q].v + 2 * (nd[q].num >> 1);
                    tree[nd[q].v] = t;
                    firstOf[nd[q].v] = root.first + p;
                }
            }
            S.key[p] = key;
        }
        __syncthreads();
        // Every node of the level sorts its own leaves: `half` threads a node, each one pair a stage.  All
        // comparisons are ascending (a merge starts by comparing mirrored positions), so the positions a node
        // lacks up to a power of two would hold the largest keys and never move: they are skipped.  Pairs of up
        // to 64 threads stay within a wave, whose LDS operations are in order.
        int half = 1;
        while (2 * half < maxNum) half <<= 1;
        Node own = Node{ 0, 0, s0 };
        const int t = tid & (half - 1);
        for (int b = levels - 1; b >= 0; --b) own = child(own, ((tid / half) >> b) & 1);
        const bool sorts = tid / half < (1 << levels);
        const auto sync = [&] {
            if (half > 64) __syncthreads();
            else {
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        };
        for (int k = 2; k <= 2 * half; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                const int block = t / j, in = t - block * j;
                const int a = block * 2 * j + in, b = j == (k >> 1) ? block * 2 * j + 2 * j - 1 - in : a + j;
                if (sorts && b < own.num) {
                    const int pa = own.first + a, pb = own.first + b;
                    const uint64_t ka = S.key[pa], kb = S.key[pb];
                    bool swap = kb < ka;
                    if ((ka >> 32) == (kb >> 32)) {
                        int sd[3];
                        dims(own.first, sd);
                        const Elem xa = element((int)(uint32_t)ka), xb = element((int)(uint32_t)kb);
                        for (int w = 1; w < 4; ++w) {
                            const uint32_t va = leafKey(xa, sd, w), vb = leafKey(xb, sd, w);
                            if (va != vb) { swap = vb < va; break; }
                        }
                    }
                    if (swap) { S.key[pa] = kb; S.key[pb] = ka; }
                }
                sync();
            }
        __syncthreads();
        for (int q = 0; q < 2; ++q) {
            const int p = tid + q * kSubThreads;
            if (p >= s0) continue;
            leaf[q] = (int)(uint32_t)S.key[p];
            if (nd[q].num > 1) nd[q] = child(nd[q], p - nd[q].first >= (nd[q].num >> 1));
        }
        __syncthreads();
    }
    for (int q = 0; q < 2; ++q) {
        const int p = tid + q * kSubThreads;
        if (p >= s0) continue;
        TreeNode t;
        for (int k = 0; k < 3; ++k) { t.box.min[k] = S.box[k][leaf[q]]; t.box.max[k] = S.box[3 + k][leaf[q]]; }
        t.l = S.face[leaf[q]];
        t.r = -1;
        tree[nd[q].v] = t;
        firstOf[nd[q].v] = root.first + p;
        dip[nd[q].v] = leafDipole(verts, tris, t.l);
    }
    for (int l = levels - 1; l >= 0; --l) {
        __threadfence_block();
        __syncthreads();
        if (tid < (1 << l)) {
            Node d = root;
            for (int b = l - 1; b >= 0 && d.num > 1; --b) d = child(d, (tid >> b) & 1);
            if (d.num > 1) addDipoles(dip, d);
        }
    }
}

// the dipoles of the levels above the subtrees, one block for all of them
__global__ __launch_bounds__(kSubThreads) void kTopDipoles(int32_t n, int level, Dipole* __restrict__ dip)
{
    for (int l = level - 1; l >= 0; --l) {
        for (uint32_t i = threadIdx.x; i < (1u << l); i += kSubThreads) addDipoles(dip, nodeAt(n, l, i));
        __threadfence_block();
        __syncthreads();
    }
}

// pos /= area (as a multiplication by 1/area), rr = squared distance to the farthest box corner
// (source/MRMesh/MRDipole.cpp:11-21, 62-70)
__global__ void kFinalizeDipoles(int32_t nn, const TreeNode* __restrict__ nodes, Dipole* __restrict__ dip)
{
    const int32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= nn) return;
    Dipole d = dip[i];
    const TreeNode nd = nodes[i];
    if (d.area > 0) {
        const float inv = 1 / d.area;
        for (int k = 0; k < 3; ++k) d.pos[k] *= inv;
    }
    float rr = 0;
    for (int k = 0; k < 3; ++k) {
        float tmin = d.pos[k] - nd.box.min[k];
        tmin = tmin * tmin;
        float tmax = d.pos[k] - nd.box.max[k];
        tmax = tmax * tmax;
        rr += tmin > tmax ? tmin : tmax;
    }
    d.rr = rr;
    dip[i] = d;
}

// the traversal layout (mi_tree.hpp): internal nodes and leaf slots in pre-order.  Before node i in pre-order
// there are firstOf[i] leaves, all those to the left of its own.  faceIds (optional): a tree built over the
// valid faces of a mesh with deleted faces names the packed face index in its leaves; the reference's leaves
// hold the real FaceId (source/MRMesh/MRAABBTree.cpp:35-49).  Packing keeps the face order, so the tree (whose
// ties fall to the face index) is the same; only the ids of the leaf nodes and triangle records are mapped back.
__global__ void kFlatten(int32_t nn, TreeNode* __restrict__ nodes, const Dipole* __restrict__ dip,
                         const int32_t* __restrict__ firstOf, const float* __restrict__ verts,
                         const int32_t* __restrict__ tris, const int32_t* __restrict__ faceIds, float4* __restrict__ dnode,
                         float4* __restrict__ tri, float4* __restrict__ dint, float4* __restrict__ dleaf)
{
    const int32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= nn) return;
    const TreeNode n = nodes[i];
    const Dipole d = dip[i];
    const float4 d0 = make_float4(d.pos[0], d.pos[1], d.pos[2], d.rr);
    const float4 d1 = make_float4(d.dirArea[0], d.dirArea[1], d.dirArea[2], d.area);
    if (n.r >= 0) {
        const int32_t j = i - firstOf[i];
        const auto refOf = [&](int32_t c) { return nodes[c].r < 0 ? ~firstOf[c] : c - firstOf[c]; };
        const Box3 L = nodes[n.l].box, R = nodes[n.r].box;
        float4* r = dnode + 4 * (int64_t)j;
        r[0] = make_float4(L.min[0], L.min[1], L.min[2], L.max[0]);
        r[1] = make_float4(L.max[1], L.max[2], R.min[0], R.min[1]);
        r[2] = make_float4(R.min[2], R.max[0], R.max[1], R.max[2]);
        r[3] = make_float4(__int_as_float(refOf(n.l)), __int_as_float(refOf(n.r)), 0.f, 0.f);
        dint[2 * (int64_t)j] = d0;
        dint[2 * (int64_t)j + 1] = d1;
    } else {
        const int32_t k = firstOf[i];
        const int32_t f = n.l;
        const int32_t* t = tris + 3 * (int64_t)f;
        const float* a = verts + 3 * (int64_t)t[0];
        const float* b = verts + 3 * (int64_t)t[1];
        const float* c = verts + 3 * (int64_t)t[2];
        const int32_t id = faceIds ? faceIds[f] : f;
        float4* r = tri + 3 * (int64_t)k;
        r[0] = make_float4(a[0], a[1], a[2], b[0]);
        r[1] = make_float4(b[1], b[2], c[0], c[1]);
        r[2] = make_float4(c[2], __int_as_float(id), 0.f, 0.f);
        dleaf[2 * (int64_t)k] = d0;
        dleaf[2 * (int64_t)k + 1] = d1;
        if (faceIds) nodes[i].l = id;
    }
}

inline size_t al(size_t b) { return (b + 255) & ~size_t(255); }
inline unsigned gridFor(int64_t n) { return (unsigned)((n + kB - 1) / kB); }

// levels of nodes of more than kSub leaves (the largest node of level l has ceil(n / 2^l) leaves)
inline int64_t largest(int32_t n, int level) { return ((int64_t)n + (int64_t(1) << level) - 1) >> level; }
inline int topLevels(int32_t n)
{
    int l = 0;
    while (largest(n, l) > kSub) ++l;
    return l;
}

struct Scratch {
    Elem* el[2];
    uint32_t *k0, *list, *hist;
    LevelNode* nodes;
    int32_t* firstOf;
};

size_t layout(int32_t nf, Scratch* s, char* base)
{
    const size_t n = (size_t)nf, nn = 2 * n - 1;
    const int top = topLevels(nf);
    const size_t wide = top > 0 ? size_t(1) << (top - 1) : 0;      // nodes of the widest level
    size_t off = 0;
    auto take = [&](size_t bytes) { char* p = base ? base + off : nullptr; off += al(bytes); return p; };
    char* e0 = take(n * sizeof(Elem));
    char* e1 = take(top ? n * sizeof(Elem) : 0);
    char* k0 = take(top ? n * 4 : 0);
    char* list = take(top ? n * 4 : 0);
    char* hist = take(wide * 3 * kBins * 4);
    char* nodes = take(2 * wide * sizeof(LevelNode));
    char* firstOf = take(nn * 4);
    if (s) {
        s->el[0] = reinterpret_cast<Elem*>(e0);
        s->el[1] = reinterpret_cast<Elem*>(e1);
        s->k0 = reinterpret_cast<uint32_t*>(k0);
        s->list = reinterpret_cast<uint32_t*>(list);
        s->hist = reinterpret_cast<uint32_t*>(hist);
        s->nodes = reinterpret_cast<LevelNode*>(nodes);
        s->firstOf = reinterpret_cast<int32_t*>(firstOf);
    }
    return off;
}

#define TG_HIP(x)                              \
    do {                                       \
        const hipError_t e_ = (x);             \
        if (e_ != hipSuccess) return e_;       \
    } while (0)

} // namespace

size_t deviceTreeScratchBytes(int32_t nf)
{
    if (nf <= 0) return 0;
    return layout(nf, nullptr, nullptr);
}

hipError_t buildDeviceTree(const float* d_verts, const int32_t* d_tris, int32_t nf, void* scratch,
                           size_t scratchBytes, const DeviceTreeOut& out, DeviceTreeInfo& info, hipStream_t st,
                           const int32_t* d_faceIds)
{
    info = DeviceTreeInfo{};
    if (nf <= 0) return hipSuccess;
    Scratch S;
    if (layout(nf, &S, static_cast<char*>(scratch)) > scratchBytes) return hipErrorInvalidValue;
    const int32_t n = nf, nn = 2 * nf - 1;
    while (largest(n, info.depth) > 1) ++info.depth;
    kLeafBoxes<<<gridFor(n), kB, 0, st>>>(d_verts, d_tris, n, S.el[0]);
    const int top = topLevels(n);
    const size_t wide = top > 0 ? size_t(1) << (top - 1) : 0;
    int cur = 0;
    for (int l = 0; l < top; ++l, cur ^= 1) {
        const int32_t count = int32_t(1) << l;
        LevelNode* const nodes = S.nodes + (l & 1) * wide;
        const Level L{ n, l, (int32_t)((largest(n, l) + kChunk - 1) / kChunk), S.el[cur], S.el[cur ^ 1], S.k0, S.list, nodes,
                       l + 1 < top ? S.nodes + (~l & 1) * wide : nullptr, S.hist };
        const dim3 blocks((unsigned)(count * L.blocksPerNode));
        if (l == 0) {
            kLevelInit<<<gridFor(3 * kBins), kB, 0, st>>>(L);
            kLevelBox<<<blocks, kB, 0, st>>>(L);
        }
        kLevelHist<0><<<blocks, kB, 0, st>>>(L);
        kLevelHist<1><<<blocks, kB, 0, st>>>(L);
        kLevelHist<2><<<blocks, kB, 0, st>>>(L);
        kLevelPivot<<<count, kB, 0, st>>>(L);
        kLevelPartition<<<blocks, kB, 0, st>>>(L, out.nodes, S.firstOf);
        TG_HIP(hipGetLastError());
    }
    TG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kSubtrees), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)sizeof(SubShared)));
    kSubtrees<<<1u << top, kSubThreads, sizeof(SubShared), st>>>(n, top, S.el[cur], d_verts, d_tris, out.nodes, out.dipoles,
                                                                 S.firstOf);
    TG_HIP(hipGetLastError());
    if (top > 0) kTopDipoles<<<1, kSubThreads, 0, st>>>(n, top, out.dipoles);
    kFinalizeDipoles<<<gridFor(nn), kB, 0, st>>>(nn, out.nodes, out.dipoles);
    kFlatten<<<gridFor(nn), kB, 0, st>>>(nn, out.nodes, out.dipoles, S.firstOf, d_verts, d_tris, d_faceIds, out.dnode, out.tri,
                                         out.dint, out.dleaf);
    TG_HIP(hipGetLastError());
    TreeNode root;
    TG_HIP(hipMemcpyAsync(&root, out.nodes, sizeof(TreeNode), hipMemcpyDeviceToHost, st));
    TG_HIP(hipStreamSynchronize(st));
    info.rootBox = root.box;
    info.rootRef = root.r < 0 ? ~0 : 0;
    return hipSuccess;
}

} // namespace mi
