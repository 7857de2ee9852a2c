// mi_lane.hpp -- the lane walk: one independent depth-first walk per query over oriented bounds
// (internal to the kernel translation units).
//
// Every child of an internal node is bounded by a flat cylinder: an axis n (the area-weighted normal of
// its triangles), a centre c, the half thickness t along n and the radius r across it (mi_volume.hip).
// A surface patch is thin along its normal, so the cylinder's distance is within a fraction of the
// patch's curvature of the true one, where an axis-aligned box of a tilted patch is off by about its
// size.  Bound tests and leaf tests per voxel of 256^3 on a 1.3 M-triangle bumpy sphere: 2,590 and 552 with boxes
// (depth-first on the CPU), 180 and 8.7 in these walks (90 nodes of two children); with vertex noise of a fifth of the
// edges 2,216 and 360 against 241 and 20.
//
// With so few visits a query no longer needs its wave's company: a wave sharing one walk visits the union
// of its lanes' nodes (about 2,500 four-wide steps per 64 voxels with boxes), while 64 separate walks
// take as many steps as the longest of them (103 on that grid), each a 64-byte gather per lane.
//
//  * stack: [entry][lane] in LDS, the child's ref and the top 16 bits of its lower bound (a truncated
//    non-negative float is a lower bound of itself), so a pop drops what the best has overtaken without
//    touching memory.  An entry takes 5 bytes (refs of 24 bits; 6 in trees of more than 2^23 faces, WIDE): the
//    walk waits for its gathers, so waves per CU count, and the stacks limit them (LDS comes in units of 1,280
//    bytes: depth 21 has 21 waves of distance walks and 18 of projections a CU; the 1.3 M-triangle volume took
//    11.9 / 14.5 / 16.5 / 20.4 ms with 18 / 14 / 12 / 10);
//  * leaf tests (FP64) are queued per wave and run one per lane when as many wait as lanes are walking:
//    dense lanes while the wave is full, no stale bests when only a few long walks are left;
//  * results are minima over candidates and do not depend on the order of visits: a subtree is dropped
//    only when its lower bound is above the best by more than all rounding (the margins in
//    mi_bound.hpp), so every leaf that could decide the result is tested.
#pragma once

#include "mi_bound.hpp"
#include "mi_walk.hpp"

namespace mi {
namespace {

// no node: neither an internal ref (>= 0) nor a leaf (~slot, slot < 2^30)
constexpr int kNoNode = (int)0x80000000u;

// LDS of one wave, sized at launch: the fixed part, the ties of projections, then the stack, per entry
// 64 x uint32 and 64 x uint8 (WIDE: uint16)
struct LaneShared {
    int32_t leaf[128];      // queued leaf tests: leaf slot
    uint8_t owner[128];     //   and the lane whose query it is for; takeovers use 64.. while fewer than 64 wait
    uint32_t best[64];      // each lane's best squared distance (float bits, >= 0)
};
// idle lanes take over pending subtrees while at most this many lanes have work left
constexpr int kTakeBelow = 48;
// entries a lane without a node may try per step
constexpr int kPops = 2;
constexpr int kLaneTies = 4;
// a query whose list has been full so many times has many ties
constexpr uint32_t kManyTies = 4;
// Projections also keep leaves that tie at the lane's best.  With many ties the last place holds the first leaf of a subtree
// (a leaf more at most) outside of which none comes before the first of those that have been compared.
struct LaneTies {
    int32_t leaf[kLaneTies][64];
    uint32_t count[64];     // leaves listed, times the list has been full (8 bits each), level of the subtree
    __device__ __forceinline__ static uint32_t level(uint32_t c) { return c >> 16; }
    __device__ __forceinline__ static uint32_t room(uint32_t c) { return c >> 16 ? kLaneTies - 1 : kLaneTies; }
};
constexpr int32_t kNarrowFaces = 1 << 23;      // refs of at most 24 bits with sign
inline bool laneWide(int32_t numFaces) { return numFaces > kNarrowFaces; }
// band: boxWalk's stack takes the place of the walk's
inline size_t laneSharedBytes(int depth, bool ties, bool wide, bool band = false)
{
    const size_t d = depth > 0 ? (size_t)depth : 1;
    return sizeof(LaneShared) + (ties ? sizeof(LaneTies) : 0) + d * 64 * (band ? 8 : wide ? 6 : 5);
}

// the wave's view of its LDS
template <bool TIES, bool WIDE>
struct LaneLds {
    LaneShared* s;
    LaneTies* ties;          // projections only
    uint32_t* word;          // WIDE: ref; else upper half of the bound, lower half of the ref
    uint8_t* rest;           // WIDE: upper half of the bound; else bits 16..23 of the ref

    __device__ __forceinline__ LaneLds(unsigned char* base, int depth)
    {
        s = reinterpret_cast<LaneShared*>(base);
        ties = TIES ? reinterpret_cast<LaneTies*>(base + sizeof(LaneShared)) : nullptr;
        unsigned char* stack = base + sizeof(LaneShared) + (TIES ? sizeof(LaneTies) : 0);
        word = reinterpret_cast<uint32_t*>(stack);
        rest = stack + (size_t)(depth > 0 ? depth : 1) * 256;
    }
    __device__ __forceinline__ int2* band() const { return reinterpret_cast<int2*>(word); }
    // entry at = 64 * index + lane; the bound is stored as its top 16 bits
    __device__ __forceinline__ void put(int at, int ref, float bound) const
    {
        if (WIDE) {
            word[at] = (uint32_t)ref;
            reinterpret_cast<uint16_t*>(rest)[at] = stackDist(bound);
        } else {
            word[at] = (__float_as_uint(bound) & 0xffff0000u) | ((uint32_t)ref & 0xffffu);
            rest[at] = (uint8_t)((uint32_t)ref >> 16);
        }
    }
    __device__ __forceinline__ int get(int at, float& bound) const
    {
        const uint32_t w = word[at];
        if (WIDE) {
            bound = stackDist(reinterpret_cast<const uint16_t*>(rest)[at]);
            return (int)w;
        }
        bound = __uint_as_float(w & 0xffff0000u);
        return ((int)(int8_t)rest[at] << 16) | (int)(w & 0xffffu);
    }
};

// Squared distance from the point to a child's cylinder, a lower bound of its triangles' distances up to
// the rounding that kLimitSlack covers.  a = (c, n.x), b = (n.y, n.z, t and r as halves in units of `unit`, ref).
// centerSq: to the centre.
__device__ __forceinline__ float cylinderDistSq(const float4& a, const float4& b, float unit, float px, float py, float pz,
                                                float& centerSq)
{
    const float yx = px - a.x, yy = py - a.y, yz = pz - a.z;
    const float h = __builtin_fmaf(b.y, yz, __builtin_fmaf(b.x, yy, a.w * yx));
    const float vx = __builtin_fmaf(-h, a.w, yx), vy = __builtin_fmaf(-h, b.x, yy), vz = __builtin_fmaf(-h, b.y, yz);
    const float rr = __builtin_fmaf(vz, vz, __builtin_fmaf(vy, vy, vx * vx));
    const float rho = __builtin_amdgcn_sqrtf(rr);
    centerSq = __builtin_fmaf(h, h, rr);
    typedef _Float16 half2 __attribute__((ext_vector_type(2)));
    const half2 tr = __builtin_bit_cast(half2, b.z);      // one mixed-precision fma each
    const float s = fmaxf(__builtin_fmaf(-(float)tr.y, unit, fabsf(h)), 0.f);
    const float q = fmaxf(__builtin_fmaf(-(float)tr.x, unit, rho), 0.f);
    return __builtin_fmaf(s, s, q * q);
}

// what a lower bound is compared with
__device__ __forceinline__ float laneLimit(float best) { return __builtin_fmaf(best, 1.f + kLimitSlack, 1e-37f); }

// Orders what lanes of one wave write to and read from each other's LDS: the hardware keeps a wave's LDS
// operations in order, the fence keeps the compiler from reusing or moving values across.
__device__ __forceinline__ void waveSync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A subtree of the leaf slots first .. first + num - 1.  Slots are in left-to-right order, every node gives the first half
// of its leaves (rounded down) to its left child, and internal nodes are numbered in pre-order: a node's children are found
// without memory.
struct TieRange {
    int node, first, num;
    __device__ __forceinline__ int mid() const { return first + (num >> 1); }
    __device__ __forceinline__ void toChild(bool left)
    {
        const int h = num >> 1;
        node += left ? 1 : h;
        first += left ? 0 : h;
        num = left ? h : num - h;
    }
};

// which child of an internal node the depth-first walk of a query visits first: the nearer, ties to the right
__device__ __forceinline__ bool leftFirst(const MeshDev& m, int node, float px, float py, float pz)
{
    const size_t rec = 4 * (size_t)node;
    const float4 n0 = gload(m.dnode, rec), n1 = gload(m.dnode, rec + 1), n2 = gload(m.dnode, rec + 2);
    return boxDistSq(n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, px, py, pz) < boxDistSq(n1.z, n1.w, n2.x, n2.y, n2.z, n2.w, px, py, pz);
}

// leaves a lane's list of `count` tied leaves with its first in the query's order at the front: of two leaves, the one on
// the side that is visited first where their paths part
__device__ __forceinline__ void resolveTies(const MeshDev& m, LaneTies* ties, float px, float py, float pz, uint32_t count)
{
    const int lane = threadIdx.x & 63;
    int win = ties->leaf[0][lane];
    for (uint32_t i = 1; i < count; ++i) {
        const int k = ties->leaf[i][lane], lo = k < win ? k : win, hi = k < win ? win : k;
        TieRange r{ 0, 0, m.numFaces };
        for (;;) {
            const bool left = hi < r.mid();
            if (!left && lo < r.mid()) break;
            r.toChild(left);
        }
        if ((k == lo) == leftFirst(m, r.node, px, py, pz)) win = k;
    }
    ties->leaf[0][lane] = win;
}

// Empties a full list but for the first of its leaves, and with many ties narrows the subtree along the path to that one
// while it takes the child that is visited first: the ties outside, nearly all of them, are dropped as they are met.  50 k
// points around a cone of 3,000 / 10,000 / 50,000 triangles a tip 3.6 / 12.1 / 70 -> 2.3 / 6.4 / 39 ms.  Narrowed at every
// full list a cone takes 15 % less, but the few ties of an ordinary vertex cost 6 % of a projection.
__device__ __forceinline__ void shortenTies(const MeshDev& m, LaneTies* ties, float px, float py, float pz)
{
    const int lane = threadIdx.x & 63;
    const uint32_t c = ties->count[lane], fulls = min(((c >> 8) & 255u) + 1u, kManyTies), known = LaneTies::level(c);
    const int before = ties->leaf[0][lane];
    resolveTies(m, ties, px, py, pz, LaneTies::room(c));
    const int win = ties->leaf[0][lane];
    uint32_t level = known;
    if (fulls == kManyTies && (!known || win != before)) {
        level = 0;
        TieRange r{ 0, 0, m.numFaces };
        for (; r.num > 1; ++level) {
            const bool left = win < r.mid();
            if (level >= known && left != leftFirst(m, r.node, px, py, pz)) break;
            r.toChild(left);
        }
        if (level) ties->leaf[kLaneTies - 1][lane] = r.first;
    }
    ties->count[lane] = (level << 16) | (fulls << 8) | 1u;
}

// Runs the last min(qn, 64) queued tests, one per lane, and returns how many stay queued.  TIES: leaves at
// exactly their owner's best are listed, unless they are outside of the subtree that holds the first.
template <bool TIES, bool WIDE>
__device__ __forceinline__ int flushLane(const MeshDev& m, const LaneLds<TIES, WIDE>& l, float px, float py, float pz, int qn)
{
    const int lane = threadIdx.x & 63;
    const int n = qn < 64 ? qn : 64, base = qn - n;
    const bool mine = lane < n;
    waveSync();
    const int owner = l.s->owner[base + (mine ? lane : 0)];
    const float ox = __shfl(px, owner), oy = __shfl(py, owner), oz = __shfl(pz, owner);
    const uint32_t before = TIES ? l.s->best[lane] : 0u;
    float d = 0.f;
    int k = 0;
    if (mine) {
        k = l.s->leaf[base + lane];
        d = leafDistSq(loadLeafLanes(m.tri, k), ox, oy, oz);
        atomicMin(&l.s->best[owner], __float_as_uint(d));
    }
    waveSync();
    if (TIES) {
        if (l.s->best[lane] < before) l.ties->count[lane] = 0;      // a new best: earlier ties are void
        bool pending = mine && l.s->best[owner] == __float_as_uint(d);
        waveSync();
        while (waveBallot(pending)) {
            if (pending) {
                const uint32_t c = l.ties->count[owner], level = LaneTies::level(c);
                if (level && (uint32_t)(k - l.ties->leaf[kLaneTies - 1][owner]) > (uint32_t)m.numFaces >> level) {
                    pending = false;
                } else {
                    const uint32_t at = atomicAdd(&l.ties->count[owner], 1u) & 255u;
                    if (at < LaneTies::room(c)) {
                        l.ties->leaf[at][owner] = k;
                        pending = false;
                    }
                }
            }
            waveSync();
            const uint32_t have = l.ties->count[lane];
            if ((have & 255u) > LaneTies::room(have)) shortenTies(m, l.ties, px, py, pz);
            waveSync();
        }
    }
    return base;
}

// The reference's walk (source/MRMesh/MRMeshProject.cpp:13-103) for one lane: depth-first over boxes, nearer box first, ending
// at the first leaf at most `lo` away.  Returns that distance and leaf, or the least ones.  put / get: the lane's stack; a
// bound that it lowers costs a visit without effect, since a leaf counts only below the best.
template <class Put, class Get>
__device__ __forceinline__ float boxWalk(const MeshDev& m, Put put, Get get, float px, float py, float pz, float up, float lo,
                                         int& leaf, uint32_t& visits)
{
    float best = up;
    leaf = -1;
    int cur = m.rootRef, sp = 0;
    bool have = boxDistSq(m.rootMin[0], m.rootMin[1], m.rootMin[2], m.rootMax[0], m.rootMax[1], m.rootMax[2], px, py, pz) < best;
    for (;;) {
        if (!have) {
            if (sp == 0) break;
            float bound;
            cur = get(--sp, bound);
            if (bound >= best) continue;
        }
        have = false;
        if (cur < 0) {
            const float d = leafDistSq(loadLeafLanes(m.tri, ~cur), px, py, pz);
            if (d < best) {
                best = d;
                leaf = ~cur;
                if (d <= lo) break;
            }
            continue;
        }
        ++visits;
        const size_t rec = 4 * (size_t)cur;
        const float4 n0 = gload(m.dnode, rec), n1 = gload(m.dnode, rec + 1), n2 = gload(m.dnode, rec + 2), n3 = gload(m.dnode, rec + 3);
        const float d1 = boxDistSq(n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, px, py, pz);
        const float d2 = boxDistSq(n1.z, n1.w, n2.x, n2.y, n2.z, n2.w, px, py, pz);
        const bool leftNear = d1 < d2;
        const int l = __float_as_int(n3.x), r = __float_as_int(n3.y);
        const float dn = leftNear ? d1 : d2, df = leftNear ? d2 : d1;
        if (df < best) put(sp++, leftNear ? r : l, df);
        if (dn < best) { cur = leftNear ? l : r; have = true; }
    }
    return best;
}

// Walks every lane's query for the leaves nearer than `up` (squared); lanes with walk = false only help.
// Returns the lane's least squared distance, or `up` where nothing is nearer.
// TIES: *leaf = the leaf that the reference's walk would return (the first in the query's own order among
// those at the least distance), -1 without one.
//
// A lane without work of its own takes over the oldest pending subtree of another lane's query (`own`: the
// query a lane works for); bests and ties are kept by query, so the results do not notice.  Walks differ in
// length -- half the lanes' visits on one grid, ten times the mean near a medial axis -- and a wave took as
// many steps as its longest.  Without and with: 1,000 points on 20 k triangles 160 -> 101 us, 64^3 on them
// 0.67 -> 0.39 ms, 2^22 points on 1.3 M triangles 3.31 -> 2.97 ms, 256^3 on them 11.6 -> 11.0 ms; thresholds
// (kTakeBelow) of 40 to 56 are alike, 16 gains less.
//
// The vector units bound the large launches (96 % of their cycles on the volume), and whatever one lane needs
// the wave issues.  So a round is one straight pass: one look for leaves, at most kPops stack entries, one
// step; a lane that has no internal node by then sits out that step, where a loop until every lane had one
// issued about 190 vector instructions a step.  With the loop and with rounds of 1 / 2 / 3 entries: 2^22
// points 2.95 -> 2.39 / 2.33 / 2.53 ms, 256^3 11.1 -> 9.19 / 9.13 / 9.51 ms, 1,000 points 97 -> 71 / 75 / 77 us.
//
// Queries farther away than m.farSq are answered by boxWalk: the relative slack of the limit grows with the distance until
// it holds the whole mesh, while boxes' distances are compared as they are.
//
// BAND: a query with a leaf at most `lo` away ends there and is answered by boxWalk, whose result depends on the
// reference's order of visits (a query without one has its least distance in any order).  Its stack (8 bytes an
// entry) costs a third of the waves, so only launches with a low limit have it.  Against the wave-cooperative walk
// that carries the order as keys: a band of 1.5 to 4.5 voxels in 190^3 around 1.3 M triangles 6.4 -> 1.4 ms, 48^3
// 14.1 -> 0.34; 300 k projections there with a limit of 0.03 36 -> 0.77, on 20 k triangles 1.9 -> 0.22 ms.
template <bool TIES, bool WIDE, bool BAND = false>
__device__ __forceinline__ float laneWalk(const MeshDev& m, const LaneLds<TIES, WIDE>& l, float qx, float qy, float qz, float up,
                                          bool walk, int statSteps, int statTests, int* leaf = nullptr, float lo = 0.f)
{
    const int lane = threadIdx.x & 63;
    const float unit = m.cylUnit;
    float px = qx, py = qy, pz = qz;
    int own = lane, cur = kNoNode, base = 0, sp = 0, qn = 0;      // pending: entries base .. sp - 1
    uint32_t nStep = 0, nVisit = 0, nTest = 0;      // measurement counts
    const auto rootDistSq = [&] {
        return boxDistSq(m.rootMin[0], m.rootMin[1], m.rootMin[2], m.rootMax[0], m.rootMax[1], m.rootMax[2], qx, qy, qz);
    };
    const bool some = walk && m.numFaces > 0;
    if (some) {
        const float d = rootDistSq();
        if (d < up && !(d > m.farSq)) cur = m.rootRef;
    }
    const uint32_t upBits = cur == kNoNode ? 0u : __float_as_uint(up);
    waveSync();
    l.s->best[lane] = upBits;
    if (TIES) l.ties->count[lane] = 0;
    float limit = laneLimit(__uint_as_float(upBits));
    for (;;) {
        // leaves go to the queue
        const bool isLeaf = cur < 0 && cur != kNoNode;
        const uint64_t lm = waveBallot(isLeaf);
        if (lm) {
            if (isLeaf) {
                const int at = qn + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(lm >> 32),
                                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)lm, 0u));
                l.s->leaf[at] = ~cur;
                l.s->owner[at] = (uint8_t)own;
                cur = kNoNode;
            }
            qn += __popcll(lm);
        }
#pragma unroll
        for (int i = 0; i < kPops; ++i) {
            if (cur == kNoNode && sp > base) {
                --sp;
                float bound;
                const int r = l.get(64 * sp + lane, bound);
                if (bound <= limit) cur = r;
            }
        }
        const uint64_t busy = waveBallot(cur != kNoNode || sp > base);
        const int walking = __popcll(busy);
        if (qn >= 64 || qn >= walking) {
            if (!qn) break;
            nTest += (uint32_t)(qn < 64 ? qn : 64);
            qn = flushLane(m, l, qx, qy, qz, qn);
            const float b = __uint_as_float(l.s->best[own]);
            limit = laneLimit(b);
            if (BAND && b < __shfl(up, own) && b <= lo) limit = -1.f;
        }
        if (walking <= kTakeBelow) {
            const bool gives = sp - base > (cur == kNoNode ? 1 : 0);
            const uint64_t gm = waveBallot(gives);
            if (gm) {
                const uint64_t im = ~busy;
                const int n = __popcll(gm) < __popcll(im) ? __popcll(gm) : __popcll(im);
                const uint64_t rankOf = gives ? gm : im;
                const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(rankOf >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)rankOf, 0u));
                if (gives) l.s->owner[64 + rank] = (uint8_t)lane;
                waveSync();
                const bool takes = ((im >> lane) & 1) && rank < n;
                const int from = takes ? l.s->owner[64 + rank] : lane;
                const int entry = 64 * __shfl(base, from) + from;
                const float x = __shfl(px, from), y = __shfl(py, from), z = __shfl(pz, from), lim = __shfl(limit, from);
                const int o = __shfl(own, from);
                if (takes) {
                    float bound;
                    const int r = l.get(entry, bound);
                    if (bound <= lim) {
                        cur = r;
                        own = o;
                        px = x; py = y; pz = z;
                        limit = lim;
                        base = sp = 0;
                    }
                }
                if (gives && rank < n) ++base;
                waveSync();
            }
        }
        const uint64_t act = waveBallot(cur >= 0);
        if (!act) continue;
        ++nStep;
        nVisit += (uint32_t)__popcll(act);
        if (cur >= 0) {
            float4 a0, b0, a1, b1;
            if (WIDE) {
                const size_t rec = 4 * (size_t)cur;
                a0 = gload(m.cyl, rec); b0 = gload(m.cyl, rec + 1); a1 = gload(m.cyl, rec + 2); b1 = gload(m.cyl, rec + 3);
            } else {
                const uint32_t rec = 4u * (uint32_t)cur;
                a0 = gload(m.cyl, rec); b0 = gload(m.cyl, rec + 1); a1 = gload(m.cyl, rec + 2); b1 = gload(m.cyl, rec + 3);
            }
            float c0, c1;
            const float d0 = cylinderDistSq(a0, b0, unit, px, py, pz, c0);
            const float d1 = cylinderDistSq(a1, b1, unit, px, py, pz, c1);
            const int r0 = __float_as_int(b0.w), r1 = __float_as_int(b1.w);
            // the child with the nearer centre first: while both bounds still hold the point (or nearly), they
            // say little, the centres say on which side the surface is nearer.  Against the nearer bound first:
            // 102 instead of 217 visits and 10 instead of 37 leaf tests per voxel at 1.3 M triangles, 256^3
            const bool first = c0 <= c1, go0 = d0 <= limit, go1 = d1 <= limit;
            cur = go0 && (first || !go1) ? r0 : go1 ? r1 : kNoNode;
            if (go0 && go1) {
                l.put(64 * sp + lane, first ? r1 : r0, first ? d1 : d0);
                ++sp;
            }
        }
    }
    waveSync();
    const uint32_t b = l.s->best[lane];
    const bool found = b < upBits;
    const bool within = BAND && found && __uint_as_float(b) <= lo;
    bool far = false;      // found again: kept across the loop it cost small volumes 1 %
    if (some && upBits == 0u) {
        const float r = rootDistSq();
        far = r < up && r > m.farSq;
    }
    const bool boxes = far || within;
    float d = found ? __uint_as_float(b) : up;
    int at = -1;
    uint32_t nBox = 0;
    if (boxes) {
        if (BAND) {
            int2* const stack = l.band();
            d = boxWalk(m, [=](int sp, int ref, float bound) { stack[64 * sp + lane] = make_int2(ref, __float_as_int(bound)); },
                        [=](int sp, float& bound) {
                            const int2 e = stack[64 * sp + lane];
                            bound = __int_as_float(e.y);
                            return e.x;
                        }, qx, qy, qz, up, lo, at, nBox);
        } else {
            d = boxWalk(m, [&](int sp, int ref, float bound) { l.put(64 * sp + lane, ref, bound); },
                        [&](int sp, float& bound) { return l.get(64 * sp + lane, bound); }, qx, qy, qz, up, -1.f, at, nBox);
        }
    }
    if (m.stats) {
        statAdd(m, kStatWalks, 1);
        statAdd(m, statSteps, nStep);
        statAdd(m, statTests, nTest);
        statAdd(m, kStatLaneVisits, nVisit);
        if (boxes) atomicAdd(&m.stats[kStatLaneVisits], (unsigned long long)nBox);
    }
    if (boxes) {
        if (TIES) *leaf = at;
        return d;
    }
    if (TIES) {
        *leaf = -1;
        if (found) {
            resolveTies(m, l.ties, qx, qy, qz, l.ties->count[lane] & 255u);
            *leaf = l.ties->leaf[0][lane];
        }
    }
    return d;
}

} // namespace
} // namespace mi
