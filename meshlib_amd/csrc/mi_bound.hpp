// mi_bound.hpp -- the margins of the lane walks' bounds (host and device; also read by the bounds' host check).
//
// A child's cylinder (mi_volume.hip) bounds its triangles if no error of the arithmetic exceeds what t and r are widened
// by and what the walk adds to its limit.  With u = 2^-24, M the node's largest coordinate, D the true distance:
//
//  of M (kWidenCoord): the leaf test rounds its closest point to float, at most u per coordinate relative to M, hence
//    sqrt(3) u M in length, 0.8661 * 2^-23 M.  An inner node's centre is moved along its axis and rounded after the
//    vertices' offsets were taken from the unmoved one, as much again at worst; what it is in each case is added to t and
//    r (200 k points on 1.3 M triangles 1,000 / 10,000 sizes from the origin: 0.74 / 5.2 ms, the worst case 1.2 / 10).
//  of t + r (kWidenSize), in units of u (t + r): the offsets from the box's centre, whose length is at most sqrt(3) times
//    sqrt(t^2 + r^2), give 7 along the axis (rounded offset and dot product) and 16 across it; the shift with an axis whose
//    squared length is 1 +- 7 u 12 along; the rounding of the half range and of the shift 4; the walk's own
//    projection of the part of its offset inside the cylinder 4 along and 10 across.  Together 27 and 30, below 32.
//  of D (kLimitSlack), in units of u D: the walk's projection of the rest of its offset 10.3, its differences and sum 2,
//    the axis's length 3.5, the leaf test's differences and squares 2.5: 18.3, hence 37 u of the squared distance.
//    Results below the normal range are covered by an absolute 1e-37.
#pragma once

namespace mi {

constexpr float kWidenCoord = 0x1.cp-24f;      // 0.875 * 2^-23
constexpr float kWidenSize = 0x1p-19f;
constexpr float kLimitSlack = 0x1.8p-19f;      // 48 u

} // namespace mi
