// Host restatement of the lane walks' bound -- the cylinder records of mi_volume.hip and cylinderDistSq of mi_lane.hpp --
// with the margins of mi_bound.hpp, and of the leaf test that it guards (the FP64 closest point of
// closestPointInTriangle, source/MRMesh/MRClosestPointInTriangle.h:27-87, rounded to float and squared in float).  The
// walks are exact only if a bound is never above the limit of its own leaves' least distance.  The raw square root is
// taken one unit too large.
// usage: lane_bound_fuzz SEED COUNT  -> exit 0 when no sample violates the bound
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>
#include "../../meshlib_amd/csrc/mi_bound.hpp"

struct Tri { float v[3][3]; };
struct Cyl { float c[3], n[3], t, r; };

static double dot3(const double* a, const double* b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }

static void closest(const double p[3], const double a[3], const double b[3], const double c[3], double pr[3])
{
    double ab[3], ac[3], ap[3], bp[3], cp[3];
    for (int k = 0; k < 3; ++k) { ab[k] = b[k] - a[k]; ac[k] = c[k] - a[k]; ap[k] = p[k] - a[k]; bp[k] = p[k] - b[k]; cp[k] = p[k] - c[k]; }
    const auto at = [&](const double* o, double v, const double* e, double w, const double* f) {
        for (int k = 0; k < 3; ++k) pr[k] = o[k] + v * e[k] + w * f[k];
    };
    const double d1 = dot3(ab, ap), d2 = dot3(ac, ap), d3 = dot3(ab, bp), d4 = dot3(ac, bp), d5 = dot3(ab, cp), d6 = dot3(ac, cp);
    if (d1 <= 0 && d2 <= 0) return at(a, 0, ab, 0, ac);
    if (d3 >= 0 && d4 <= d3) return at(b, 0, ab, 0, ac);
    if (d6 >= 0 && d5 <= d6) return at(c, 0, ab, 0, ac);
    const double vc = d1 * d4 - d3 * d2;
    if (vc <= 0 && d1 >= 0 && d3 <= 0) return at(a, d1 / (d1 - d3), ab, 0, ac);
    const double vb = d5 * d2 - d1 * d6;
    if (vb <= 0 && d6 <= 0 && d2 >= 0) return at(a, 0, ab, d2 / (d2 - d6), ac);
    const double va = d3 * d6 - d5 * d4;
    if (va <= 0) {
        if (d4 < d3) return at(b, 0, ab, 0, ac);
        if (d5 < d6) return at(c, 0, ab, 0, ac);
        const double bc[3] = { c[0] - b[0], c[1] - b[1], c[2] - b[2] };
        return at(b, (d4 - d3) / ((d4 - d3) + (d5 - d6)), bc, 0, ac);
    }
    const double den = 1 / (va + vb + vc);
    at(a, vb * den, ab, vc * den, ac);
}

static float leafDistSq(const Tri& T, const float p[3])
{
    double q[3][3], pd[3] = { p[0], p[1], p[2] }, pr[3];
    for (int i = 0; i < 3; ++i) for (int k = 0; k < 3; ++k) q[i][k] = T.v[i][k];
    closest(pd, q[0], q[1], q[2], pr);
    const float x = (float)pr[0] - p[0], y = (float)pr[1] - p[1], z = (float)pr[2] - p[2];
    return x * x + y * y + z * z;
}

static float halfUp(float x)
{
    if (!(x <= 65504.f)) return INFINITY;
    const double step = std::ldexp(1.0, std::max(std::ilogb(std::max(x, 1e-30f)), -14) - 10);
    return (float)(std::ceil((double)x / step) * step);
}

static void axis(const float d[3], float n[3])
{
    const float big = std::max(std::fabs(d[0]), std::max(std::fabs(d[1]), std::fabs(d[2])));
    n[0] = 1; n[1] = n[2] = 0;
    if (big > 0 && big < INFINITY) {
        const float x = d[0] / big, y = d[1] / big, z = d[2] / big, len = std::sqrt(x * x + y * y + z * z);
        n[0] = x / len; n[1] = y / len; n[2] = z / len;
    }
}

static void along(const Cyl& f, const float* v, float& h, float& rr)
{
    const float x = v[0] - f.c[0], y = v[1] - f.c[1], z = v[2] - f.c[2];
    h = x * f.n[0] + y * f.n[1] + z * f.n[2];
    const float a = x - h * f.n[0], b = y - h * f.n[1], c = z - h * f.n[2];
    rr = a * a + b * b + c * c;
}

static float longest(const Tri& T, float e[3])
{
    float best = -1;
    for (int i = 0; i < 3; ++i) {
        const float *p = T.v[i], *q = T.v[(i + 1) % 3];
        const float x = q[0] - p[0], y = q[1] - p[1], z = q[2] - p[2], l = x * x + y * y + z * z;
        if (l > best) { best = l; e[0] = x; e[1] = y; e[2] = z; }
    }
    return best;
}

static void finish(Cyl& f, float t, float r, float big, float unit)
{
    const float wide = big * mi::kWidenCoord + (t + r) * mi::kWidenSize;
    f.t = halfUp((t + wide) / unit);
    f.r = halfUp((r + wide) / unit);
}

// kRodArea of mi_volume.hip
static const float kRodArea = 0.1f;

static Cyl inner(const std::vector<Tri>& ts, float unit)
{
    Cyl f;
    float mn[3], mx[3], dir[3] = { 0, 0, 0 }, area = 0, big = 0;
    for (int k = 0; k < 3; ++k) { mn[k] = INFINITY; mx[k] = -INFINITY; }
    for (const Tri& T : ts) {
        for (int i = 0; i < 3; ++i) for (int k = 0; k < 3; ++k) { mn[k] = std::min(mn[k], T.v[i][k]); mx[k] = std::max(mx[k], T.v[i][k]); }
        float ab[3], ac[3];
        for (int k = 0; k < 3; ++k) { ab[k] = T.v[1][k] - T.v[0][k]; ac[k] = T.v[2][k] - T.v[0][k]; }
        const float c[3] = { 0.5f * (ab[1] * ac[2] - ab[2] * ac[1]), 0.5f * (ab[2] * ac[0] - ab[0] * ac[2]), 0.5f * (ab[0] * ac[1] - ab[1] * ac[0]) };
        for (int k = 0; k < 3; ++k) dir[k] += c[k];
        area += std::sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
    }
    float dd = 0;
    for (int k = 0; k < 3; ++k) {
        mn[k] = std::nextafter(mn[k], -INFINITY); mx[k] = std::nextafter(mx[k], INFINITY);
        f.c[k] = 0.5f * mn[k] + 0.5f * mx[k];
        big = std::max(big, std::max(std::fabs(mn[k]), std::fabs(mx[k])));
        dd += (mx[k] - mn[k]) * (mx[k] - mn[k]);
    }
    axis(dir, f.n);
    float e[3];
    if (area < kRodArea * dd && longest(ts[ts.size() / 2], e) >= 0.25f * dd) axis(e, f.n);
    float hi = -INFINITY, lo = -INFINITY, rr = 0;
    for (const Tri& T : ts) for (int i = 0; i < 3; ++i) {
        float a, b;
        along(f, T.v[i], a, b);
        hi = std::max(hi, a); lo = std::max(lo, -a); rr = std::max(rr, b);
    }
    lo = -lo;
    const float mid = 0.5f * hi + 0.5f * lo;
    double off = 0, offSq = 0;
    for (int k = 0; k < 3; ++k) {
        const float c = f.c[k] + mid * f.n[k];
        const double e1 = c - ((double)f.c[k] + (double)mid * f.n[k]);
        off += e1 * f.n[k];
        offSq += e1 * e1;
        f.c[k] = c;
    }
    finish(f, 0.5f * hi - 0.5f * lo + 1.001f * (float)std::fabs(off),
           std::sqrt(rr) + 1.001f * std::sqrt((float)std::max(offSq - off * off, 0.0)), big, unit);
    return f;
}

static Cyl leafCylinder(const Tri& T, float unit)
{
    Cyl f;
    double e[3][3], len[3];
    float big = 0;
    for (int i = 0; i < 3; ++i) {
        len[i] = 0;
        for (int k = 0; k < 3; ++k) { e[i][k] = (double)T.v[(i + 1) % 3][k] - T.v[i][k]; len[i] += e[i][k] * e[i][k]; big = std::max(big, std::fabs(T.v[i][k])); }
    }
    const float nn[3] = { (float)(e[0][1] * e[1][2] - e[0][2] * e[1][1]), (float)(e[0][2] * e[1][0] - e[0][0] * e[1][2]),
                          (float)(e[0][0] * e[1][1] - e[0][1] * e[1][0]) };
    const int l = len[1] > len[0] ? (len[2] > len[1] ? 2 : 1) : (len[2] > len[0] ? 2 : 0), i1 = (l + 1) % 3, i2 = (l + 2) % 3;
    double w[3] = { 0, 0, 0 };
    const double wa = len[1] * (len[0] + len[2] - len[1]), wb = len[2] * (len[0] + len[1] - len[2]), wc = len[0] * (len[1] + len[2] - len[0]), sum = wa + wb + wc;
    if (len[l] < len[i1] + len[i2] && sum > 0) { w[0] = wa / sum; w[1] = wb / sum; w[2] = wc / sum; }
    else { w[l] = 0.5; w[i1] = 0.5; }
    for (int k = 0; k < 3; ++k) f.c[k] = (float)(w[0] * T.v[0][k] + w[1] * T.v[1][k] + w[2] * T.v[2][k]);
    axis(nn, f.n);
    float edge[3];
    const float ls = longest(T, edge);
    if (0.5f * std::sqrt(nn[0] * nn[0] + nn[1] * nn[1] + nn[2] * nn[2]) < kRodArea * ls) axis(edge, f.n);
    float t = 0, rr = 0;
    for (int i = 0; i < 3; ++i) {
        float h, q;
        along(f, T.v[i], h, q);
        t = std::max(t, std::fabs(h)); rr = std::max(rr, q);
    }
    finish(f, t, std::sqrt(rr), big, unit);
    return f;
}

static float boundSq(const Cyl& f, float unit, const float p[3])
{
    const float yx = p[0] - f.c[0], yy = p[1] - f.c[1], yz = p[2] - f.c[2];
    const float h = std::fmaf(f.n[2], yz, std::fmaf(f.n[1], yy, f.n[0] * yx));
    const float vx = std::fmaf(-h, f.n[0], yx), vy = std::fmaf(-h, f.n[1], yy), vz = std::fmaf(-h, f.n[2], yz);
    const float rr = std::fmaf(vz, vz, std::fmaf(vy, vy, vx * vx));
    const float rho = std::nextafter(std::sqrt(rr), INFINITY);
    const float s = std::fmax(std::fmaf(-f.t, unit, std::fabs(h)), 0.f), q = std::fmax(std::fmaf(-f.r, unit, rho), 0.f);
    return std::fmaf(s, s, q * q);
}

int main(int argc, char** argv)
{
    std::mt19937_64 g(argc > 1 ? atoll(argv[1]) : 1);
    const long count = argc > 2 ? atol(argv[2]) : 1000000;
    std::uniform_real_distribution<double> U(-1, 1);
    long n = 0, bad = 0;
    double used = 0;
    for (long it = 0; it < count; ++it) {
        // a flat, oblique patch of a few triangles, small against its coordinates, which lie just above powers of two
        // (one patch in four: anywhere, any shape)
        const bool any = it % 4 == 3;
        const double at[] = { 1, 2, 32, 1024, 0.25, 1 };
        const double base = at[g() % 6], size = base * std::pow(10.0, -1 - 4.5 * std::fabs(U(g)));
        double o[3], n3[3], e1[3], e2[3];
        for (int k = 0; k < 3; ++k) {
            o[k] = any ? base * 3 * U(g) : base * (1 + 0.05 * std::fabs(U(g))) * (it % 5 == 4 && g() % 2 ? -1 : 1);
            n3[k] = any ? U(g) : 1 + 0.1 * U(g);
            e1[k] = U(g);
        }
        if (it % 5 == 4) for (int k = 0; k < 3; ++k) if (o[k] < 0) n3[k] = -n3[k];
        const double ln = std::sqrt(dot3(n3, n3));
        for (int k = 0; k < 3; ++k) n3[k] /= ln;
        double d = dot3(e1, n3);
        for (int k = 0; k < 3; ++k) e1[k] -= d * n3[k];
        const double l1 = std::sqrt(dot3(e1, e1)) + 1e-9;
        for (int k = 0; k < 3; ++k) e1[k] /= l1;
        for (int k = 0; k < 3; ++k) e2[k] = n3[(k + 1) % 3] * e1[(k + 2) % 3] - n3[(k + 2) % 3] * e1[(k + 1) % 3];
        const int tris = 1 + (int)(g() % 4);
        const double thin = g() % 4 == 0 ? std::pow(10.0, -4 * std::fabs(U(g))) : 1, bump = any ? 0.3 * size : g() % 2 ? 1e-3 * size : 0;
        std::vector<Tri> ts(tris);
        for (Tri& T : ts) for (int i = 0; i < 3; ++i) {
            const double a = size * U(g), b = size * thin * U(g), c = bump * U(g);
            for (int k = 0; k < 3; ++k) T.v[i][k] = (float)(o[k] + a * e1[k] + b * e2[k] + c * n3[k]);
        }
        // the unit of a mesh from this patch's size up to 10,000 times that
        const float unit = (float)std::ldexp(1.0, std::ilogb(size * std::pow(10.0, 4 * std::fabs(U(g)))) + 2 - 15);
        std::vector<Cyl> cyl;
        cyl.push_back(inner(ts, unit));
        for (const Tri& T : ts) cyl.push_back(leafCylinder(T, unit));
        for (int q = 0; q < 8; ++q) {
            const Tri& T = ts[g() % tris];
            double u = std::fabs(U(g)), w = std::fabs(U(g));
            if (u + w > 1) { u = 1 - u; w = 1 - w; }
            if (q % 4 == 1) { u = 0; w = 0; }
            if (q % 4 == 2) w = 0;
            const double h = size * std::pow(10.0, 2.0 - 6.0 * std::fabs(U(g))) * (g() % 2 ? 1 : -1), side = q % 2 ? h : h * 1e-2;
            float p[3];
            for (int k = 0; k < 3; ++k)
                p[k] = (float)(T.v[0][k] + u * (T.v[1][k] - T.v[0][k]) + w * (T.v[2][k] - T.v[0][k]) + h * n3[k] + side * (U(g) * e1[k] + U(g) * e2[k]));
            std::vector<float> own;
            float least = INFINITY;
            for (const Tri& L : ts) { own.push_back(leafDistSq(L, p)); least = std::fmin(least, own.back()); }
            for (size_t k = 0; k < cyl.size(); ++k) {
                const float b = boundSq(cyl[k], unit, p), dist = k ? own[k - 1] : least;
                if (!(dist < INFINITY)) continue;      // a triangle without area may have none
                ++n;
                if (!(b <= std::fmaf(dist, 1.f + mi::kLimitSlack, 1e-37f))) {
                    if (++bad < 6) printf("BAD %s: bound %.9g, leaf %.9g (coordinates %g, size %g)\n", k ? "leaf" : "node", b, dist, base, size);
                }
                if (dist > 0) used = std::max(used, ((double)b / dist - 1) / mi::kLimitSlack);
            }
        }
    }
    printf("bounds %ld, largest share of the limit's slack %.3f, bad %ld\n", n, used, bad);
    return bad != 0;
}
