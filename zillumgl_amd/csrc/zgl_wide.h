// zgl_wide.h -- closest-hit and any-hit walks over a 4-wide tree, with results equal to
// the reference's MTBVH walk (intersection.glsl:367-427) bit for bit; host and device.
//
// What bounds the reference's walk is its rows: on the 819,400-triangle scene a walk visits
// 56 of them on average, each a dependent 32-byte load and an exact box test of about 45
// vector instructions.  Only two things of that walk reach its result: which triangles' own
// boxes and all their ancestors' boxes pass the box test, and the order in which hits
// shrink the distance.  The walk here visits a collapsed tree of the same leaves (four
// children per 64-byte node, FP16 planes rounded outwards and padded, nearest child
// first), tests no box exactly, and then shows for the triangle it found that the
// reference's walk finds it too; a ray for which that cannot be shown is walked again over
// the reference's rows.
//
// Why the result is the reference's.  Write lo/hi for a box's slab distances as boxHit
// computes them.  Subtraction of the origin and multiplication by 1/d are monotone in
// FP32, so a leaf's slab intervals lie inside every ancestor's, exactly, and of the box
// test's conditions `hi >= 0`, `hi >= lo` and `entry <= dist` hold for all ancestors when
// they hold for the leaf.  The overlap tests (dt.y + dt.z > tyz, that is mx.y > mn.z, and
// the other two pairs) are not monotone, because each side is rounded; but the rounding
// error of an ancestor's test is below 5 u (Ty + Tz), where u = 2^-24 and T bounds the slab
// distances of the whole scene's box, and the ancestor's margin mx.y - mn.z is at least
// the leaf's.  So a leaf whose margins exceed 8 u (Ty + Tz) passes together with all its
// ancestors.
//   * The walk here visits every leaf whose box passes in the reference (its boxes
//     contain the exact ones, with room for the rounding of both sides), up to the
//     distance at which it drops subtrees (wideLimit).
//   * Let W be its closest hit at t, t2 the next larger hit distance it met (the ray's
//     limit if none), b the entry distance of W's exact box, and T a little more than t.  No
//     triangle in a dropped subtree has a hit distance of T or less (below).  If W's box
//     passes with those margins, t < t2, b <= t2 and b <= T, then whenever the
//     reference's walk comes to W its distance is still above t and at least b: W is
//     tested, and nothing is nearer.  So the reference's closest hit is W whatever order
//     it visits the leaves in.  Where only the margins fail (about one hit in a thousand),
//     the reference's box test can be made on W's ancestors themselves (CHAIN), a fifth of
//     a walk over the rows.
//   * Without a hit the reference has none either.  For an any-hit ray, which drops
//     nothing, one hit that passes with these margins and b <= the limit shows that it is
//     occluded.
//
// How far a hit lies from its triangle.  Write X = |ab| |ac|, R = |a - o|, |d| = 1, and det as
// intersectTriangle computes it.  Cramer's identity det ao + num d = u ab + v ac holds
// exactly for exact determinants; the computed ones, all of them small beside their terms
// where the ray is nearly edge-on, are each off by at most 3.66 u times the product of
// their three vectors' lengths.  With u, v >= 0 and u + v <= det the point o + t d is
// therefore within 14.7 u X R / det (and a few u R) of the triangle.  Edge-on, where det
// comes near its cut-off of 1e-6, that is 0.9 X R: not small unless X is, and t can lie
// well in front of the triangle's own box.  So no fixed widening of the distance lets a
// walk drop subtrees; each triangle has to be of one of four kinds (wideClassify):
//   * small: X at most kWideSmall and its box's diagonal at most bound / 8.  The ray is in
//     the box at its entry e and within 0.9 X R of the triangle at t, so e - t is at most
//     the diagonal and 1.03 * 0.9 X (t + diagonal) / (1 - 0.9 X).
//   * flat: in a plane of constant x, y or z.  Every product of det, num and of the errors
//     then carries the same component of d or of o - a, t is accurate to 6 u / s whatever
//     the angle (s the sine of the angle at a) and e is at most the flat slab's distance.
//   * never hit: det stays below its cut-off for every ray.
//   * large: everything else.  det >= g s X (but for 0.4%) where g = |d.N|.  Of the four terms
//     of the offset between the point at t and the triangle two are along d and two along
//     ab and ac, each pair 7.4 u (R + edge / 2) / (g s) at most; only the latter move the
//     ray's entry, by their component on the entry's axis over d's, which is at least the
//     smallest component h of d.  So e - t <= (7.4 (1 / h + 2) / (g s) + 10 / h) u (t + 1.5
//     edge), and a ray with g s (h - 10 K u) >= 7.6 K u (1 + 2 h) for every large triangle's
//     plane (wideClear) has e - t <= (t + 1.5 edge) / K.  A walk of another ray, one in a
//     few hundred, is made again and drops no subtree (wideWhole).  The planes are few
//     where a scene has large triangles, walls and floors; of a scene with more than
//     kWidePlanes no walk drops any.  Dropping nothing costs 25 to 50% on the caustics box,
//     whose rays go on through the sphere's back.
// wideMargins makes from the scene's largest X, diagonal and edge the limit (rel, slack)
// up to which a walk has to keep subtrees.
//
// Measured: the headline launch's walks visit 15 nodes and 3 triangles each (as it was counted
// with subtrees dropped at 1.001 t: 14 and 2.8); 64 passes at 1080p take 100 ms, 169 over the
// rows, 95 with subtrees dropped at 1.001 t.  A node step is about 110 vector instructions
// for four boxes (fma_mix reads the FP16 planes in place) against 45 for one row.
//
// Rays the argument does not cover take the reference's rows from the start: nearly
// axis-parallel ones (RayPre::mode != 0), components below 1e-6, not finite, from far
// outside the scene, or with a direction longer than 1 or shorter (any-hits: than 0.5).
// For a ray with one component below 1e-6 the reference's test drops that axis' slab, and
// its walk visits every box of a slice through the scene (one ray in a 1280 x 720 pass over
// 205,000 triangles held up the launch to 15 ms).  Boxes further from the ray on that axis
// than a hit can lie beside its triangle are left out of that walk (rowHit), which leaves
// about 80 rows: the pass takes 1.4 ms alone and 0.9 among others.
#pragma once

#include "zgl_box.h"

namespace zgl {

// A slot of the wide tree is 64 bytes: a node or a triangle.
//   node:     {origin.xyz, child} {loX, loY} {loZ, hiX} {hiY, hiZ}; each lo/hi group is four
//             FP16 offsets from origin, one per child, in units of WalkMem::unit; `child` is
//             the first child's slot (28 bits) and a leaf bit per child (bits 28..31).
//             Children lie in consecutive slots; a missing child's box is empty.
//   triangle: {a.xyz, b.x} {b.yz, c.xy} {c.z, primitive, its rows in the six tables}
// Slot 0 is the root.
constexpr uint32_t kWideSlotMask = 0x0fffffffu;
constexpr int kWideLeafBit = (int)0x80000000;
constexpr uint32_t kHalfInf = 0x7c00u, kHalfNegInf = 0xfc00u;

// Walk stack: entries per lane, in LDS: 36 KB for a workgroup of 256, so that four
// workgroups fit a compute unit.  A ray that comes to a node with fewer than three free
// entries is walked over the rows.
constexpr int kWalkStack = 18;
constexpr int kWalkLanes = 256;

#if defined(__HIP_DEVICE_COMPILE__)
typedef uint32_t WideU4 __attribute__((ext_vector_type(4)));
typedef const WideU4 __attribute__((address_space(1)))* WideSlots;
typedef float GFloat4 __attribute__((ext_vector_type(4)));
typedef const GFloat4 __attribute__((address_space(1)))* GRows;
#else
struct WideU4 { uint32_t x, y, z, w; };
typedef const WideU4* WideSlots;
struct GFloat4 { float x, y, z, w; };
typedef const GFloat4* GRows;
#endif
// A stacked subtree: its parent's child word and its key (entry distance and child number).
struct WalkEntry { uint32_t word, key; };

// A plane of large triangles (wideClear).  kWideClear is K at the top of the file: a larger
// one drops more and walks more rays twice.
constexpr double kWideClear = 64.0;
constexpr int kWidePlanes = 16;
struct WidePlane { float x, y, z, w; };

// Up to what distance a walk keeps subtrees, for which rays, and how far beside its triangle
// a hit can lie (see the top of the file).
struct WideMargins {
    float rel, slack;            // the limit is rel * distance + slack (infinite: nothing is dropped)
    float grow, growRel, reach;  // wideGrowth
    int nPlanes;
    WidePlane planes[kWidePlanes];
};

// The scene as a walk sees it.
struct WalkMem {
    GRows rows;        // the reference's row tables
    GRows tris;        // 48 bytes per triangle
    WideSlots wide;    // null: every ray takes the rows
    int bvhSize;
    float unit;        // world length of one FP16 unit of the planes (a power of two)
    float bound;       // largest absolute coordinate of the scene's box
    float rel, slack;  // margins->rel, ->slack
    const WideMargins* margins;
};

// Sizes derived from the scene's box: bound = its largest absolute coordinate, pad = what
// every box is grown by on each side, unit = the planes' quantum.  `ok` is false where the
// FP16 planes or the error bounds would not hold (empty, tiny, huge or not finite).
struct WideScale {
    float bound, pad, unit;
    bool ok;
};

ZGL_HD WideScale wideScale(const float* lo, const float* hi)
{
    WideScale w{0.0f, 0.0f, 1.0f, false};
    float extent = 0.0f;
    for (int c = 0; c < 3; c++) {
        const float a = __builtin_fabsf(lo[c]), b = __builtin_fabsf(hi[c]), e = hi[c] - lo[c];
        w.bound = __builtin_fmaxf(w.bound, __builtin_fmaxf(a, b));
        extent = __builtin_fmaxf(extent, e);
        if (!(a <= 1e9f && b <= 1e9f && e >= 0.0f)) return w;
    }
    if (!(w.bound >= 1e-9f)) return w;
    // Errors of one slab distance as a length along its axis: with |plane - o| <= 5 bound
    // (origins are within 4 bound) at most 5 bound 3 2^-24 here and 5 bound 2 2^-24 in the
    // reference, 1.5e-6 bound together; 2^-18 bound is 2.5 times that.
    w.pad = w.bound * 3.814697265625e-06f;
    // extents reach [2^14, 2^15) units: inside FP16's range with one binade to spare
    const uint32_t e = (fbits(extent + 4.0f * w.pad) >> 23) & 0xffu;
    w.unit = bitsf((e - 14u) << 23);
    w.ok = true;
    return w;
}

// What a scene's triangles are to the bound at the top of the file: the largest X and box
// diagonal of the small ones, the longest edge of the large ones, and the large ones' planes,
// each with the smallest sine at a.  The floats are nonnegative and kept as their bits, whose
// order is theirs.
constexpr float kWideSmall = 0.25f;
constexpr int kWidePlaneSlots = 64;
struct WideStats {
    uint32_t x, diagonal, edge;
    uint32_t overflow;  // planes that found no slot
    uint32_t key[kWidePlaneSlots], sine[kWidePlaneSlots];  // key 0: free
};
enum : int { kWideTriSmall, kWideTriFlat, kWideTriNever, kWideTriLarge, kWideTriBad };
struct WideTriClass {
    int kind;
    float x, diagonal, edge, sine;  // rounded up, the sine down
    uint32_t key;                   // a large one's plane (wideNormal)
};
// p: the corners a, b, c.
ZGL_HD WideTriClass wideClassify(const float* p, float bound)
{
    WideTriClass r{kWideTriBad, 0.0f, 0.0f, 0.0f, 0.0f, 0u};
    // the edges as intersectTriangle rounds them
    double ab[3], ac[3], ab2 = 0.0, ac2 = 0.0, bc2 = 0.0, diag2 = 0.0;
    bool flat = false;
    for (int c = 0; c < 3; c++) {
        ab[c] = p[3 + c] - p[c];
        ac[c] = p[6 + c] - p[c];
        ab2 += ab[c] * ab[c];
        ac2 += ac[c] * ac[c];
        bc2 += (ac[c] - ab[c]) * (ac[c] - ab[c]);
        const double less = ab[c] < ac[c] ? ab[c] : ac[c], more = ab[c] < ac[c] ? ac[c] : ab[c];
        const double extent = (more > 0.0 ? more : 0.0) - (less < 0.0 ? less : 0.0);
        diag2 += extent * extent;
        flat = flat || (ab[c] == 0.0 && ac[c] == 0.0);
    }
    const double n[3] = {ab[1] * ac[2] - ab[2] * ac[1], ab[2] * ac[0] - ab[0] * ac[2], ab[0] * ac[1] - ab[1] * ac[0]};
    const double x = __builtin_sqrt(ab2 * ac2), len = __builtin_sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    if (!(x <= 1e30)) return r;  // not finite
    r.x = (float)x * 1.00001f;
    r.diagonal = (float)__builtin_sqrt(diag2) * 1.00001f;
    // |det| <= 1.7321 |n| + 3.66 u 1.7321 X for directions of components up to 1
    if (1.74 * len + 4e-7 * x < 0.9e-6) r.kind = kWideTriNever;
    else if (flat && len >= 0.0625 * x) r.kind = kWideTriFlat;
    else r.kind = r.x <= kWideSmall && r.diagonal <= bound * 0.125f ? kWideTriSmall : kWideTriLarge;
    if (r.kind != kWideTriLarge) return r;
    const double longest = ab2 > ac2 ? (ab2 > bc2 ? ab2 : bc2) : (ac2 > bc2 ? ac2 : bc2);
    r.edge = (float)__builtin_sqrt(longest) * 1.00001f;
    r.sine = (float)(len / x) * 0.99999f;
    if (!(len > 0.0)) return r;  // no plane: key 0
    // the normal's largest component, and the other two over it in steps of 2^-11
    const double m[3] = {n[0] < 0.0 ? -n[0] : n[0], n[1] < 0.0 ? -n[1] : n[1], n[2] < 0.0 ? -n[2] : n[2]};
    const int k = m[0] >= m[1] && m[0] >= m[2] ? 0 : m[1] >= m[2] ? 1 : 2;
    const double ni = k == 0 ? n[1] : n[0], nj = k == 2 ? n[1] : n[2], nk = k == 0 ? n[0] : k == 1 ? n[1] : n[2];
    r.key = ((uint32_t)(k + 1) << 26) | ((uint32_t)(int)(ni / nk * 2048.0 + 2048.5) << 13) |
            (uint32_t)(int)(nj / nk * 2048.0 + 2048.5);
    return r;
}

// The unit normal a key stands for, within 2^-11 / sqrt 2 of every normal of that key up to
// its sign.
ZGL_HD void wideNormal(uint32_t key, double n[3])
{
    const int k = (int)(key >> 26) - 1, i = k == 0 ? 1 : 0, j = k == 2 ? 1 : 2;
    n[k] = 1.0;
    n[i] = ((double)((key >> 13) & 0x1fffu) - 2048.0) / 2048.0;
    n[j] = ((double)(key & 0x1fffu) - 2048.0) / 2048.0;
    const double s = 1.0 / __builtin_sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    for (int c = 0; c < 3; c++) n[c] *= s;
}

inline WideMargins wideMargins(const WideStats& st, const WideScale& sc)
{
    WideMargins m{};
    const double x = bitsf(st.x), c = 0.9 * x, diagonal = bitsf(st.diagonal), edge = bitsf(st.edge);
    // planes: keys next to each other (one plane's triangles round apart) make one
    const double cell = 3.46e-4;
    double n[kWidePlanes][3], away[kWidePlanes], sine[kWidePlanes];
    bool drop = st.overflow == 0;
    for (int i = 0; i < kWidePlaneSlots && drop; i++) {
        if (st.key[i] == 0) continue;
        double v[3], d = 0.0;
        wideNormal(st.key[i], v);
        int at = 0;
        for (; at < m.nPlanes; at++) {
            const double dot = v[0] * n[at][0] + v[1] * n[at][1] + v[2] * n[at][2], sign = dot < 0.0 ? -1.0 : 1.0;
            double d2 = 0.0;
            for (int a = 0; a < 3; a++) d2 += (v[a] - sign * n[at][a]) * (v[a] - sign * n[at][a]);
            d = __builtin_sqrt(d2) + cell;
            if (d <= 5.0 * cell) break;
        }
        if (at == kWidePlanes) {
            drop = false;
        } else if (at == m.nPlanes) {
            for (int a = 0; a < 3; a++) n[at][a] = v[a];
            away[at] = cell;
            sine[at] = bitsf(st.sine[i]);
            m.nPlanes++;
        } else {
            away[at] = d > away[at] ? d : away[at];
            sine[at] = sine[at] < bitsf(st.sine[i]) ? sine[at] : bitsf(st.sine[i]);
        }
    }
    if (!drop) {
        m.nPlanes = 0;
        m.rel = 1.0f;
        m.slack = __builtin_inff();
        m.grow = 8.0f * sc.bound;  // past the scene's end, whatever the distance
        return m;
    }
    double rel = 1.03 * c / (1.0 - c), abs = 1.03 * diagonal / (1.0 - c);
    const bool large = edge > 0.0;
    if (large) {
        rel = rel > 1.05 / kWideClear ? rel : 1.05 / kWideClear;
        abs = abs > 1.6 * edge / kWideClear ? abs : 1.6 * edge / kWideClear;
    }
    m.rel = (float)(1.0009765625 * (1.0 + rel) * 1.00001);
    m.slack = (float)((16.0 * sc.pad + abs) * 1.00001);
    // beside the triangle on an axis with |d_axis| < 1e-6, where of the four terms of the
    // identity's error two are left: small ones 0.22 X (2 R + diagonal) / (1 - 0.22 X); large
    // ones that the ray is clear of with h = 1/16, (R + edge) / 500; flat ones 22 u R / s; the
    // ray's own drift and the box's rounding
    m.grow = (float)(sc.bound * 2.44140625e-4);
    m.growRel = (float)((large && 0.5 * x < 2.1e-3 ? 2.1e-3 : 0.5 * x) * 1.00001);
    m.reach = (float)((diagonal > edge ? diagonal : edge) * 1.00001);
    for (int i = 0; i < m.nPlanes; i++) {
        const double k = sine[i] / (7.6 * kWideClear * 5.9604644775390625e-08);
        m.planes[i].x = (float)(n[i][0] * k);
        m.planes[i].y = (float)(n[i][1] * k);
        m.planes[i].z = (float)(n[i][2] * k);
        m.planes[i].w = (float)((away[i] * 1.02 + 1e-6) * k);
    }
    return m;
}

ZGL_HD float halfToFloat(uint32_t h)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return (float)__builtin_bit_cast(_Float16, (unsigned short)h);
#else
    const uint32_t sign = (h & 0x8000u) << 16, e = (h >> 10) & 31u, m = h & 0x3ffu;
    if (e == 31u) return bitsf(sign | 0x7f800000u | (m << 13));
    if (e == 0u) return bitsf(sign | fbits((float)m * 5.9604644775390625e-08f));
    return bitsf(sign | ((e + 112u) << 23) | (m << 13));
#endif
}
// FP16 at or below / at or above v, 0 <= v < 65504.
ZGL_HD uint32_t halfDown(double v)
{
    if (!(v > 0.0)) return 0u;
    float f = (float)v;
    if ((double)f > v) f = bitsf(fbits(f) - 1u);
    if (f < 6.103515625e-05f) return (uint32_t)(f * 16777216.0f);
    return (fbits(f) >> 13) - (112u << 10);
}
ZGL_HD uint32_t halfUp(double v)
{
    const uint32_t h = halfDown(v);
    return (double)halfToFloat(h) < v ? h + 1u : h;
}

// Gathers the up to four subtrees that the binary node at row k (table 0) gets as
// children: its two children, then the children of whichever inner one has the largest
// surface, until there are four or only leaves.  Rows are 8 floats
// {pMin.xyz, pMax.xyz, primitive, miss}; k must be an inner row.  Returns how many.
ZGL_HD float wideArea(const float* r)
{
    const float x = r[3] - r[0], y = r[4] - r[1], z = r[5] - r[2];
    return x * y + y * z + z * x;
}
ZGL_HD int wideGather(const float* rows, int k, int out[4])
{
    int n = 2;
    out[0] = k + 1;
    out[1] = fbitsi(rows[(size_t)(k + 1) * 8 + 7]);
    while (n < 4) {
        int best = -1;
        float area = -1.0f;
        for (int i = 0; i < n; i++) {
            const float* r = rows + (size_t)out[i] * 8;
            if (fbitsi(r[6]) >= 0) continue;
            const float a = wideArea(r);
            if (best < 0 || a > area) { best = i; area = a; }
        }
        if (best < 0) break;
        const int open = out[best];
        out[best] = open + 1;
        out[n++] = fbitsi(rows[(size_t)(open + 1) * 8 + 7]);
    }
    return n;
}

// The 16 words of a node whose box is the row `self` and whose children are `rows[out[i]]`,
// the first of them in slot `base`.
ZGL_HD void wideEncode(const float* rows, const float* self, const int out[4], int n, uint32_t base,
                       const WideScale& sc, uint32_t w[16])
{
    const double inv = 1.0 / (double)sc.unit, pad = sc.pad;
    double org[3];
    for (int c = 0; c < 3; c++) {
        const double x = (double)self[c] - pad;
        float f = (float)x;
        // round down (towards the smaller value)
        if ((double)f > x) f = f > 0.0f ? bitsf(fbits(f) - 1u) : (f < 0.0f ? bitsf(fbits(f) + 1u) : -1e-38f);
        w[c] = fbits(f);
        org[c] = f;
    }
    uint32_t leaf = 0, h[6][4];
    for (int i = 0; i < 4; i++)
        for (int c = 0; c < 3; c++) {
            h[c][i] = kHalfInf;
            h[3 + c][i] = kHalfNegInf;
            if (i < n) {
                const float* r = rows + (size_t)out[i] * 8;
                h[c][i] = halfDown(((double)r[c] - pad - org[c]) * inv);
                h[3 + c][i] = halfUp(((double)r[3 + c] + pad - org[c]) * inv);
                if (fbitsi(r[6]) >= 0) leaf |= 1u << i;
            }
        }
    w[3] = base | (leaf << 28);
    for (int g = 0; g < 6; g++) {
        w[4 + 2 * g] = h[g][0] | (h[g][1] << 16);
        w[5 + 2 * g] = h[g][2] | (h[g][3] << 16);
    }
}

namespace f32 {

enum : int {
    kWalkAny = 1,      // any-hit: ends at the first hit
    kWalkRows = 2,     // over the reference's rows
    kWalkPending = 4,  // ended over the wide tree with a result still to be settled
    kWalkNear = 8,     // over the rows: leaves out boxes beyond wideGrowth on a dropped axis
    kWalkWhole = 16,   // drops no subtree: dist stays at its limit, t2 is the closest hit's
    kWalkDoubt = 32,   // kWalkWhole: another hit lies within W's T
};
constexpr int kWalkNone = 0x7fffffff;  // Walk::cur: at no slot, the next stacked one is due
constexpr int kWalkRedo = -2;          // Walk::closest: to be walked over the rows

// One walk, advanced a few nodes at a time.  `cur` is the slot it stands at (the leaf bit
// set at a triangle) or, over the rows, the next row; `leaf` a triangle's slot put by to be
// tested, or -1; `sp` the stack's entries or the table's end; `closest` a triangle's slot
// until wideSettle makes it a primitive.
struct Walk {
    vec3 o, d, inv;
    float dist, t2;
    int cur, leaf, sp, closest, flags;
};

ZGL_HD void walkIdle(Walk& w)
{
    w.o = v3(0.0f); w.d = v3(0.0f); w.inv = v3(0.0f);
    w.dist = 0.0f; w.t2 = 0.0f;
    w.cur = 0; w.leaf = -1; w.sp = 0; w.closest = -1; w.flags = 0;
}

// Whether the ray is far enough from edge-on to every large triangle, h being the smallest
// component of its direction that enters a box test.
ZGL_HD bool wideClear(const WalkMem& m, const Walk& w, float h)
{
    const WideMargins& mg = *m.margins;
    bool clear = true;
    const float k = h - 10.0f * (float)kWideClear * 5.9604644775390625e-08f, one = 1.0f + 2.0f * h;
    for (int i = 0; i < mg.nPlanes; i++) {
        const WidePlane p = mg.planes[i];
        clear = clear && (fabsG((w.d.x * p.x + w.d.y * p.y) + w.d.z * p.z) - p.w) * k >= one;
    }
    return clear;
}

// The reach and the length of direction that the bounds hold for; false for NaN.
ZGL_HD bool wideCovers(const WalkMem& m, const Walk& w, float shortest)
{
    const float one = 1.0f - 1e-6f, reach = 4.0f * m.bound, dd = dot(w.d, w.d);
    return m.wide && fabsG(w.d.x) <= one && fabsG(w.d.y) <= one && fabsG(w.d.z) <= one && dd >= shortest &&
           dd <= 1.02f && fabsG(w.o.x) <= reach && fabsG(w.o.y) <= reach && fabsG(w.o.z) <= reach;
}

// Whether a closest-hit walk of the ray may drop subtrees.
ZGL_HD bool wideDrops(const WalkMem& m, const Walk& w)
{
    return wideClear(m, w, ieeeMin(ieeeMin(fabsG(w.d.x), fabsG(w.d.y)), fabsG(w.d.z)));
}
// Starts (again) over the wide tree, dropping nothing.
ZGL_HD void wideWhole(Walk& w)
{
    w.flags = kWalkWhole;
    w.dist = w.t2 = 1e8f;
    w.cur = 0;
    w.leaf = -1;
    w.sp = 0;
    w.closest = -1;
}

// Starts (again) over the reference's rows.
ZGL_HD void walkRows(const WalkMem& m, Walk& w)
{
    const float eps = 1e-6f;
    const int dropped = (fabsG(w.d.x) < eps ? 1 : 0) + (fabsG(w.d.y) < eps ? 1 : 0) + (fabsG(w.d.z) < eps ? 1 : 0);
    w.flags = (w.flags & kWalkAny) | kWalkRows;
    if (dropped == 1 && wideCovers(m, w, 0.98f) && wideClear(m, w, 0.0625f)) w.flags |= kWalkNear;
    if (!(w.flags & kWalkAny)) w.dist = 1e8f;
    w.cur = cubemapFace(-w.d) * m.bvhSize;
    w.sp = w.cur + m.bvhSize;
    w.closest = -1;
}

// A closest-hit walk (any = false, tmax 1e8) or an any-hit walk up to tmax.  A ray that
// has to take the rows ends at its first step, to be redone.
ZGL_HD void walkStart(const WalkMem& m, Walk& w, vec3 o, vec3 d, bool any, float tmax)
{
    const float eps = 1e-6f;
    w.o = o;
    w.d = d;
    w.dist = tmax;
    w.t2 = tmax;
    w.flags = any ? kWalkAny : 0;
    // an any-hit drops nothing, so its direction may be shorter
    const bool wide = wideCovers(m, w, any ? 0.25f : 0.98f) && fabsG(d.x) >= eps && fabsG(d.y) >= eps && fabsG(d.z) >= eps;
    w.inv = v3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    w.cur = wide ? 0 : kWalkNone;
    w.leaf = -1;
    w.sp = 0;
    w.closest = wide ? -1 : kWalkRedo;
}

// The distance boxes are compared with: a subtree that begins beyond it holds no hit as
// near as W's T.
ZGL_HD float wideLimit(const WalkMem& m, const Walk& w)
{
    return __builtin_fmaf(w.dist, m.rel, m.slack);
}

ZGL_HD uint32_t umin32(uint32_t a, uint32_t b) { return a < b ? a : b; }
ZGL_HD uint32_t umax32(uint32_t a, uint32_t b) { return a < b ? b : a; }

// The slot of the child a key names, with the leaf bit at a triangle.
ZGL_HD int wideChild(uint32_t word, uint32_t key)
{
    const uint32_t i = key & 3u;
    return (int)(((word & kWideSlotMask) + i) | ((word << (3u - i)) & 0x80000000u));
}

// One step from kWalkNone with a subtree stacked: takes it if it begins within the
// distance.
template <class Stack> ZGL_HD void widePop(const WalkMem& m, Walk& w, Stack& st)
{
    w.sp--;
    const WalkEntry e = st.get(w.sp);
    w.cur = bitsf(e.key) <= wideLimit(m, w) ? wideChild(e.word, e.key) : kWalkNone;
}

// The node the walk stands at: tests its four children, goes to the nearest that is hit
// (kWalkNone without one) and stacks the others, farthest first.  A box is entered when
// its padded interval meets [0, limit].  The stack writes are unconditional, each over
// the last unless that one counted, which costs less than branching around them.
template <class Stack> ZGL_HD void wideNode(const WalkMem& m, Walk& w, Stack& st)
{
    const WideSlots n = m.wide + (size_t)(uint32_t)w.cur * 4;
    const WideU4 q0 = n[0], q1 = n[1], q2 = n[2], q3 = n[3];
    const float cx = (bitsf(q0.x) - w.o.x) * w.inv.x, cy = (bitsf(q0.y) - w.o.y) * w.inv.y,
                cz = (bitsf(q0.z) - w.o.z) * w.inv.z;
    const float ix = w.inv.x * m.unit, iy = w.inv.y * m.unit, iz = w.inv.z * m.unit;
    const bool sx = w.inv.x < 0.0f, sy = w.inv.y < 0.0f, sz = w.inv.z < 0.0f;
    // near and far planes of the four children per axis, two FP16 to a word
    const uint32_t nx[2] = {sx ? q2.z : q1.x, sx ? q2.w : q1.y}, fx[2] = {sx ? q1.x : q2.z, sx ? q1.y : q2.w};
    const uint32_t ny[2] = {sy ? q3.x : q1.z, sy ? q3.y : q1.w}, fy[2] = {sy ? q1.z : q3.x, sy ? q1.w : q3.y};
    const uint32_t nz[2] = {sz ? q3.z : q2.x, sz ? q3.w : q2.y}, fz[2] = {sz ? q2.x : q3.z, sz ? q2.y : q3.w};
    const float lim = wideLimit(m, w);
    uint32_t key[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int p = i >> 1, sh = (i & 1) * 16;
        const float ax = __builtin_fmaf(halfToFloat((nx[p] >> sh) & 0xffffu), ix, cx);
        const float ay = __builtin_fmaf(halfToFloat((ny[p] >> sh) & 0xffffu), iy, cy);
        const float az = __builtin_fmaf(halfToFloat((nz[p] >> sh) & 0xffffu), iz, cz);
        const float bx = __builtin_fmaf(halfToFloat((fx[p] >> sh) & 0xffffu), ix, cx);
        const float by = __builtin_fmaf(halfToFloat((fy[p] >> sh) & 0xffffu), iy, cy);
        const float bz = __builtin_fmaf(halfToFloat((fz[p] >> sh) & 0xffffu), iz, cz);
        const float t0 = ieeeMax(ieeeMax(ieeeMax(ax, ay), az), 0.0f);
        const float t1 = ieeeMin(ieeeMin(ieeeMin(bx, by), bz), lim);
        // entry distance (>= 0, so ordered as an integer) with the child in its low bits
        key[i] = t0 <= t1 ? ((fbits(t0) & ~3u) | (uint32_t)i) : 0xffffffffu;
    }
    const uint32_t a0 = umin32(key[0], key[1]), a1 = umax32(key[0], key[1]);
    const uint32_t a2 = umin32(key[2], key[3]), a3 = umax32(key[2], key[3]);
    const uint32_t k0 = umin32(a0, a2), b1 = umax32(a0, a2), b2 = umin32(a1, a3), k3 = umax32(a1, a3);
    const uint32_t k1 = umin32(b1, b2), k2 = umax32(b1, b2);
    if (w.sp > kWalkStack - 3) {  // no room for three more
        w.closest = kWalkRedo;
        w.cur = kWalkNone;
        w.leaf = -1;
        w.sp = 0;
        return;
    }
    st.put(w.sp, WalkEntry{q0.w, k3});
    w.sp += k3 != 0xffffffffu ? 1 : 0;
    st.put(w.sp, WalkEntry{q0.w, k2});
    w.sp += k2 != 0xffffffffu ? 1 : 0;
    st.put(w.sp, WalkEntry{q0.w, k1});
    w.sp += k1 != 0xffffffffu ? 1 : 0;
    w.cur = k0 != 0xffffffffu ? wideChild(q0.w, k0) : kWalkNone;
}

ZGL_HD void wideTri(const WalkMem& m, int slot, vec3& a, vec3& b, vec3& c, int& prim)
{
    const WideSlots n = m.wide + (size_t)(uint32_t)(slot & 0x7fffffff) * 4;
    const WideU4 q0 = n[0], q1 = n[1], q2 = n[2];
    a = v3(bitsf(q0.x), bitsf(q0.y), bitsf(q0.z));
    b = v3(bitsf(q0.w), bitsf(q1.x), bitsf(q1.y));
    c = v3(bitsf(q1.z), bitsf(q1.w), bitsf(q2.x));
    prim = (int)q2.y;
}

// One step over the wide tree: the node the walk stands at, then the next stacked subtree
// if there is nothing to go on with, and a triangle come to is put by while the walk goes
// on to the next subtree, unless one is put by already.
template <class Stack> ZGL_HD void wideStep(const WalkMem& m, Walk& w, Stack& st)
{
    if (w.cur >= 0 && w.cur != kWalkNone) wideNode(m, w, st);
    if (w.cur < 0 && w.leaf < 0) {
        w.leaf = w.cur & 0x7fffffff;
        w.cur = kWalkNone;
    }
    if (w.cur == kWalkNone && w.sp > 0) widePop(m, w, st);
}

// W's T for a hit at t.
ZGL_HD float wideNear(const WalkMem& m, float t)
{
    return __builtin_fmaf(t, 1.0009765625f, m.bound * 1.52587890625e-05f);
}

// Tests the triangle put by; true when it ends the walk (an any-hit).
ZGL_HD bool wideLeaf(const WalkMem& m, Walk& w)
{
    vec3 a, b, c;
    int prim;
    const int slot = w.leaf;
    wideTri(m, slot, a, b, c, prim);
    w.leaf = -1;
    float t;
    if (intersectTriangle(a, b, c, w.o, w.d, t)) {
        const bool whole = (w.flags & kWalkWhole) != 0;
        const float best = whole ? w.t2 : w.dist;
        const bool nearer = t < best;
        w.closest = nearer ? slot : w.closest;
        if (w.flags & kWalkAny) return nearer;
        if (whole) {
            w.t2 = nearer ? t : best;
            const bool doubt = (nearer ? best : t) <= wideNear(m, w.t2);
            w.flags = doubt ? w.flags | kWalkDoubt : nearer ? w.flags & ~kWalkDoubt : w.flags;
        } else {
            w.t2 = nearer ? w.dist : ieeeMin(w.t2, t);
            w.dist = nearer ? t : w.dist;
        }
    }
    return false;
}

// The walk's ray as the reference's box test reads it.
ZGL_HD RayPre walkRay(const Walk& w)
{
    const float eps = 1e-6f, one = 1.0f - eps;
    RayPre p;
    p.o = w.o;
    p.d = w.d;
    p.dInv = w.inv;
    p.mode = (fabsG(w.d.x) > one) ? 1 : (fabsG(w.d.y) > one) ? 2 : (fabsG(w.d.z) > one) ? 3 : 0;
    p.nx = fabsG(w.d.x) < eps;
    p.ny = fabsG(w.d.y) < eps;
    p.nz = fabsG(w.d.z) < eps;
    return p;
}

// The reference's box test on the row k; `general`: boxHitGeneral does.  For a kWalkNear ray
// `grow` is how far beside its triangle a hit can lie on the axis that the test drops: a box
// further than that from the origin holds no hit and counts as missed.  (Infinite: no such
// ray.)
ZGL_HD bool rowHit(const WalkMem& m, const RayPre& p, bool general, float grow, int k, float& boxDist, int& prim,
                   int& miss)
{
    const GRows row = m.rows + (size_t)(uint32_t)k * 2;
    const GFloat4 lo = row[0], hi = row[1];
    const vec3 bMin = v3(lo.x, lo.y, lo.z), bMax = v3(lo.w, hi.x, hi.y);
    prim = fbitsi(hi.z);
    miss = fbitsi(hi.w);
    bool hit = boxHitGeneral(bMin, bMax, p, boxDist);
    if (!general) {
        hit = boxHit(bMin, bMax, p, boxDist);
        if (grow < __builtin_inff()) {
            // nor is any triangle of the box further away than its furthest corner
            const vec3 far = v3(ieeeMax(p.o.x - bMin.x, bMax.x - p.o.x), ieeeMax(p.o.y - bMin.y, bMax.y - p.o.y),
                                ieeeMax(p.o.z - bMin.z, bMax.z - p.o.z));
            const WideMargins& mg = *m.margins;
            const float g = ieeeMin(grow, mg.grow + mg.growRel * (1.001f * length(far) + mg.reach));
            hit = hit && !(p.nx && (bMin.x - g > p.o.x || bMax.x + g < p.o.x));
            hit = hit && !(p.ny && (bMin.y - g > p.o.y || bMax.y + g < p.o.y));
            hit = hit && !(p.nz && (bMin.z - g > p.o.z || bMax.z + g < p.o.z));
        }
    }
    return hit;
}

// How far beside its triangle a hit nearer than the distance can lie on the axis that a
// kWalkNear ray's box test drops.
ZGL_HD float wideGrowth(const WalkMem& m, const Walk& w)
{
    const WideMargins& mg = *m.margins;
    return mg.grow + mg.growRel * (1.4f * (w.dist + mg.reach) + mg.reach);
}

// Rays for which the three-slab box test alone is the reference's (RayPre::special false).
ZGL_HD bool generalRay(const Walk& w)
{
    const float eps = 1e-6f, one = 1.0f - eps;
    const float ax = fabsG(w.d.x), ay = fabsG(w.d.y), az = fabsG(w.d.z), big = 3.4028235e38f;
    return ax >= eps && ay >= eps && az >= eps && ax <= one && ay <= one && az <= one && fabsG(w.o.x) <= big &&
           fabsG(w.o.y) <= big && fabsG(w.o.z) <= big;
}

// Whether the ray passes the reference's box test on every row from the root of its table
// down to the row of the triangle in `slot`.  Tables a caller hands over may be different
// trees, so another table's ancestors would not do.
ZGL_HD bool wideChain(const WalkMem& m, const Walk& w, int slot)
{
    const RayPre p = walkRay(w);
    const int table = cubemapFace(-w.d);
    const WideSlots n = m.wide + (size_t)(uint32_t)slot * 4;
    const WideU4 q2 = n[2], q3 = n[3];
    const int row = (int)(table == 0 ? q2.z : table == 1 ? q2.w : table == 2 ? q3.x : table == 3 ? q3.y
                          : table == 4 ? q3.z : q3.w);
    int k = table * m.bvhSize;
    for (;;) {
        float dist;
        int prim, miss;
        if (!rowHit(m, p, true, 0.0f, k, dist, prim, miss)) return false;
        if (k == row) return true;
        const GFloat4 first = m.rows[(size_t)(uint32_t)(k + 1) * 2 + 1];
        k = row < fbitsi(first.w) ? k + 1 : fbitsi(first.w);
    }
}

// Whether the reference's walk finds the triangle this one found (see the top of the
// file), or how the walk has to be repeated.  `closest` becomes the primitive before the
// ancestors are asked: set after that loop, ROCm 7.2's compiler left the slot in it for the lanes that had
// been through the loop.
enum : int { kSettled, kSettleWhole, kSettleRows };
template <bool CHAIN> ZGL_HD int wideSettle(const WalkMem& m, Walk& w)
{
    if (w.closest < 0) return kSettleRows;
    if (!(w.flags & (kWalkAny | kWalkWhole)) && !wideDrops(m, w)) return kSettleWhole;
    if (w.flags & kWalkWhole) {
        w.dist = w.t2;
        w.t2 = w.flags & kWalkDoubt ? w.dist : 1e8f;
    }
    vec3 a, b, c;
    int prim;
    const int slot = w.closest;
    wideTri(m, slot, a, b, c, prim);
    w.closest = prim;
    const vec3 lo = v3(ieeeMin(ieeeMin(a.x, b.x), c.x), ieeeMin(ieeeMin(a.y, b.y), c.y), ieeeMin(ieeeMin(a.z, b.z), c.z));
    const vec3 hi = v3(ieeeMax(ieeeMax(a.x, b.x), c.x), ieeeMax(ieeeMax(a.y, b.y), c.y), ieeeMax(ieeeMax(a.z, b.z), c.z));
    const vec3 ta = (lo - w.o) * w.inv, tb = (hi - w.o) * w.inv;
    const vec3 mn = v3(ieeeMin(ta.x, tb.x), ieeeMin(ta.y, tb.y), ieeeMin(ta.z, tb.z));
    const vec3 mx = v3(ieeeMax(ta.x, tb.x), ieeeMax(ta.y, tb.y), ieeeMax(ta.z, tb.z));
    // 8 u T per axis
    const float u8 = 4.76837158203125e-07f;
    const float nx = (m.bound + fabsG(w.o.x)) * fabsG(w.inv.x) * u8;
    const float ny = (m.bound + fabsG(w.o.y)) * fabsG(w.inv.y) * u8;
    const float nz = (m.bound + fabsG(w.o.z)) * fabsG(w.inv.z) * u8;
    const bool pairs = mx.y - mn.z > ny + nz && mx.z - mn.x > nz + nx && mx.x - mn.y > nx + ny;
    const float l = ieeeMax(ieeeMax(mn.x, mn.y), mn.z), h = ieeeMin(ieeeMin(mx.x, mx.y), mx.z);
    const bool order = (w.flags & kWalkAny) || (w.t2 > w.dist && l <= wideNear(m, w.dist));
    if (!(h >= 0.0f && h >= l && l <= w.t2 && order)) return kSettleRows;
    // too near an edge of its box for the margins: asked of the ancestors themselves
    if constexpr (CHAIN) return pairs || wideChain(m, w, slot) ? kSettled : kSettleRows;
    return pairs ? kSettled : kSettleRows;
}

// Up to four of the reference's rows and the triangle of a leaf met on the way, with the
// reference's tests in its order; true when the walk has ended.  `general`: no lane
// stepping with this one has a ray for which boxHitGeneral would not do.  Adds what it
// visited to `rows` and `tests`.
ZGL_HD bool rowsStep(const WalkMem& m, Walk& w, bool general, uint32_t& rows, uint32_t& tests)
{
    const RayPre p = walkRay(w);
    const float grow = w.flags & kWalkNear ? wideGrowth(m, w) : __builtin_inff();
    int leaf = -1;
#pragma nounroll
    for (int u = 0; u < 4; u++) {
        if (w.cur != w.sp && leaf < 0) {
            rows++;
            float boxDist;
            int prim, miss;
            const bool hit = rowHit(m, p, general, grow, w.cur, boxDist, prim, miss);
            const bool take = hit && !(boxDist > w.dist);
            leaf = take && prim >= 0 ? prim : leaf;
            w.cur = take ? (prim >= 0 ? w.cur : w.cur + 1) : miss;
        }
    }
    if (leaf >= 0) {
        const GRows tri = m.tris + (size_t)leaf * 3;
        const GFloat4 t0 = tri[0], t1 = tri[1], t2 = tri[2];
        tests++;
        float t;
        if (intersectTriangle(v3(t0.x, t0.y, t0.z), v3(t0.w, t1.x, t1.y), v3(t1.z, t1.w, t2.x), w.o, w.d, t) &&
            t < w.dist) {
            w.closest = leaf;
            if (w.flags & kWalkAny) return true;
            w.dist = t;
        }
        w.cur++;
    }
    return w.cur == w.sp;
}

}  // namespace f32
}  // namespace zgl
