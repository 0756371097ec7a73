// zgl_wide.h -- closest-hit and any-hit walks over a 4-wide tree, with results equal to
// the reference's MTBVH walk (intersection.glsl:367-427) bit for bit; host and device.
//
// What bounds the reference's walk is its rows: on the 819,400-triangle scene a ray visits
// 47 of them, each a dependent 32-byte load and an exact box test of about 45 vector
// instructions.  Only two things of that walk reach its result: which triangles' own
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
//     contain the exact ones, with room for the rounding of both sides), so it tests
//     every triangle the reference may test, and more.
//   * Let W be its closest hit at t, t2 the next larger hit distance it met (the ray's
//     limit if none), b the entry distance of W's exact box.  If W's box passes with those
//     margins, t < t2 and b <= t2, then whenever the reference's walk comes to W its
//     distance is still at least t2: W is tested, and nothing is nearer.  So the
//     reference's closest hit is W whatever order it visits the leaves in.  Where only the
//     margins fail (about one hit in a thousand), the reference's box test can be made on
//     W's ancestors themselves (CHAIN), a fifth of a walk over the rows.
//   * Without a hit the reference has none either.  For an any-hit ray one hit that passes
//     with these margins and b <= the limit shows that it is occluded.
// Measured: 47 rows become 13 nodes and 3 triangles a ray on the headline scene; the
// 64-pass 1080p launch went from 169 to 114 ms, one 720p pass of a 205,000-triangle scene
// from 15.7 to 2.0 ms (see the last paragraph), ten batched scenes from 28.8 to 22.2 ms.
// A node step is about 110 vector instructions for four boxes (fma_mix reads the FP16
// planes in place) against 45 for one row.
//
// Rays the argument does not cover take the reference's rows from the start: nearly
// axis-parallel ones (RayPre::mode != 0), two components below 1e-6, not finite, from far
// outside the scene, or with a direction shorter than 0.5.  A ray with one component
// below 1e-6, whose box test drops that axis' slab, is covered with the remaining pair's
// margin; the reference's walk of such a ray visits every box of a slice through the scene
// (15 ms for one ray on a 205,000-triangle scene), the walk here a ray's worth.
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

// The scene as a walk sees it.
struct WalkMem {
    GRows rows;        // the reference's row tables
    GRows tris;        // 48 bytes per triangle
    WideSlots wide;    // null: every ray takes the rows
    int bvhSize;
    float unit;        // world length of one FP16 unit of the planes (a power of two)
    float slack;       // added to the distance when a box is compared with it
    float bound;       // largest absolute coordinate of the scene's box
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

// Starts (again) over the reference's rows.
ZGL_HD void walkRows(const WalkMem& m, Walk& w)
{
    w.inv = v3(1.0f / w.d.x, 1.0f / w.d.y, 1.0f / w.d.z);
    w.flags = (w.flags & kWalkAny) | kWalkRows;
    if (!(w.flags & kWalkAny)) w.dist = 1e8f;
    w.cur = cubemapFace(-w.d) * m.bvhSize;
    w.sp = w.cur + m.bvhSize;
    w.closest = -1;
}

// A closest-hit walk (any = false, tmax 1e8) or an any-hit walk up to tmax.  A ray that
// has to take the rows ends at its first step, to be redone.
ZGL_HD void walkStart(const WalkMem& m, Walk& w, vec3 o, vec3 d, bool any, float tmax)
{
    const float eps = 1e-6f, one = 1.0f - eps;
    w.o = o;
    w.d = d;
    w.dist = tmax;
    w.t2 = tmax;
    w.flags = any ? kWalkAny : 0;
    const float ax = fabsG(d.x), ay = fabsG(d.y), az = fabsG(d.z);
    const bool tx = ax < eps, ty = ay < eps, tz = az < eps;
    const float reach = 4.0f * m.bound;
    // NaN fails the comparisons on o and on d.d
    const bool wide = m.wide && ax <= one && ay <= one && az <= one && (ax * ax + ay * ay) + az * az >= 0.25f &&
                      !((tx && ty) || (ty && tz) || (tx && tz)) && fabsG(o.x) <= reach && fabsG(o.y) <= reach &&
                      fabsG(o.z) <= reach;
    // a dropped axis (below 1e-6) keeps a finite reciprocal: its slab is tested here, and
    // over the scene a component below 1e-15 moves the ray by less than the pad
    const float tiny = 1e-15f;
    w.inv = v3(1.0f / (ax < tiny ? __builtin_copysignf(tiny, d.x) : d.x),
               1.0f / (ay < tiny ? __builtin_copysignf(tiny, d.y) : d.y),
               1.0f / (az < tiny ? __builtin_copysignf(tiny, d.z) : d.z));
    w.cur = wide ? 0 : kWalkNone;
    w.leaf = -1;
    w.sp = 0;
    w.closest = wide ? -1 : kWalkRedo;
}

ZGL_HD uint32_t umin32(uint32_t a, uint32_t b) { return a < b ? a : b; }
ZGL_HD uint32_t umax32(uint32_t a, uint32_t b) { return a < b ? b : a; }

// The distance boxes are compared with: dist widened by 2^-10 and the slack, so that a
// triangle slightly nearer than its box's computed entry is still tested.
ZGL_HD float wideLimit(const WalkMem& m, const Walk& w) { return __builtin_fmaf(w.dist, 1.0009765625f, m.slack); }

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
        const bool nearer = t < w.dist;
        w.closest = nearer ? slot : w.closest;
        if (w.flags & kWalkAny) return nearer;
        w.t2 = nearer ? w.dist : ieeeMin(w.t2, t);
        w.dist = nearer ? t : w.dist;
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

// The reference's box test on the row k.
ZGL_HD bool rowHit(const WalkMem& m, const RayPre& p, bool general, int k, float& boxDist, int& prim, int& miss)
{
    const GRows row = m.rows + (size_t)(uint32_t)k * 2;
    const GFloat4 lo = row[0], hi = row[1];
    const vec3 bMin = v3(lo.x, lo.y, lo.z), bMax = v3(lo.w, hi.x, hi.y);
    prim = fbitsi(hi.z);
    miss = fbitsi(hi.w);
    bool hit = boxHitGeneral(bMin, bMax, p, boxDist);
    if (!general) hit = boxHit(bMin, bMax, p, boxDist);
    return hit;
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
    const bool general = generalRay(w);
    const int table = cubemapFace(-w.d);
    const WideSlots n = m.wide + (size_t)(uint32_t)slot * 4;
    const WideU4 q2 = n[2], q3 = n[3];
    const int row = (int)(table == 0 ? q2.z : table == 1 ? q2.w : table == 2 ? q3.x : table == 3 ? q3.y
                          : table == 4 ? q3.z : q3.w);
    int k = table * m.bvhSize;
    for (;;) {
        float dist;
        int prim, miss;
        if (!rowHit(m, p, general, k, dist, prim, miss)) return false;
        if (k == row) return true;
        const GFloat4 first = m.rows[(size_t)(uint32_t)(k + 1) * 2 + 1];
        k = row < fbitsi(first.w) ? k + 1 : fbitsi(first.w);
    }
}

// Whether the reference's walk finds the triangle this one found (see the top of the
// file); false where the walk has to be repeated over the rows.  `closest` becomes the
// primitive either way, before the ancestors are asked: set after that loop, ROCm 7.2's
// compiler left the slot in it for the lanes that had been through the loop.
template <bool CHAIN> ZGL_HD bool wideSettle(const WalkMem& m, Walk& w)
{
    if (w.closest < 0) return false;
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
    const float u8 = 4.76837158203125e-07f, eps = 1e-6f;
    const float nx = (m.bound + fabsG(w.o.x)) * fabsG(w.inv.x) * u8;
    const float ny = (m.bound + fabsG(w.o.y)) * fabsG(w.inv.y) * u8;
    const float nz = (m.bound + fabsG(w.o.z)) * fabsG(w.inv.z) * u8;
    const bool cx = mx.y - mn.z > ny + nz, cy = mx.z - mn.x > nz + nx, cz = mx.x - mn.y > nx + ny;
    const bool tx = fabsG(w.d.x) < eps, ty = fabsG(w.d.y) < eps, tz = fabsG(w.d.z) < eps;
    // an axis below 1e-6 drops out of the slabs and leaves one pair
    const float ninf = -__builtin_inff(), pinf = __builtin_inff();
    const float l = ieeeMax(ieeeMax(tx ? ninf : mn.x, ty ? ninf : mn.y), tz ? ninf : mn.z);
    const float h = ieeeMin(ieeeMin(tx ? pinf : mx.x, ty ? pinf : mx.y), tz ? pinf : mx.z);
    const bool pairs = tx ? cx : ty ? cy : tz ? cz : (cx && cy && cz);
    const bool order = (w.flags & kWalkAny) || w.t2 > w.dist;
    if (!(h >= 0.0f && h >= l && l <= w.t2 && order)) return false;
    // too near an edge of its box for the margins: asked of the ancestors themselves
    if constexpr (CHAIN) return pairs || wideChain(m, w, slot);
    return pairs;
}

// Up to four of the reference's rows and the triangle of a leaf met on the way, with the
// reference's tests in its order; true when the walk has ended.  `general`: no lane
// stepping with this one has a ray for which boxHitGeneral would not do.  Adds what it
// visited to `rows` and `tests`.
ZGL_HD bool rowsStep(const WalkMem& m, Walk& w, bool general, uint32_t& rows, uint32_t& tests)
{
    const RayPre p = walkRay(w);
    int leaf = -1;
#pragma nounroll
    for (int u = 0; u < 4; u++) {
        if (w.cur != w.sp && leaf < 0) {
            rows++;
            float boxDist;
            int prim, miss;
            const bool hit = rowHit(m, p, general, w.cur, boxDist, prim, miss);
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
