// Host build of the product's walk over the 4-wide tree (zillumgl_amd/csrc/zgl_wide.h), for
// comparison with the oracle's walk over the reference's rows.  probe_wide_build collapses
// an MTBVH as the device builder does (the slots in breadth-first order) and returns the
// slot count, or 0 where the scene has no wide tree; probe_wide_trace walks rays and
// repeats over the rows those the wide walk cannot vouch for, as the kernels do.
#include <algorithm>
#include <cstdint>
#include <cstring>
#include <vector>

#include "../../zillumgl_amd/csrc/zgl_wide.h"

using namespace zgl;

namespace {
struct HostStack {
    WalkEntry e[kWalkStack];
    WalkEntry get(int i) const { return e[i]; }
    void put(int i, WalkEntry x) { e[i] = x; }
};
struct Tree {
    std::vector<float> rows, tris;
    std::vector<uint32_t> slots;
    WideScale scale;
    WideMargins margins;
    int bvhSize;
};
Tree g;

// k_wide_tris' sums, one triangle after the other
void collect(WideStats& st, const WideTriClass& c)
{
    if (c.kind == kWideTriSmall) {
        st.x = std::max(st.x, fbits(c.x));
        st.diagonal = std::max(st.diagonal, fbits(c.diagonal));
    }
    if (c.kind != kWideTriLarge) return;
    st.edge = std::max(st.edge, fbits(c.edge));
    int i = 0;
    while (i < kWidePlaneSlots && st.key[i] != 0 && st.key[i] != c.key) i++;
    if (c.key == 0 || i == kWidePlaneSlots) {
        st.overflow = 1;
        return;
    }
    st.sine[i] = st.key[i] == 0 ? fbits(c.sine) : std::min(st.sine[i], fbits(c.sine));
    st.key[i] = c.key;
}
}  // namespace

extern "C" int64_t probe_wide_build(const float* vertices, const int32_t* indices, int64_t nTri, const float* bounds,
                                    const int32_t* hit)
{
    const int B = (int)(2 * nTri - 1);
    g.bvhSize = B;
    g.rows.assign((size_t)6 * B * 8, 0.0f);
    for (int t = 0; t < 6; t++)
        for (int k = 0; k < B; k++) {
            const int32_t* r = hit + ((size_t)t * B + k) * 3;
            float* o = g.rows.data() + ((size_t)t * B + k) * 8;
            std::memcpy(o, bounds + (size_t)r[0] * 6, 24);
            const int32_t miss = t * B + r[2];
            std::memcpy(o + 6, &r[1], 4);
            std::memcpy(o + 7, &miss, 4);
        }
    g.tris.assign((size_t)nTri * 12, 0.0f);
    for (int64_t i = 0; i < nTri; i++)
        for (int v = 0; v < 3; v++)
            for (int c = 0; c < 3; c++) g.tris[i * 12 + v * 3 + c] = vertices[(size_t)indices[3 * i + v] * 3 + c];
    g.slots.clear();
    const float* root = g.rows.data();
    g.scale = wideScale(root, root + 3);
    if (!g.scale.ok) return 0;
    std::vector<int> rowOf((size_t)6 * nTri, -1);
    for (int k = 0; k < 6 * B; k++) {
        const int prim = fbitsi(root[(size_t)k * 8 + 6]);
        if (prim >= 0) rowOf[(size_t)prim * 6 + k / B] = k;
    }
    WideStats st{};
    for (int64_t i = 0; i < nTri; i++) collect(st, wideClassify(&g.tris[i * 12], g.scale.bound));
    g.margins = wideMargins(st, g.scale);
    std::vector<int> row(1, 0);  // row of every slot
    g.slots.assign(16, 0u);
    for (size_t s = 0; s < row.size(); s++) {
        const float* self = root + (size_t)row[s] * 8;
        const int prim = fbitsi(self[6]);
        if (prim >= 0 && s > 0) {
            std::memcpy(&g.slots[s * 16], &g.tris[(size_t)prim * 12], 36);
            g.slots[s * 16 + 9] = (uint32_t)prim;
            std::memcpy(&g.slots[s * 16 + 10], &rowOf[(size_t)prim * 6], 24);
            continue;
        }
        int out[4] = {row[s], 0, 0, 0};
        const int n = prim >= 0 ? 1 : wideGather(root, row[s], out);
        const uint32_t base = (uint32_t)row.size();
        for (int i = 0; i < n; i++) row.push_back(out[i]);
        g.slots.resize(row.size() * 16, 0u);
        wideEncode(root, self, out, n, base, g.scale, &g.slots[s * 16]);
    }
    return (int64_t)row.size();
}

// rowsOnly: every ray over the rows.  stats: [0] walks over the wide tree, [1] of them repeated over the rows, [2] nodes,
// [3] triangles, [4] largest stack, [5] rays that took the rows from the start, [6] walks that
// ran out of stack, [7] rows, [8] walks made again that drop nothing
extern "C" void probe_wide_trace(const float* rays, int64_t n, const float* tmax, int any, int rowsOnly,
                                 int32_t* prim, float* t, int64_t* stats)
{
    WalkMem m;
    m.rows = (GRows)g.rows.data();
    m.tris = (GRows)g.tris.data();
    m.wide = g.slots.empty() || rowsOnly ? nullptr : (WideSlots)g.slots.data();
    m.bvhSize = g.bvhSize;
    m.unit = g.scale.unit;
    m.bound = g.scale.bound;
    m.rel = g.margins.rel;
    m.slack = g.margins.slack;
    m.margins = &g.margins;
    for (int64_t i = 0; i < n; i++) {
        f32::Walk w;
        f32::walkStart(m, w, v3(rays[i], rays[n + i], rays[2 * n + i]), v3(rays[3 * n + i], rays[4 * n + i], rays[5 * n + i]),
                       any != 0, any ? tmax[i] : 1e8f);
        HostStack st;
        stats[w.closest == f32::kWalkRedo ? 5 : 0]++;
        if (w.closest == f32::kWalkRedo) f32::walkRows(m, w);
        while (!(w.flags & f32::kWalkRows)) {
            bool done = false;
            while (!done) {
                if (w.cur >= 0 && w.cur != f32::kWalkNone) stats[2]++;
                f32::wideStep(m, w, st);
                if (w.sp > stats[4]) stats[4] = w.sp;
                if (w.closest == f32::kWalkRedo) stats[6]++;
                if (w.leaf >= 0) { stats[3]++; done = f32::wideLeaf(m, w); }
                done = done || (w.cur == f32::kWalkNone && w.sp == 0);
            }
            const int how = w.closest == -1 ? f32::kSettled : f32::wideSettle<true>(m, w);
            if (how == f32::kSettled) break;
            stats[how == f32::kSettleWhole ? 8 : 1]++;
            if (how == f32::kSettleWhole) f32::wideWhole(w);
            else f32::walkRows(m, w);
        }
        uint32_t rows = 0, tests = 0;
        if (w.flags & f32::kWalkRows)
            while (!f32::rowsStep(m, w, f32::generalRay(w), rows, tests)) {}
        stats[7] += rows;
        prim[i] = w.closest;
        t[i] = w.dist;
    }
}

// The margins of the built tree.
extern "C" void probe_wide_margins(float out[6])
{
    const float v[6] = {g.margins.rel,     g.margins.slack, g.margins.grow,
                        g.margins.growRel, g.margins.reach, (float)g.margins.nPlanes};
    std::memcpy(out, v, sizeof(v));
}
