// zgl_wide.hip -- builds a scene's 4-wide tree (zgl_wide.h) on the device from its MTBVH
// rows and triangles.
//
// The walk over the wide tree equals the walk over the rows only if each of the six tables
// threads a binary tree over the same leaves: every inner row's box contains its children's
// and lies in table 0's root box, every leaf's box is its triangle's, and every triangle is
// a leaf of every table.  k_wide_check and k_wide_tris show that (rows handed over by a
// caller may say anything that points forward); a scene that fails it keeps no wide tree
// and all its rays take the rows.  The six trees need not be the same one: the wide tree
// is table 0's, and a hit's ancestors are asked in the ray's own table.
//
// The tree is built breadth first, a level a launch: a work item is a binary inner row and
// the slot of its node; its thread gathers the node's up to four children, reserves
// consecutive slots for them (one atomic per wave), writes the node and its triangles and
// queues its inner children.  The slots' order within a level depends on the atomics, the
// walks' results do not.  The host looks at the queue every kLevelsPerLook levels.
#include "zgl_internal.h"
#include "zgl_wide.h"

#include <algorithm>

namespace zgl {

namespace {

// Scenes of 10,000 to 1.3M triangles have 10 to 14 levels; looks every 12, 14 or 16 make no
// difference to an upload (within 1%).
constexpr int kLevelsPerLook = 14;
constexpr int kMaxLevels = 96;  // deeper trees (one triangle split off per level) keep the rows
// Triangles one workgroup builds for by itself.  An upload by one workgroup / by levels takes
// 310 / 363 us for 36 triangles, 547 / 578 for 138, 902 / 868 for 546, 1,158 / 994 for 1,226
// and 1,448 / 1,085 for 2,178.
constexpr int kSmallBuild = 256;

struct WideCounters {
    float root[8];               // the root's row
    int bad;                     // rows that fail the check
    int slots;                   // slots reserved
    int count[kMaxLevels + 1];   // items of each level
    WideStats stats;
};
struct WideBuild {
    const float* rows;  // 6 tables of S rows
    const float* tris;
    int n, S, capacity;
    uint4* slots;
    int2* queue[2];     // items of the even and the odd levels: a row and its node's slot
    int* rowOf;         // six per triangle: its row in each table, -1 where it was not met
    WideCounters* c;
};

// The parts below run over `threads` threads, this one the `tid`-th.
__device__ __forceinline__ void wideInit(const WideBuild& b, int tid, int threads)
{
    for (int64_t g = tid; g < (int64_t)6 * b.n; g += threads) b.rowOf[g] = -1;
    for (int g = tid; g <= kMaxLevels; g += threads) b.c->count[g] = g == 0 ? 1 : 0;
    for (int g = tid; g < kWidePlaneSlots; g += threads) {
        b.c->stats.key[g] = 0;
        b.c->stats.sine[g] = 0x7f7fffffu;
    }
    if (tid < 8) b.c->root[tid] = b.rows[tid];
    if (tid == 0) {
        b.c->bad = 0;
        b.c->slots = 1;
        b.c->stats.x = b.c->stats.diagonal = b.c->stats.edge = b.c->stats.overflow = 0;
        b.queue[0][0] = make_int2(0, 0);  // the root's row and slot
    }
}

__device__ __forceinline__ bool contains(const float* a, const float* b)
{
    return a[0] <= b[0] && a[1] <= b[1] && a[2] <= b[2] && a[3] >= b[3] && a[4] >= b[4] && a[5] >= b[5];
}

__device__ __forceinline__ void wideCheck(const WideBuild& b, int tid, int threads)
{
    int bad = 0;
    for (int64_t g = tid; g < (int64_t)6 * b.S; g += threads) {
        const int t = (int)(g / b.S);
        const int k = (int)g, end = (t + 1) * b.S;  // 6 S fits int32
        const float* r = b.rows + (size_t)k * 8;
        const int prim = __float_as_int(r[6]), miss = __float_as_int(r[7]);
        bool ok = (k != t * b.S || miss == end) && contains(b.rows, r);
        if (prim >= 0) {
            ok = ok && prim < b.n && miss == k + 1;
            if (ok) {
                const float* p = b.tris + (size_t)prim * 12;
                for (int a = 0; a < 3; a++) {
                    const float lo = fminf(fminf(p[a], p[3 + a]), p[6 + a]), hi = fmaxf(fmaxf(p[a], p[3 + a]), p[6 + a]);
                    ok = ok && r[a] == lo && r[3 + a] == hi;
                }
                b.rowOf[(size_t)prim * 6 + t] = k;
            }
        } else {
            const int c1 = k + 1;
            ok = ok && c1 < end;
            if (ok) {
                const float* r1 = b.rows + (size_t)c1 * 8;
                const int c2 = __float_as_int(r1[7]);
                ok = c2 > c1 && c2 < end && c2 < miss;
                if (ok) {
                    const float* r2 = b.rows + (size_t)c2 * 8;
                    ok = __float_as_int(r2[7]) == miss && contains(r, r1) && contains(r, r2);
                }
            }
        }
        if (!ok) bad++;
    }
    if (bad) atomicAdd(&b.c->bad, bad);
}

__device__ __forceinline__ uint32_t loadStat(const uint32_t* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The wave's largest value into *p, all 64 lanes together.
__device__ __forceinline__ void waveMax(uint32_t* p, uint32_t v)
{
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o));
    if ((threadIdx.x & 63) == 0 && v > loadStat(p)) atomicMax(p, v);
}
// A large triangle's plane: its slot in the open-addressed table, claimed where it is new.
__device__ __forceinline__ void notePlane(WideStats* st, uint32_t key, uint32_t sine)
{
    if (key != 0) {
        const uint32_t home = (key * 2654435761u) >> 26;
        for (int i = 0; i < kWidePlaneSlots; i++) {
            const uint32_t at = (home + i) % kWidePlaneSlots;
            uint32_t have = loadStat(&st->key[at]);
            if (have == 0) {
                have = atomicCAS(&st->key[at], 0u, key);
                have = have == 0 ? key : have;
            }
            if (have == key) {
                if (sine < loadStat(&st->sine[at])) atomicMin(&st->sine[at], sine);
                return;
            }
        }
    }
    if (loadStat(&st->overflow) == 0) atomicMax(&st->overflow, 1u);
}

// Every triangle is a leaf of every table (which has n leaves, so it holds each of them
// once), and what it is to the error bound of zgl_wide.h.
__device__ __forceinline__ void wideTris(const WideBuild& b, int tid, int threads)
{
    const WideScale sc = wideScale(b.rows, b.rows + 3);
    int bad = 0;
    uint32_t x = 0, diagonal = 0, edge = 0;
    for (int64_t g = tid; g < b.n; g += threads) {
        for (int t = 0; t < 6; t++)
            if (b.rowOf[g * 6 + t] < 0) bad++;
        const WideTriClass c = wideClassify(b.tris + g * 12, sc.bound);
        if (c.kind == kWideTriBad) bad++;
        if (c.kind == kWideTriSmall) {
            x = max(x, fbits(c.x));
            diagonal = max(diagonal, fbits(c.diagonal));
        }
        if (c.kind == kWideTriLarge) {
            edge = max(edge, fbits(c.edge));
            notePlane(&b.c->stats, c.key, fbits(c.sine));
        }
    }
    waveMax(&b.c->stats.x, x);
    waveMax(&b.c->stats.diagonal, diagonal);
    waveMax(&b.c->stats.edge, edge);
    if (bad) atomicAdd(&b.c->bad, bad);
}

// Exclusive prefix over the wave of a count in 0..4, and the wave's total.
__device__ __forceinline__ int wavePrefix(int v, int& total)
{
    const unsigned long long below = (1ull << (threadIdx.x & 63)) - 1ull;
    int pre = 0;
    total = 0;
#pragma unroll
    for (int b = 0; b < 3; b++) {
        const unsigned long long m = __ballot((v >> b) & 1);
        pre += __popcll(m & below) << b;
        total += __popcll(m) << b;
    }
    return pre;
}
__device__ __forceinline__ int waveReserve(int* counter, int v)
{
    int total;
    const int pre = wavePrefix(v, total);
    int base = 0;
    if ((threadIdx.x & 63) == 0 && total > 0) base = atomicAdd(counter, total);
    return __shfl(base, 0) + pre;
}

// A level's items, by workgroups of which this is the `group`-th of `groups`; whole waves
// stay in the loop for the reservations.
__device__ __forceinline__ void wideLevel(const WideBuild& b, int level, int items, int group, int groups)
{
    const WideScale sc = wideScale(b.rows, b.rows + 3);
    if (!sc.ok) return;
    const int2* in = b.queue[level & 1];
    int2* out = b.queue[(level + 1) & 1];
    for (int base = group * (int)blockDim.x; base < items; base += groups * (int)blockDim.x) {
        const int i = base + (int)threadIdx.x;
        const bool have = i < items;
        int2 item = make_int2(0, 0);
        int child[4] = {0, 0, 0, 0};
        int m = 0, inner = 0;
        if (have) {
            item = in[i];
            if (__float_as_int(b.rows[(size_t)item.x * 8 + 6]) >= 0) {  // a scene of one triangle
                child[0] = item.x;
                m = 1;
            } else {
                m = wideGather(b.rows, item.x, child);
            }
            for (int j = 0; j < 4; j++)
                if (j < m && __float_as_int(b.rows[(size_t)child[j] * 8 + 6]) < 0) inner++;
        }
        const int first = waveReserve(&b.c->slots, m);
        int q = waveReserve(&b.c->count[level + 1], inner);
        if (have && first + m <= b.capacity) {
            uint32_t w[16];
            wideEncode(b.rows, b.rows + (size_t)item.x * 8, child, m, (uint32_t)first, sc, w);
            uint4* o = b.slots + (size_t)item.y * 4;
            for (int j = 0; j < 4; j++) o[j] = make_uint4(w[4 * j], w[4 * j + 1], w[4 * j + 2], w[4 * j + 3]);
            for (int j = 0; j < 4; j++) {
                if (j >= m) break;
                const int prim = __float_as_int(b.rows[(size_t)child[j] * 8 + 6]);
                if (prim < 0) {
                    if (q < b.n) out[q] = make_int2(child[j], first + j);
                    q++;
                } else {
                    const float4* p = reinterpret_cast<const float4*>(b.tris + (size_t)prim * 12);
                    float4* d = reinterpret_cast<float4*>(b.slots + (size_t)(first + j) * 4);
                    const float4 p0 = p[0], p1 = p[1], p2 = p[2];
                    d[0] = p0;
                    d[1] = p1;
                    const int* k = b.rowOf + (size_t)prim * 6;
                    d[2] = make_float4(p2.x, __int_as_float(prim), __int_as_float(k[0]), __int_as_float(k[1]));
                    d[3] = make_float4(__int_as_float(k[2]), __int_as_float(k[3]), __int_as_float(k[4]),
                                       __int_as_float(k[5]));
                }
            }
        }
    }
}

__global__ __launch_bounds__(256) void k_wide_init(WideBuild b)
{
    wideInit(b, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}
__global__ __launch_bounds__(256) void k_wide_check(WideBuild b)
{
    wideCheck(b, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}
__global__ __launch_bounds__(256) void k_wide_tris(WideBuild b)
{
    wideTris(b, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}
__global__ __launch_bounds__(256) void k_wide_level(WideBuild b, int level)
{
    if (b.c->bad) return;
    wideLevel(b, level, b.c->count[level], blockIdx.x, gridDim.x);
}

// Everything by one workgroup, for scenes whose build is launches more than work.
__global__ __launch_bounds__(256) void k_wide_small(WideBuild b)
{
    wideInit(b, threadIdx.x, blockDim.x);
    __syncthreads();
    wideCheck(b, threadIdx.x, blockDim.x);
    __syncthreads();
    wideTris(b, threadIdx.x, blockDim.x);
    __syncthreads();
    if (__hip_atomic_load(&b.c->bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
    for (int level = 0; level < kMaxLevels; level++) {
        const int items = __hip_atomic_load(&b.c->count[level], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (items == 0) break;
        wideLevel(b, level, items, 0, 1);
        __threadfence();
        __syncthreads();
    }
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace

// A node with fewer than four children has only triangles, so at most n / 2 nodes sit
// above triangles alone and a third of that above those: n + 2 n / 3 slots.
int64_t wideCapacity(int64_t n) { return n + (2 * n) / 3 + 16; }

size_t wideWorkBytes(int64_t n) { return align256(sizeof(WideCounters)) + 2 * align256((size_t)n * 8 + 8) + (size_t)n * 24; }

hipError_t buildWide(const float4* rows, const float4* tris, int64_t nTri, void* work, uint4* slots, hipStream_t st,
                     WideScale& scale, WideMargins& margins)
{
    scale = WideScale{0.0f, 0.0f, 1.0f, false};
    margins = WideMargins{};
    const int n = (int)nTri, S = 2 * n - 1;
    const int64_t capacity = wideCapacity(nTri);
    if (capacity > (int64_t)kWideSlotMask) return hipSuccess;
    char* p = static_cast<char*>(work);
    WideBuild b;
    b.rows = reinterpret_cast<const float*>(rows);
    b.tris = reinterpret_cast<const float*>(tris);
    b.n = n;
    b.S = S;
    b.capacity = (int)capacity;
    b.slots = slots;
    b.c = reinterpret_cast<WideCounters*>(p);
    p += align256(sizeof(WideCounters));
    for (int i = 0; i < 2; i++) {
        b.queue[i] = reinterpret_cast<int2*>(p);
        p += align256((size_t)n * 8 + 8);
    }
    b.rowOf = reinterpret_cast<int*>(p);
    const bool small = n <= kSmallBuild;
    if (small) {
        hipLaunchKernelGGL(k_wide_small, dim3(1), dim3(256), 0, st, b);
    } else {
        const unsigned perTri = (unsigned)((n + 255) / 256);
        hipLaunchKernelGGL(k_wide_init, dim3(perTri), dim3(256), 0, st, b);
        hipLaunchKernelGGL(k_wide_check, dim3((unsigned)std::min<int64_t>(8192, ((int64_t)6 * S + 255) / 256)), dim3(256),
                           0, st, b);
        hipLaunchKernelGGL(k_wide_tris, dim3(perTri), dim3(256), 0, st, b);
    }
    WideCounters host;
    for (int level = 0; level < kMaxLevels;) {
        const int stop = small ? kMaxLevels : std::min(kMaxLevels, level + kLevelsPerLook);
        for (; level < stop; level++) {
            if (small) continue;
            // a level has at most 4^level items
            const int64_t most = level < 14 ? std::min<int64_t>(n, (int64_t)1 << (2 * level)) : n;
            const unsigned blocks = (unsigned)std::min<int64_t>(1024, (most + 255) / 256);
            hipLaunchKernelGGL(k_wide_level, dim3(blocks), dim3(256), 0, st, b, level);
        }
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(&host, b.c, sizeof(host), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) return e;
        if (host.bad || host.slots > capacity) return hipSuccess;
        if (host.count[level] == 0) {
            scale = wideScale(host.root, host.root + 3);
            margins = wideMargins(host.stats, scale);
            return hipSuccess;
        }
    }
    return hipSuccess;
}

}  // namespace zgl
