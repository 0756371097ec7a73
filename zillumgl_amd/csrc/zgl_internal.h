// zgl_internal.h -- launch interface between the C ABI layer and the kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "zgl_device.h"

namespace zgl {

// Integrator identifiers (the reference's NaivePath / LightPath / TriplePath).
constexpr int IntegNaive = 0;
constexpr int IntegLight = 1;
constexpr int IntegTriple = 2;

struct PassParams {
    int firstPass;      // uSpp of the first pass in the launch
    int nPasses;        // passes rendered by this launch
    int freeCounter;    // uFreeCounter of the first pass (incremented per pass)
    int maxDepth;
    int russianRoulette;
    int sampleLight;
    int lightEnvUniform;
    float lightPortion;
    int pathsPerPass;   // light tracer: workgroup size 1536 x blocks per pass
    int loopsPerPass;   // triple LPT loops per thread
    float lptScale;     // triple LPT uScale
};

// Counter slots (uint64): 0 bytes, 1 rows, 2 leaf tests, 3 traversals, 4 samples
constexpr int NumCounters = 8;

// Unit regions of the persistent schedules, one per XCD: each has its own counter (a
// batch has kUnitRegions counters per scene).
constexpr int kUnitRegions = 8;
// Ints between two regions' counters: a region's waves run on one XCD, and counters that
// share a cache line move it between the XCDs' L2s on every fetch.  In lines of their own:
// a 256 x 256 pass of the Cornell box 620 -> 330 us (every wave asks all regions at the
// end), the headline launch 105.6 -> 102 ms, ten batched scenes 18.4 -> 15.8 ms, the triple
// tracer 13.2 -> 11.9 ms.
constexpr int kCounterStride = 64;
constexpr size_t kCounterBytes = (size_t)kUnitRegions * kCounterStride * sizeof(int);

// A wave's place in the work: the region it takes units from and how many regions it has
// found used up in a row (the same in every lane).
struct UnitFetch {
    int region, exhausted;
};
ZGL_D UnitFetch unitFetch() { return UnitFetch{(int)(blockIdx.x % kUnitRegions), 0}; }  // workgroups go to XCDs in turn

// Units for the lanes that want one, all lanes of the wave together, one atomic for all of
// them: an index below nUnits, or -1 (ask again; every region is used up once
// f.exhausted is kUnitRegions).  The wave's own region first, then the others, one a call:
// at a launch's end the wave's other lanes walk on meanwhile (trying all eight in one call
// takes ten batched scenes from 15.8 to 16.3 ms and the material scene from 2.36 to 2.42).
ZGL_D int takeUnits(UnitFetch& f, int* counters, int nUnits, bool want)
{
    const unsigned long long need = __ballot(want);
    if (need == 0ull || f.exhausted >= kUnitRegions) return -1;
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((long long)need) - 1;
    const int len = (nUnits / (kUnitRegions * 64) + (nUnits % (kUnitRegions * 64) ? 1 : 0)) * 64;
    const int start = min(nUnits, f.region * len), limit = min(nUnits, start + len);
    int* c = counters + f.region * kCounterStride;
    int base = limit - start;
    // after a region that was used up the next one is looked at before it is added to
    if (lane == leader &&
        (f.exhausted == 0 || __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < base))
        base = atomicAdd(c, __popcll(need));
    base = __shfl(base, leader) + start;
    if (base >= limit) {
        f.region = (f.region + 1) % kUnitRegions;
        f.exhausted++;
        return -1;
    }
    f.exhausted = 0;
    const int idx = base + __popcll(need & ((1ull << lane) - 1ull));
    return want && idx < limit ? idx : -1;
}

// One scene of a batched persistent launch (device-resident table).
struct BatchScene {
    DevScene s;
    PassParams prm;
    float4* frame;
    float4* res;    // prm.nPasses x filmW x filmH sample values
    int threshold;  // lanes still walking when a wave working on this scene stops to shade
};

// The 4-wide tree of a scene's rows and triangles (zgl_wide.hip): slots holds
// wideCapacity(n) slots of 64 bytes, work wideWorkBytes(n) bytes.  scale.ok is false where
// the scene has no wide tree (its rays then take the rows); margins: up to what distance its
// walks keep subtrees.  Synchronises the stream.
int64_t wideCapacity(int64_t nTri);
size_t wideWorkBytes(int64_t nTri);
hipError_t buildWide(const float4* rows, const float4* tris, int64_t nTri, void* work, uint4* slots, hipStream_t st,
                     WideScale& scale, WideMargins& margins);
hipError_t launchSobolTable(const uint32_t* sobolM, uint32_t* tab, int first, int count, hipStream_t st);
// A scene's 48-byte triangles from its vertices and indices, and its RGB16F environment
// texels padded to 8 bytes.
hipError_t launchPackTriangles(const float* vertices, const int32_t* indices, int64_t n, float4* tris, hipStream_t st);
hipError_t launchPackEnv(const uint16_t* rgb, ushort4* env, int64_t n, hipStream_t st);
hipError_t launchFill(float* p, int64_t n, float v, hipStream_t st);
hipError_t launchSrgbExpand(const uint8_t* rgb, const float* lut, float4* out, int64_t n, hipStream_t st);
hipError_t launchPostProcess(const float4* frame, float4* out, unsigned char* rgb8, int w, int h, float scale, int tone,
                             hipStream_t st);
hipError_t launchFilmToFrame(const float* film, float4* frame, int w, int h, hipStream_t st);
hipError_t launchTraceClosest(const DevScene& s, const float* rays, int64_t n, int32_t* prim, float* t,
                              uint32_t* bin, unsigned long long* counters, hipStream_t st);
hipError_t launchTraceAny(const DevScene& s, const float* rays, const float* tmax, int64_t n,
                          uint8_t* occluded, hipStream_t st);
// res: per-sample values of up to resPasses passes (resPasses * W * H float4); the
// launch runs the passes in chunks of resPasses and adds each chunk to the frame in order.
hipError_t launchNaivePersistent(const DevScene& s, const PassParams& p, float4* frame, float4* res, int resPasses,
                                 int* pixelCounter, int threshold, int blocks, unsigned long long* counters,
                                 hipStream_t st);
// Workgroups of `threads` threads of `kernel` that one compute unit holds at once: the
// larger of `queried` (the runtime's occupancy query) and the residency computed from the
// kernel's VGPR count and static LDS for a CDNA3/4 compute unit (4 SIMDs, 512 VGPRs per
// lane allocated in granules of 8, at most 8 waves per SIMD, 160 KiB of LDS).  ROCm
// 7.2's runtime answered 2 for a 124-VGPR kernel of 256 threads that holds 4 per CU (so
// the ROCm 7.0 runtime, the measured launch times and the wave counters), and a process
// may bind the library to either runtime.  Launching more workgroups than fit is safe for
// these kernels (no workgroup waits on another); fewer leaves SIMDs idle.
int residentBlocksPerCU(const void* kernel, int threads, int queried);
int naivePersistentBlocksPerCU();
// The triple tracer's camera pass on the persistent schedule: p.nPasses passes in chunks
// of resPasses (res holds resPasses x W x H values), added to the planar film in order.
hipError_t launchTriplePersistent(const DevScene& s, const PassParams& p, float* film, float4* res, int resPasses,
                                  int* pixelCounter, int threshold, int blocks, hipStream_t st);
int triplePersistentBlocksPerCU();
// Traversal results logged per sample for the adjoint (see launchNaiveLogged).
constexpr int kHitLogQueries = 16;
// The persistent naive tracer over p's passes (all of them in one launch: res holds
// p.nPasses x W x H values, hitLog p.nPasses x W x H x kHitLogQueries entries), writing
// each sample's value to res and its traversal results to hitLog; the frame is untouched.
hipError_t launchNaiveLogged(const DevScene& s, const PassParams& p, float4* res, int2* hitLog, int* pixelCounter,
                             int threshold, int blocks, hipStream_t st);
int naiveBatchBlocksPerCU();
// maxPixels: the largest filmW x filmH of the batch (sizes the accumulate launch).
// The naive integrator's passes in FP64, one thread per pixel (zgl_reference.hip); sum
// holds W*H*3 per-pixel RGB sums and is added to.
hipError_t launchNaiveF64(const DevScene& s, const PassParams& p, double* sum, hipStream_t st);
hipError_t launchNaiveBatch(const BatchScene* items, int nScenes, int maxPixels, int* sceneCounters,
                            int blocks, hipStream_t st);
// Differentiable naive estimator: dFrame == null renders the replay estimator into
// frame; otherwise accumulates FP64 gradients into dMat (nMaterials x 5) and the envCopies
// copies of dEnv, summed into envSum (envW x envH x 3).
// hitLog (adjoint only, may be null): the traversal results of p's passes written by
// launchNaiveLogged; the replay then walks the MTBVH only for queries past the log.
hipError_t launchNaiveReplay(const DevScene& s, const PassParams& p, const float4* evalMat, const float4* evalEnv,
                             float4* frame, const float4* dFrame, double* dMat, double* dEnv, int envCopies,
                             double* envSum, const int2* hitLog, hipStream_t st);
// Global-queue path tracer: device bytes of the two item queues for a w x h film, blocks
// per CU of the extension kernel, and the launch of p.nPasses passes (counts: maxDepth + 1
// ints of device memory).
size_t globalQueueBytes(int w, int h);
int globalQueueBlocks();
hipError_t launchGlobalQueue(const DevScene& s, const PassParams& p, float4* frame, void* queues, int* counts,
                             int extendBlocks, hipStream_t st);
// Naive path tracer on the wavefront schedule (same frame as launchNaivePersistent):
// device bytes of its work buffer for a w x h film, blocks per CU of its trace and shade
// kernels, and the launch.
size_t wavefrontBytes(int w, int h, int passes);
// Passes rendered together (memory budget in bytes), spread evenly over the batches.
int wavefrontBatch(int w, int h, int nPasses, size_t budget);
void wavefrontBlocks(int& traceBlocksPerCU, int& shadeBlocksPerCU);
hipError_t launchNaiveWavefront(const DevScene& s, const PassParams& p, float4* frame, void* work, int batch,
                                int traceBlocks, int shadeBlocks, hipStream_t st);
hipError_t launchEnvExpand(const ushort4* env, float4* out, int64_t n, hipStream_t st);
// The light tracer (triple = false) or the triple tracer's light pass (triple = true)
// on the persistent schedule (zgl_lightpath.hip): p.nPasses passes of p.pathsPerPass
// units, splatted into the planar film; counter: one int of work queue.
hipError_t launchLightPersistent(const DevScene& s, const PassParams& p, bool triple, float* film, int* counter,
                                 int threshold, int blocks, hipStream_t st);
int lightPersistentBlocksPerCU(bool triple);
hipError_t launchLight(const DevScene& s, const PassParams& p, float* film, unsigned long long* counters,
                       hipStream_t st);
hipError_t launchTriplePT(const DevScene& s, const PassParams& p, float* film, unsigned long long* counters,
                          hipStream_t st);
hipError_t launchTripleLPT(const DevScene& s, const PassParams& p, float* film, unsigned long long* counters,
                           hipStream_t st);

}  // namespace zgl
