// omv_kernels.h -- host-side entry points of the gfx950 kernels (kernels.hip).
#ifndef OMV_KERNELS_H
#define OMV_KERNELS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/omv.h"
#include "omv_types.h"

#define OMV_BLOCK 128   // two wave64s per workgroup

namespace omv {

// Sample kernel over samples [sample0, sample0 + nsamples) of a chunk that
// covers whole pixels; rad receives 3 floats per sample (chunk-relative).
hipError_t launchBdpt(const OmvSceneView& S, const omv_camera_desc& cam, const omv_renderer_params& p, uint64_t sample0,
                      uint64_t nsamples, float* rad, float* lv, uint32_t* gstack, unsigned long long* counters, int blocks, float* splat,
                      hipStream_t stream);
// Ordered per-pixel reduction + PinholeCamera::stop for pixels [pix0, pix0 + npix).
// OMV_EXT_LIGHT_SPLAT: film (float4 per pixel) += splat (3 floats per pixel) * inv
hipError_t launchSplatAdd(const float* splat, uint64_t npix, float inv, float* film, hipStream_t stream);
hipError_t launchFilm(const float* rad, int spp, uint64_t pix0, uint64_t npix, float* film, hipStream_t stream);
hipError_t launchFc(const OmvSceneView& S, const omv_camera_desc& cam, uint32_t seed, float* film, int32_t* ids, uint8_t* tie,
                    uint32_t* gstack, unsigned long long* counters, int blocks, hipStream_t stream);
// Batched jobs: the device job record is opaque to the host; packBatchJob
// writes one record of batchJobBytes() bytes.  tileEnd[j] is the exclusive
// end of job j's range of work tiles (tilePixels(256 * tileWaves, spp) pixels each).
// counters: 16 u64 (8 statistics + the work counter), cleared by the launch.
hipError_t launchFillU64(unsigned long long* p, int n, hipStream_t stream);   // zero-fill, graph-capturable
size_t batchJobBytes();
void packBatchJob(void* dst, const OmvSceneView& S, const omv_camera_desc& cam, const omv_renderer_params& p, float* film,
                  uint64_t npix);
hipError_t launchBatch(const void* jobs, int njobs, const uint64_t* tileEnd, uint64_t totalTiles, int tileWaves,
                       unsigned long long* counters, float* lv, uint32_t* gstack, int blocks, bool nee, hipStream_t stream);
// Allocation-free render (noalloc.hip): one persistent launch over tiles with
// the file-scope scratch array; statsOut (may be null: no wait) receives the
// 8 counters after the stream has finished.  On failure err / what say why.
int renderNoalloc(const OmvSceneView& S, const omv_camera_desc& cam, const omv_renderer_params& p, float* film, hipStream_t stream,
                  unsigned long long statsOut[8], hipError_t& err, const char*& what);
// Wavefront render of one chunk of whole pixels (wavefront.hip).
struct WfLaunch {
    OmvSceneView S;
    omv_camera_desc cam;
    omv_renderer_params p;
    uint64_t sample0;          // first sample of the chunk
    uint32_t nslots;           // samples in the chunk
    int lvCap, lc;             // light vertices kept, connections per camera vertex
    void* arena;               // wavefrontArenaBytes(nslots, lvCap, lc, lights, nee, splat, sortRays, blocksShade, blocksGen)
    uint32_t* qcount;          // wavefrontCounterCount(B, lvCap) counters
    float* rad;                // 3 floats per sample of the chunk
    uint32_t* gstack;          // spill stacks of blocksTrace * OMV_BLOCK lanes
    unsigned long long* counters;
    int blocksGen, blocksTrace, blocksShade;
    int traceKeep;             // > 0: idle lanes refilled below this many busy ones; 0: the default of each launch
    hipEvent_t* traceEv;       // optional: an event pair around every traversal launch
    int traceEvCap;            // events available from traceEv
    int* traceEvUsed;          // events recorded so far (in/out)
    float* splat;              // OMV_EXT_LIGHT_SPLAT sums (3 floats per pixel), or null
    bool sortRays;             // reorder secondary camera rays before each traversal
    hipEvent_t roundEv;        // optional: recorded once camera round roundEvAt is
    int roundEvAt;             // done (or at the end when there are fewer rounds)
    int xcdBands;              // > 1: traversal queues dealt to this many XCDs in chunks (L2 locality); else plain stride
    int tailRound;             // >= 2: camera rounds tailRound .. B run as one launch (omv_wf_tail); else round by round
    // tailEarly >= 3: already from round tailEarly on if at most 3/4 of the paths start round 2.  Their number goes
    // to `alive` (pinned memory, with an event), and the host waits for it while the device runs that round
    int tailEarly;
    uint32_t* alive;
    hipEvent_t aliveEv;
    int blocksPacket;          // > 0: round-1 camera rays traced as wave packets (omv_wf_trace_cam1) on this many workgroups
};
// Pixels of a tile that one wave renders sample by sample (renderTile): about
// `samples` of them, at least one batch of 64 and at most 16 (the last batch
// of a tile is partly empty), in whole pixels, at most one a lane.
__host__ __device__ inline uint64_t tilePixels(uint64_t samples, int spp) {
    const uint64_t want = samples < 64 ? 64 : (samples > 1024 ? 1024 : samples), n = spp > 1 ? (uint64_t)spp : 1;
    const uint64_t pix = want / n;
    return pix < 1 ? 1 : (pix > 64 ? 64 : pix);
}
// A whole film as one persistent launch over such tiles (noalloc.hip): work is
// a zeroed work counter, gstack and lv hold blocks * OMV_BLOCK lanes.
int tileBlocksPerCU(bool lights, bool nee);
hipError_t launchTiles(const OmvSceneView& S, const omv_camera_desc& cam, const omv_renderer_params& p, float* film,
                       unsigned long long* counters, unsigned long long* work, uint32_t* gstack, float* lv, int blocks, hipStream_t stream);
// Ray queues are appended to through OMV_QSEG counters each (one per group of
// producing workgroups); wavefrontSegCap is the entries of one group's region
// for a producing launch of gridShade workgroups (blocksShade).
#define OMV_QSEG 64
uint32_t wavefrontSegCap(uint32_t nslots, int gridShade, int gridGen);
size_t wavefrontArenaBytes(uint32_t nslots, int lvCap, int lc, bool lights, bool nee, bool splat, bool sortRays, int gridShade, int gridGen);
int wavefrontCounterCount(int B, int lvCap);
// Resident workgroups per CU of the traversal, the generation, the round-1
// packet trace and the camera shading [lights][nee] kernels.
struct WfOccupancy { int trace, gen, packet, shade[2][2]; };
WfOccupancy wavefrontBlocksPerCU();
// Camera round from which the wavefront hands the remaining paths of a chunk
// to one tail launch (omv_wf_tail).  A round costs two or three launches that
// each wait for their longest ray, whatever its size; the tail waits for its
// longest path once but traces one path a lane.  So the fewer samples, the
// earlier.  MI355X, ms per render from round 2 / 3 / 4 / 5:
//   600 K samples: torus knot 0.63 0.76 0.89 1.00, with NEE 1.10 1.20 1.31
//     1.43, asset with a light 0.83 0.96 1.04 1.11, 60 instances and lights
//     0.76 0.84 0.94 1.04, mixed materials 0.97 0.80 0.90 0.92, masked with
//     lights among them 2.07 1.93 1.95 2.00
//   1.5 M: 0.98 0.99 1.11 1.21, 1.79 1.51 1.62 1.74, 1.15 1.21 1.30 1.38,
//     0.95 1.01 1.10 1.21, 1.68 1.33 1.17 1.27, 3.62 2.95 2.92 2.93
//   NEE 5.4 M: - 4.00 3.48 3.64; masked with lights 4.9 M: - - 5.94 5.80
//   16.8 M torus knot: - 5.07 4.59 4.72; 33 M instanced: - - 9.39 8.78
// (At 1.5 M scenes of one material type would gain from an earlier round still:
// with lights from 2, NEE from 3; mixed and masked ones from 4.)
// That holds while most paths escape: 0.12 - 0.65 of them start round 2 in those
// scenes, 0.01 - 0.18 round 3.  In a closed room 0.86 - 0.95 start round 2 and
// the tail is full of long paths: from round 3 / 4 / 5, 1 M samples, depth 20,
// 5.16 4.28 3.84 without lights, 30.5 26.5 23.6 with; 2 M, depth 8, 5.46 4.84
// 4.57, 29.6 25.8 23.3.  There the tail starts at lateTailRound.  A render
// counts the paths that start round 2; batches, which are captured, go by
// where the camera is (RenderScene::encloses).
inline int lateTailRound(bool lights, bool nee) { return lights || nee ? 5 : 4; }
inline int earlyTailRound(uint64_t slots, bool lights, bool nee) {
    if (!lights && !nee) return slots <= (1u << 21) ? 3 : 4;
    if (slots <= (1u << 20)) return 3;
    return slots <= (lights ? 1u << 22 : 1u << 23) ? 4 : 5;
}
hipError_t launchWavefront(const WfLaunch& L, hipStream_t stream);
// Path-replay adjoint over samples [sample0, sample0 + nsamples) (adjoint.hip).
int adjointBlocksPerCU();
hipError_t launchAdjoint(const OmvSceneView& S, const omv_camera_desc& cam, const omv_renderer_params& p, uint64_t sample0,
                         uint64_t nsamples, const float* dfilm, const int* texSlot, float* const* texGrad, const int* omSlot,
                         float* omGrad, float* lv, uint32_t* gstack, unsigned long long* counters, int blocks, hipStream_t stream);
// FP64 detached film (adjoint.hip): directions from S0, weights with S1's
// parameters, W*H*4 doubles; gstack holds blocks * OMV_BLOCK spill stacks.
int detachedBlocksPerCU();
hipError_t launchDetached(const OmvSceneView& S0, const OmvSceneView& S1, const omv_camera_desc& cam, const omv_renderer_params& p,
                          uint64_t npix, double* film, uint32_t* gstack, unsigned long long* counters, int blocks, hipStream_t stream);
// Film post pass (post.hip): gamma (+ 3x3 median when denoise) into outF, and
// the 8-bit truncation of outF into outU8 when non-null; tmp holds w*h float4.
hipError_t launchPost(const float* film, float* tmp, float* outF, uint8_t* outU8, int w, int h, float A, float gamma, bool denoise,
                      hipStream_t stream);
// Environment alias tables (env.hip); scratch holds 4*W*H + 2*H + 2 words.
// A box plane p relative to a pivot, rounded outward.
__host__ __device__ inline float planeFrom(float p, float pivot, bool upper) {
    const float d = p - pivot;
    const double exact = (double)p - (double)pivot;
    if (upper ? (double)d < exact : (double)d > exact) return nextafterf(d, upper ? INFINITY : -INFINITY);
    return d;
}
// bvh_device.hip: one mesh's BLAS built on the device (linear BVH collapsed
// into OmvNode4) into nodes[nodeBase ...] and records[12 * recBase ...], its
// boxes relative to pivot (on the host)
size_t blasDeviceScratchBytes(uint32_t n);
hipError_t buildBlasDevice(const float* vtx, uint32_t vtxOff, uint32_t stride, const uint32_t* faces, uint32_t faceOff, uint32_t n,
                           const float pivot[3], int leafMax, int recBase, int nodeBase, uint32_t nodeCap, OmvNode4* nodes, float* records, void* scratch,
                           hipStream_t stream, int* root, int* nodeCount, int* depth);
// mesh_device.hip: commitMesh's normals / tangents of one mesh on the device
size_t meshDeviceScratchBytes(uint32_t vn, uint32_t fn);
hipError_t preprocessMeshDevice(float* vertices, uint32_t stride, uint32_t vn, const uint32_t* faces, uint32_t fn, bool normals,
                                bool tangents, int uvOff, void* scratch, hipStream_t stream, uint32_t* badIndices);
// bvh_device.hip: one pass over the instances at commit.  World box of every
// instance and, per axis, the largest sum of the magnitudes of the terms
// behind a coordinate (rounding goes with it); of an instance without a BLAS
// (blas_root < 0) an empty box.  And the range of 1 / area over the world
// triangles of an area above FLT_EPSILON, infinity and 0 if there are none.
// (pivots: OmvSceneView::pivots)
struct OmvInstanceBox { double lo[3], hi[3], reach[3]; };
struct OmvDensityRange { float lo, hi; };
hipError_t instancePassDevice(const float* vtx, const uint32_t* faces, const OmvMesh* meshes, const OmvNode4* nodes, const OmvInstance* insts,
                              const float* pivots, uint32_t n, uint32_t maxFaces, OmvInstanceBox* boxes, OmvDensityRange* range, hipStream_t stream);
hipError_t launchEnvBuild(const float* bg, int W, int H, float* rowProb, int* rowAlias, float* colProb, int* colAlias, float* texPdf,
                          void* scratch, hipStream_t stream);
// 0: sample kernel (scene with lights), 1: FC kernel, 2: sample kernel (no lights), 3: batch kernel;
// 4, 5, 6: the sample kernels and the batch kernel with OMV_EXT_HDRI_NEE code
int occupancyBlocksPerCU(int which);

}  // namespace omv
#endif
