// bvh_device.hip -- bottom-level BVH build on the device, the alternative to
// the host binned-SAH builder (bvh.cpp) when commit time matters more than
// the last node visit (batched validation jobs).
//
//   1. one lane per triangle: box (relative to the mesh's pivot) and centroid
//      from the vertex pool; centroid bounds by a block reduction;
//   2. 30-bit Morton code of each centroid in those bounds; stable LSD radix
//      sort of (code, triangle) in four 8-bit passes (device_sort.h), so
//      equal codes keep triangle order;
//   3. the binary radix tree over the sorted codes (Karras, "Maximizing
//      parallelism in the construction of BVHs, octrees, and k-d trees",
//      2012), codes made unique by appending the sorted position;
//   4. a node's box is the union of a run of sorted leaves: boxes of every
//      aligned run of 2^k leaves first (lbRuns), of which a node takes at
//      most two of each length;
//   5. collapse into the 128-byte 4-wide nodes the traversal reads, one
//      level per launch: a node takes its binary node's two children and
//      keeps replacing the largest-area one by its children until it has
//      four; subtrees of <= leafMax triangles become leaves (their triangles
//      are contiguous in sorted order); child boxes widened outward,
//      as the host builder does;
//   6. triangle records (v0 + id, v1, v2) in sorted order.
//
// The closest hit does not depend on the tree (watertight test, ties broken
// by (t, instance, primitive); see Trav for grazing hits), so films equal the
// host-built scene's bit for bit; only node and triangle counts change.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cstdint>
#include <utility>

#include "device_sort.h"
#include "omv_kernels.h"

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kLeafBit = 0x80000000u;
constexpr int kCollapseLevels = 16;  // collapse levels launched between two readbacks (even)

// boxes of the aligned runs of 2^k sorted leaves, k = 0 .. count - 1: run j of
// length 2^k is box off[k] + j, the last of a length possibly shorter
struct LbRuns { uint32_t off[30]; int count; };

__device__ inline float padDown(float v) { for (int k = 0; k < OMV_BOX_PAD_ULPS; ++k) v = nextafterf(v, -INFINITY); return v; }
__device__ inline float padUp(float v) { for (int k = 0; k < OMV_BOX_PAD_ULPS; ++k) v = nextafterf(v, INFINITY); return v; }

// 1. triangle boxes and centroids; block partials of the centroid bounds
__global__ void lbBoxes(const float* __restrict__ vtx, uint32_t vtxOff, uint32_t stride, const uint32_t* __restrict__ faces,
                        uint32_t faceOff, uint32_t n, float3 pivot, float* __restrict__ box, float* __restrict__ cen, float* __restrict__ part) {
    __shared__ float red[6][kBlock];
    const uint32_t f = blockIdx.x * kBlock + threadIdx.x;
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    float c[3] = {INFINITY, INFINITY, INFINITY}, cm[3] = {-INFINITY, -INFINITY, -INFINITY};
    if (f < n) {
        for (int k = 0; k < 3; ++k) {
            const float* p = vtx + vtxOff + (size_t)faces[faceOff + 3 * f + k] * stride;
            for (int a = 0; a < 3; ++a) { lo[a] = fminf(lo[a], p[a]); hi[a] = fmaxf(hi[a], p[a]); }
        }
        for (int a = 0; a < 3; ++a) {
            const float at = a == 0 ? pivot.x : (a == 1 ? pivot.y : pivot.z);
            box[(size_t)6 * f + a] = omv::planeFrom(lo[a], at, false);
            box[(size_t)6 * f + 3 + a] = omv::planeFrom(hi[a], at, true);
            c[a] = cm[a] = 0.5f * lo[a] + 0.5f * hi[a];
            cen[(size_t)3 * f + a] = c[a];
        }
    }
    for (int a = 0; a < 3; ++a) { red[a][threadIdx.x] = c[a]; red[3 + a][threadIdx.x] = cm[a]; }
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int a = 0; a < 3; ++a) {
                red[a][threadIdx.x] = fminf(red[a][threadIdx.x], red[a][threadIdx.x + s]);
                red[3 + a][threadIdx.x] = fmaxf(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int a = 0; a < 6; ++a) part[(size_t)6 * blockIdx.x + a] = red[a][0];
}

// one block folds the partials
__global__ void lbBounds(const float* __restrict__ part, uint32_t nb, float* __restrict__ out) {
    __shared__ float red[6][kBlock];
    float v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (uint32_t b = threadIdx.x; b < nb; b += kBlock)
        for (int a = 0; a < 3; ++a) {
            v[a] = fminf(v[a], part[(size_t)6 * b + a]);
            v[3 + a] = fmaxf(v[3 + a], part[(size_t)6 * b + 3 + a]);
        }
    for (int a = 0; a < 6; ++a) red[a][threadIdx.x] = v[a];
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int a = 0; a < 3; ++a) {
                red[a][threadIdx.x] = fminf(red[a][threadIdx.x], red[a][threadIdx.x + s]);
                red[3 + a][threadIdx.x] = fmaxf(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int a = 0; a < 6; ++a) out[a] = red[a][0];
}

__device__ inline uint32_t spread10(uint32_t v) {   // 10 bits -> every third bit
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// 2a. Morton codes
__global__ void lbMorton(const float* __restrict__ cen, const float* __restrict__ bounds, uint32_t n, uint32_t* __restrict__ key,
                         uint32_t* __restrict__ val) {
    const uint32_t f = blockIdx.x * kBlock + threadIdx.x;
    if (f >= n) return;
    uint32_t q[3];
    for (int a = 0; a < 3; ++a) {
        const float ext = bounds[3 + a] - bounds[a];
        const float t = ext > 0.0f ? (cen[(size_t)3 * f + a] - bounds[a]) / ext : 0.0f;
        const float s = fminf(fmaxf(t * 1024.0f, 0.0f), 1023.0f);
        q[a] = (uint32_t)s;
    }
    key[f] = (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
    val[f] = f;
}

// 4a. Run boxes of lengths 2^(k0 + 1) .. 2^(k0 + 8) from those of 2^k0; at
// k0 = 0 the leaves' boxes too, gathered into sorted order.  A leaf box is
// read once and about two boxes a leaf are written, in up to four launches.
__global__ __launch_bounds__(kBlock) void lbRuns(const uint32_t* __restrict__ val, const float* __restrict__ triBox, uint32_t n, int k0,
                                                 LbRuns R, float* __restrict__ runs) {
    __shared__ float red[6][kBlock];
    const uint32_t t = threadIdx.x, i = blockIdx.x * kBlock + t;
    const uint32_t m = (uint32_t)(((uint64_t)n + (1ull << k0) - 1) >> k0);
    float v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (i < m) {
        const float* b = k0 == 0 ? triBox + (size_t)6 * val[i] : runs + (size_t)6 * (R.off[k0] + i);
        for (int a = 0; a < 6; ++a) v[a] = b[a];
        if (k0 == 0)
            for (int a = 0; a < 6; ++a) runs[(size_t)6 * i + a] = v[a];
    }
    for (int a = 0; a < 6; ++a) red[a][t] = v[a];
    for (int s = 1; s <= 8 && k0 + s < R.count; ++s) {
        __syncthreads();
        const uint32_t half = kBlock >> s, o = blockIdx.x * half + t;
        if (t < half)
            for (int a = 0; a < 3; ++a) {
                v[a] = fminf(red[a][2 * t], red[a][2 * t + 1]);
                v[3 + a] = fmaxf(red[3 + a][2 * t], red[3 + a][2 * t + 1]);
            }
        __syncthreads();
        if (t < half) {
            for (int a = 0; a < 6; ++a) red[a][t] = v[a];
            if (o < (uint32_t)(((uint64_t)n + (1ull << (k0 + s)) - 1) >> (k0 + s)))
                for (int a = 0; a < 6; ++a) runs[(size_t)6 * (R.off[k0 + s] + o) + a] = v[a];
        }
    }
}

// 3. radix tree; codes extended by the sorted position make them unique
__device__ inline int prefixLen(const uint32_t* __restrict__ key, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    const uint64_t a = ((uint64_t)key[i] << 32) | (uint32_t)i, b = ((uint64_t)key[j] << 32) | (uint32_t)j;
    return __clzll(a ^ b);
}

// and 4b. each node's box from the run boxes.  200 K triangles: 38 us with the
// run boxes made (MI355X); climbing from the leaves, a lane per leaf with a fence
// for the device and a counter at every node, took 927 us.
__global__ void lbTree(const uint32_t* __restrict__ key, int n, LbRuns R, const float* __restrict__ runs, uint32_t* __restrict__ left,
                       uint32_t* __restrict__ right, int* __restrict__ first, int* __restrict__ last, float* __restrict__ nodeBox) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n - 1) return;
    const int d = prefixLen(key, n, i, i + 1) > prefixLen(key, n, i, i - 1) ? 1 : -1;
    const int dmin = prefixLen(key, n, i, i - d);
    int lmax = 2;
    while (prefixLen(key, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (prefixLen(key, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = prefixLen(key, n, i, j);
    int s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (prefixLen(key, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    const int gamma = i + s * d + min(d, 0);
    const int lo = min(i, j), hi = max(i, j);
    first[i] = lo;
    last[i] = hi;
    left[i] = lo == gamma ? kLeafBit | (uint32_t)gamma : (uint32_t)gamma;
    right[i] = hi == gamma + 1 ? kLeafBit | (uint32_t)(gamma + 1) : (uint32_t)(gamma + 1);
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    auto take = [&](uint32_t run) {
        const float* q = runs + (size_t)6 * run;
        for (int a = 0; a < 3; ++a) { b[a] = fminf(b[a], q[a]); b[3 + a] = fmaxf(b[3 + a], q[3 + a]); }
    };
    uint32_t from = (uint32_t)lo, to = (uint32_t)hi + 1u;   // whole runs of 2^k leaves in [lo, hi], k rising
    for (int k = 0; from < to; ++k, from >>= 1, to >>= 1) {
        if (from & 1u) take(R.off[k] + from++);
        if (to & 1u) take(R.off[k] + --to);
    }
    for (int a = 0; a < 6; ++a) nodeBox[(size_t)6 * i + a] = b[a];
}

struct BinRef {   // a binary tree node: internal index, or a leaf with kLeafBit
    uint32_t ref;
};

__device__ inline int countOf(uint32_t ref, const int* first, const int* last) {
    return (ref & kLeafBit) ? 1 : last[ref] - first[ref] + 1;
}
__device__ inline int firstOf(uint32_t ref, const int* first) { return (ref & kLeafBit) ? (int)(ref & ~kLeafBit) : first[ref]; }
__device__ inline float halfArea(const float lo[3], const float hi[3]) {
    const float d0 = fmaxf(0.0f, hi[0] - lo[0]), d1 = fmaxf(0.0f, hi[1] - lo[1]), d2 = fmaxf(0.0f, hi[2] - lo[2]);
    return d0 * d1 + d1 * d2 + d2 * d0;
}

// Counters of the collapse: [0] output nodes, [1] overflow, [2 + l] jobs of
// level l of this batch of levels.  A later batch starts with the jobs left.
__global__ void lbCollapseInit(uint32_t* __restrict__ c, uint2* __restrict__ jobs, bool start, uint32_t root) {
    const uint32_t t = threadIdx.x;
    const uint32_t left = start ? 1u : c[2 + kCollapseLevels];
    __syncthreads();
    if (t <= kCollapseLevels) c[2 + t] = t == 0 ? left : 0u;
    if (t == 0 && start) { c[0] = 1u; c[1] = 0u; jobs[0] = make_uint2(root, 0u); }
}

// 5. one level of the collapse: jobs are (binary node, output node).  Their
// number stays on the device, so a whole batch of levels is launched at once.
__global__ void lbCollapse(const uint2* __restrict__ jobs, const uint32_t* __restrict__ jobCount, const uint32_t* __restrict__ left, const uint32_t* __restrict__ right,
                           const int* __restrict__ first, const int* __restrict__ last, const float* __restrict__ leafBox,
                           const float* __restrict__ nodeBox, int leafMax, int recBase, int nodeBase, uint32_t nodeCap,
                           OmvNode4* __restrict__ out, uint32_t* __restrict__ nodeCount, uint2* __restrict__ next, uint32_t* __restrict__ nextCount,
                           uint32_t* __restrict__ overflow) {
    const uint32_t njobs = *jobCount;
    for (uint32_t t = blockIdx.x * kBlock + threadIdx.x; t < njobs; t += gridDim.x * kBlock) {
        const uint32_t b = jobs[t].x, o = jobs[t].y;
        uint32_t kids[4];
        int nk = 0;
        if ((b & kLeafBit) || countOf(b, first, last) <= leafMax) {
            kids[nk++] = b;   // a small root: one-child node holding a leaf
        } else {
            kids[nk++] = left[b];
            kids[nk++] = right[b];
            while (nk < 4) {
                int best = -1;
                float bestA = -1.0f;
                for (int k = 0; k < nk; ++k) {
                    if ((kids[k] & kLeafBit) || countOf(kids[k], first, last) <= leafMax) continue;
                    float lo[3], hi[3];
                    for (int a = 0; a < 3; ++a) { lo[a] = nodeBox[(size_t)6 * kids[k] + a]; hi[a] = nodeBox[(size_t)6 * kids[k] + 3 + a]; }
                    const float ar = halfArea(lo, hi);
                    if (ar > bestA) { bestA = ar; best = k; }
                }
                if (best < 0) break;
                const uint32_t inner = kids[best];
                kids[best] = left[inner];
                kids[nk++] = right[inner];
            }
        }
        OmvNode4 nd;
        for (int k = 0; k < 4; ++k) {
            if (k >= nk) {
                nd.child[k] = OMV_EMPTY_CHILD;
                nd.entry[k] = OMV_ENT_NONE;
                nd.lox[k] = nd.loy[k] = nd.loz[k] = nd.hix[k] = nd.hiy[k] = nd.hiz[k] = INFINITY;   // no ray hits it
                continue;
            }
            const uint32_t c = kids[k];
            const float* bx = (c & kLeafBit) ? leafBox + (size_t)6 * (c & ~kLeafBit) : nodeBox + (size_t)6 * c;
            nd.lox[k] = padDown(bx[0]); nd.loy[k] = padDown(bx[1]); nd.loz[k] = padDown(bx[2]);
            nd.hix[k] = padUp(bx[3]); nd.hiy[k] = padUp(bx[4]); nd.hiz[k] = padUp(bx[5]);
            const int cnt = countOf(c, first, last);
            if (cnt <= leafMax) {
                nd.child[k] = -(recBase + firstOf(c, first) + 1);
                nd.entry[k] = OMV_ENT(OMV_ENT_BLAS_LEAF, ((uint32_t)(recBase + firstOf(c, first)) << 3) | ((uint32_t)(cnt - 1) & 7u));
            } else {
                const uint32_t idx = atomicAdd(nodeCount, 1u);
                if (idx >= nodeCap) {   // cannot happen (one output node per binary node); keep the launch in bounds
                    atomicAdd(overflow, 1u);
                    nd.child[k] = OMV_EMPTY_CHILD;
                    nd.entry[k] = OMV_ENT_NONE;
                    continue;
                }
                nd.child[k] = nodeBase + (int)idx;
                nd.entry[k] = OMV_ENT(OMV_ENT_BLAS_NODE, nodeBase + (int)idx);
                const uint32_t q = atomicAdd(nextCount, 1u);
                next[q] = make_uint2(c, idx);
            }
        }
        out[o] = nd;
    }
}

// 6. triangle records in sorted order
__global__ void lbRecords(const float* __restrict__ vtx, uint32_t vtxOff, uint32_t stride, const uint32_t* __restrict__ faces,
                          uint32_t faceOff, const uint32_t* __restrict__ val, uint32_t n, float* __restrict__ rec) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t prim = val[i];
    float* r = rec + (size_t)12 * i;
    for (int k = 0; k < 3; ++k) {
        const float* p = vtx + vtxOff + (size_t)faces[faceOff + 3 * prim + k] * stride;
        r[4 * k + 0] = p[0]; r[4 * k + 1] = p[1]; r[4 * k + 2] = p[2];
        r[4 * k + 3] = k == 0 ? __uint_as_float(prim) : 0.0f;
    }
}

// World boxes of instances, one wave each.  A lane follows one of the 64
// paths of three steps down the mesh's tree and turns the boxes of the up to
// four children it arrives at (or the box it ends in) by the instance's
// matrix: centre +- sum |M| * half extent.  The union of up to 256 turned
// boxes is far tighter on a rotated mesh than its turned root box, so rays
// enter fewer instances that they miss: 200 rotated meshes of 10 K triangles
// under lights, 1080p x 16 (MI355X), 6.59 -> 6.21 nodes per ray and 8.78 ->
// 8.39 ms per render.
__global__ __launch_bounds__(kBlock) void lbInstanceBoxes(const OmvNode4* __restrict__ nodes, const OmvInstance* __restrict__ insts,
                                                          const float* __restrict__ pivots, uint32_t n, omv::OmvInstanceBox* __restrict__ out, omv::OmvDensityRange* __restrict__ range) {
    if (blockIdx.x == 0 && threadIdx.x == 0) { range->lo = INFINITY; range->hi = 0.0f; }   // for lbDensity after this launch
    const uint32_t i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
    if (i >= n) return;
    const int lane = threadIdx.x & 63;
    const OmvInstance& in = insts[i];
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY}, reach[3] = {0.0, 0.0, 0.0};
    auto add = [&](const OmvNode4& nd, int k) {
        const float bl[3] = {nd.lox[k], nd.loy[k], nd.loz[k]}, bh[3] = {nd.hix[k], nd.hiy[k], nd.hiz[k]};
        for (int a = 0; a < 3; ++a) {
            const double t = (double)in.xfm[4 * a + 3];
            double mid = t, half = 0.0, terms = fabs(t);
            for (int c = 0; c < 3; ++c) {
                const double m = (double)in.xfm[4 * a + c], at = pivots ? pivots[4 * i + c] : 0.0f, l = at + bl[c], h = at + bh[c];
                mid += m * 0.5 * (l + h);
                half += fabs(m) * 0.5 * (h - l);
                terms += fabs(m) * fmax(fabs(l), fabs(h));
            }
            lo[a] = fmin(lo[a], mid - half);
            hi[a] = fmax(hi[a], mid + half);
            reach[a] = fmax(reach[a], terms);
        }
    };
    int node = in.blas_root;
    for (int shift = 4; node >= 0 && shift >= 0; shift -= 2) {
        const int k = (lane >> shift) & 3, c = nodes[node].child[k];
        if (c < 0 && c != OMV_EMPTY_CHILD) add(nodes[node], k);   // a leaf: the path ends
        node = c >= 0 && c != OMV_EMPTY_CHILD ? c : -1;
    }
    if (node >= 0)
        for (int k = 0; k < 4; ++k)
            if (nodes[node].child[k] != OMV_EMPTY_CHILD) add(nodes[node], k);
    for (int s = 32; s > 0; s >>= 1)
        for (int a = 0; a < 3; ++a) {
            lo[a] = fmin(lo[a], __shfl_xor(lo[a], s));
            hi[a] = fmax(hi[a], __shfl_xor(hi[a], s));
            reach[a] = fmax(reach[a], __shfl_xor(reach[a], s));
        }
    if (lane == 0)
        for (int a = 0; a < 3; ++a) { out[i].lo[a] = lo[a]; out[i].hi[a] = hi[a]; out[i].reach[a] = reach[a]; }
}

// Range of 1 / area over the world triangles.  1 / area is positive, so its
// bits order as it does and the result does not depend on the order.  Bound by
// the gathered vertices of a mesh; its many instances read them from the
// caches.  A loop on the host before: 200 K triangles 1.3 ms -> 13 us, 100 000
// instances of 5120 triangles 2330 -> 104 ms for the whole commit (MI355X).
__global__ __launch_bounds__(kBlock) void lbDensity(const float* __restrict__ vtx, const uint32_t* __restrict__ faces,
                                                    const OmvMesh* __restrict__ meshes, const OmvInstance* __restrict__ insts, uint32_t n,
                                                    uint32_t* __restrict__ range) {
    __shared__ uint32_t blockLo, blockHi;
    if (threadIdx.x == 0) { blockLo = 0x7F800000u; blockHi = 0u; }
    __syncthreads();
    uint32_t lo = 0x7F800000u, hi = 0u;
    for (uint32_t i = blockIdx.y; i < n; i += gridDim.y) {
        const OmvInstance& in = insts[i];
        if (in.mesh_id < 0) continue;
        const OmvMesh m = meshes[in.mesh_id];
        for (uint32_t f = blockIdx.x * kBlock + threadIdx.x; f < m.num_faces; f += gridDim.x * kBlock) {
            const uint32_t* F = faces + m.face_offset + (size_t)3 * f;
            float P[3][3];
            for (int k = 0; k < 3; ++k) {
                const float* p = vtx + m.vtx_offset + (size_t)F[k] * m.stride;
                for (int a = 0; a < 3; ++a) P[k][a] = in.xfm[4 * a] * p[0] + in.xfm[4 * a + 1] * p[1] + in.xfm[4 * a + 2] * p[2] + in.xfm[4 * a + 3];
            }
            const float u[3] = {P[1][0] - P[0][0], P[1][1] - P[0][1], P[1][2] - P[0][2]};
            const float v[3] = {P[2][0] - P[0][0], P[2][1] - P[0][1], P[2][2] - P[0][2]};
            const float c[3] = {u[1] * v[2] - u[2] * v[1], u[2] * v[0] - u[0] * v[2], u[0] * v[1] - u[1] * v[0]};
            const float area = sqrtf(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]) / 2.0f;
            if (area > FLT_EPSILON) {
                const uint32_t d = __float_as_uint(1.0f / (0.0f + area));
                lo = min(lo, d);
                hi = max(hi, d);
            }
        }
    }
    for (int s = 32; s > 0; s >>= 1) { lo = min(lo, __shfl_xor(lo, s)); hi = max(hi, __shfl_xor(hi, s)); }
    if ((threadIdx.x & 63) == 0) { atomicMin(&blockLo, lo); atomicMax(&blockHi, hi); }
    __syncthreads();
    if (threadIdx.x == 0) { atomicMin(&range[0], blockLo); atomicMax(&range[1], blockHi); }
}

inline uint32_t blocks(uint64_t n) { return (uint32_t)((n + kBlock - 1) / kBlock); }

}  // namespace

namespace omv {

// Scratch sizes for n triangles, in bytes (one allocation, carved below).
size_t blasDeviceScratchBytes(uint32_t n) {
    // 19 arrays, each rounded up to an even number of words
    return 4 * ((uint64_t)6 * n + 3 * n + 6 * blocks(n) + 8 + 4 * (uint64_t)n + sortHistWords(n) + 4 * (uint64_t)n +
                6 * (2 * (uint64_t)n + 32) + 6 * (uint64_t)n + 4 * (uint64_t)n + 2 + kCollapseLevels + 1 + 2 * 19) + 256;
}

hipError_t buildBlasDevice(const float* vtx, uint32_t vtxOff, uint32_t stride, const uint32_t* faces, uint32_t faceOff, uint32_t n,
                           const float pivot[3], int leafMax, int recBase, int nodeBase, uint32_t nodeCap, OmvNode4* nodes, float* records, void* scratch,
                           hipStream_t stream, int* root, int* nodeCount, int* depth) {
    *root = -1; *nodeCount = 0; *depth = 0;
    if (n == 0 || nodeCap == 0) return hipSuccess;
    if (nodeCap > n) nodeCap = n;   // one output node per binary node at most: the job queues hold n entries
    const uint32_t nb = blocks(n);
    uint32_t* p = static_cast<uint32_t*>(scratch);
    auto take = [&p](uint64_t words) { uint32_t* q = p; p += (words + 1) & ~(uint64_t)1; return q; };   // 8-byte aligned
    float* triBox = reinterpret_cast<float*>(take((uint64_t)6 * n));
    float* cen = reinterpret_cast<float*>(take((uint64_t)3 * n));
    float* part = reinterpret_cast<float*>(take((uint64_t)6 * nb));
    float* bounds = reinterpret_cast<float*>(take(8));
    uint32_t* keyA = take(n);
    uint32_t* valA = take(n);
    uint32_t* keyB = take(n);
    uint32_t* valB = take(n);
    uint32_t* hist = take(sortHistWords(n));
    uint32_t* left = take(n);
    uint32_t* right = take(n);
    int* first = reinterpret_cast<int*>(take(n));
    int* last = reinterpret_cast<int*>(take(n));
    float* runs = reinterpret_cast<float*>(take(6 * (2 * (uint64_t)n + 32)));
    float* nodeBox = reinterpret_cast<float*>(take((uint64_t)6 * n));
    uint2* jobsA = reinterpret_cast<uint2*>(take((uint64_t)2 * n));
    uint2* jobsB = reinterpret_cast<uint2*>(take((uint64_t)2 * n));
    uint32_t* counters = take(2 + kCollapseLevels + 1);

    LbRuns R;
    R.count = 0;
    for (uint64_t at = 0, m = n;; m = (m + 1) / 2) {   // n < 2^27: at most 28 lengths, fewer than 2 n + 32 boxes
        R.off[R.count++] = (uint32_t)at;
        at += m;
        if (m == 1) break;
    }
    hipError_t e;
    lbBoxes<<<nb, kBlock, 0, stream>>>(vtx, vtxOff, stride, faces, faceOff, n, make_float3(pivot[0], pivot[1], pivot[2]), triBox, cen, part);
    lbBounds<<<1, kBlock, 0, stream>>>(part, nb, bounds);
    lbMorton<<<nb, kBlock, 0, stream>>>(cen, bounds, n, keyA, valA);
    if ((e = sortPairs32(keyA, valA, keyB, valB, hist, n, 30, stream)) != hipSuccess) return e;
    for (int k0 = 0; k0 == 0 || k0 + 1 < R.count; k0 += 8)
        lbRuns<<<blocks(((uint64_t)n + (1ull << k0) - 1) >> k0), kBlock, 0, stream>>>(valA, triBox, n, k0, R, runs);
    if (n > 1) lbTree<<<blocks(n - 1), kBlock, 0, stream>>>(keyA, (int)n, R, runs, left, right, first, last, nodeBox);
    lbRecords<<<nb, kBlock, 0, stream>>>(vtx, vtxOff, stride, faces, faceOff, valA, n, records + (size_t)12 * recBase);
    if ((e = hipGetLastError()) != hipSuccess) return e;

    // Collapse, level by level from the root (binary node 0, or the single
    // leaf); the host reads the counts once per kCollapseLevels levels.  Level
    // l holds at most 4^l jobs; a grid of more than 1024 workgroups strides.
    const float* leafBox = runs;
    int levels = 0;
    for (bool more = true, start = true; more; start = false) {
        lbCollapseInit<<<1, 64, 0, stream>>>(counters, jobsA, start, n > 1 ? 0u : kLeafBit);
        uint2* cur = jobsA; uint2* nxt = jobsB;
        for (int l = 0; l < kCollapseLevels; ++l, std::swap(cur, nxt)) {
            const uint64_t most = levels + l < 16 ? std::min<uint64_t>(n, 1ull << (2 * (levels + l))) : n;
            lbCollapse<<<std::min(blocks(most), 1024u), kBlock, 0, stream>>>(cur, counters + 2 + l, left, right, first, last, leafBox, nodeBox,
                                                                             leafMax, recBase, nodeBase, nodeCap, nodes + nodeBase, counters,
                                                                             nxt, counters + 3 + l, counters + 1);
        }
        if ((e = hipGetLastError()) != hipSuccess) return e;
        uint32_t c[2 + kCollapseLevels + 1];
        if ((e = hipMemcpyAsync(c, counters, sizeof(c), hipMemcpyDeviceToHost, stream)) != hipSuccess) return e;
        if ((e = hipStreamSynchronize(stream)) != hipSuccess) return e;
        if (c[1]) return hipErrorInvalidValue;
        for (int l = 0; l < kCollapseLevels; ++l) levels += c[2 + l] != 0;
        more = c[2 + kCollapseLevels] != 0;
        *nodeCount = (int)c[0];
    }
    *root = nodeBase;
    *depth = levels;
    return hipGetLastError();
}

hipError_t instancePassDevice(const float* vtx, const uint32_t* faces, const OmvMesh* meshes, const OmvNode4* nodes, const OmvInstance* insts,
                              const float* pivots, uint32_t n, uint32_t maxFaces, OmvInstanceBox* boxes, OmvDensityRange* range, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    lbInstanceBoxes<<<(n + kBlock / 64 - 1) / (kBlock / 64), kBlock, 0, stream>>>(nodes, insts, pivots, n, boxes, range);
    // about four triangles a lane of the largest mesh, 4096 workgroups in all
    const uint32_t gx = std::min(std::max(blocks((uint64_t)maxFaces) / 4, 1u), 1024u), gy = std::min(n, std::max(4096u / gx, 1u));
    lbDensity<<<dim3(gx, gy), kBlock, 0, stream>>>(vtx, faces, meshes, insts, n, reinterpret_cast<uint32_t*>(range));
    return hipGetLastError();
}

}  // namespace omv
