// The traversal of path_device.h, run on the CPU one lane at a time over small
// two-level scenes, under AddressSanitizer: an entry taken for an instance
// that it is not reads far outside the instance array and ends the program.
// build: test_traversal_hostsim.py, which makes PATH_DEVICE (path_device.h
// with its inline assembly replaced by C++).
//
// Usage: trav_host < cases.  A case is
//   nmesh  { nvert nface  xyz..  faces.. }  ninst { mesh  xfm[12] inv[12] }
//   nray   { o[3] d[3] tnear tfar }
// in binary (int32 / float32).  Per ray it prints the closest hit of the
// traversal and of a loop over all triangles of all instances:
//   inst prim bits(t) nodes  inst prim bits(t)
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include <hip/hip_runtime.h>

#include "bvh.h"

namespace {
uint32_t bitsOf(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }
float floatOf(uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }
// v_rcp_f32: within one ulp of the quotient, here one ulp off either way by turns
int rcpOff = 0;
float rcpApprox(float x) {
    const float r = 1.0f / x;
    if (!std::isfinite(r) || r == 0.0f || std::fabs(x) > 8e37f) return r;
    rcpOff = (rcpOff + 1) % 3;
    return rcpOff == 0 ? r : std::nextafter(r, rcpOff == 1 ? INFINITY : -INFINITY);
}
using std::isfinite;
struct Dim { uint32_t x; };
const Dim threadIdx = {0}, blockIdx = {0}, gridDim = {1}, blockDim = {1};
// one lane: a ballot is the lane's own bit, a shuffle its own value
uint64_t __ballot(bool b) { return b ? 1ull : 0ull; }
template <class T> T __shfl(T v, int, int = 64) { return v; }
template <class T> T __shfl_xor(T v, int, int = 64) { return v; }
uint32_t __float_as_uint(float f) { return bitsOf(f); }
int __float_as_int(float f) { return (int)bitsOf(f); }
float __uint_as_float(uint32_t u) { return floatOf(u); }
float __int_as_float(int i) { return floatOf((uint32_t)i); }
int __ffsll(unsigned long long v) { return __builtin_ffsll((long long)v); }
int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
template <class T> T atomicAdd(T* p, T v) { T o = *p; *p += v; return o; }
template <class T> T min(T a, T b) { return b < a ? b : a; }
template <class T> T max(T a, T b) { return a < b ? b : a; }
double minF64(double a, double b) { return a < b ? a : b; }
double maxF64(double a, double b) { return a < b ? b : a; }
}  // namespace
#define __builtin_amdgcn_rcpf rcpApprox
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_wave_barrier() ((void)0)

#include PATH_DEVICE

uint32_t omv_lds_stack[OMV_STACK_LDS * OMV_BLOCK];

namespace {
template <class T> T rd() {
    T v;
    if (std::fread(&v, sizeof(v), 1, stdin) != 1) std::exit(3);
    return v;
}
}  // namespace

int main() {
    std::vector<OmvNode4> nodes;
    std::vector<float> tris;
    struct Mesh { int root, first, count; float lo[3], hi[3], pivot[3]; bool far; };
    std::vector<Mesh> meshes(rd<int32_t>());
    for (Mesh& m : meshes) {
        std::vector<float> v((size_t)3 * rd<int32_t>());
        std::vector<uint32_t> f((size_t)3 * rd<int32_t>());
        for (float& x : v) x = rd<float>();
        for (uint32_t& i : f) i = rd<uint32_t>();
        m.far = omv::meshPivot(v.data(), 3, f.data(), (int)(f.size() / 3), m.pivot);
        std::vector<omv::BuildBox> boxes(f.size() / 3);
        for (int a = 0; a < 3; ++a) { m.lo[a] = INFINITY; m.hi[a] = -INFINITY; }
        for (size_t t = 0; t < boxes.size(); ++t)
            for (int a = 0; a < 3; ++a) {
                const float p = v[3 * f[3 * t] + a], q = v[3 * f[3 * t + 1] + a], r = v[3 * f[3 * t + 2] + a];
                boxes[t].lo[a] = std::fmin(p, std::fmin(q, r));
                boxes[t].hi[a] = std::fmax(p, std::fmax(q, r));
                m.lo[a] = std::fmin(m.lo[a], boxes[t].lo[a]);
                m.hi[a] = std::fmax(m.hi[a], boxes[t].hi[a]);
                boxes[t].lo[a] = omv::planeFrom(boxes[t].lo[a], m.pivot[a], false);
                boxes[t].hi[a] = omv::planeFrom(boxes[t].hi[a], m.pivot[a], true);
            }
        m.first = (int)(tris.size() / 12);
        m.count = (int)boxes.size();
        const omv::Bvh4Result r = omv::buildBvh4(boxes, OMV_BVH_LEAF_MAX, m.first, nodes, false);
        m.root = r.root;
        for (int prim : r.order)
            for (int k = 0; k < 3; ++k) {
                for (int a = 0; a < 3; ++a) tris.push_back(v[3 * f[3 * prim + k] + a]);
                tris.push_back(k == 0 ? floatOf((uint32_t)prim) : 0.0f);
            }
    }
    std::vector<OmvInstance> insts(rd<int32_t>());
    std::vector<omv::BuildBox> iboxes;
    std::vector<float> pivots;
    bool anyPivot = false;
    for (const Mesh& m : meshes) anyPivot = anyPivot || m.far;
    for (OmvInstance& in : insts) {
        std::memset(&in, 0, sizeof(in));
        in.mesh_id = rd<int32_t>();
        for (float& x : in.xfm) x = rd<float>();
        for (float& x : in.inv) x = rd<float>();
        const Mesh& m = meshes[in.mesh_id];
        in.blas_root = m.root;
        pivots.insert(pivots.end(), {m.pivot[0], m.pivot[1], m.pivot[2], 0.0f});
        omv::BuildBox b;
        for (int a = 0; a < 3; ++a) {
            double mid = in.xfm[4 * a + 3], half = 0.0, reach = std::fabs(mid);
            for (int c = 0; c < 3; ++c) {
                const double x = in.xfm[4 * a + c];
                mid += x * 0.5 * ((double)m.lo[c] + m.hi[c]);
                half += std::fabs(x) * 0.5 * ((double)m.hi[c] - m.lo[c]);
                reach += std::fabs(x) * std::fmax(std::fabs(m.lo[c]), std::fabs(m.hi[c]));
            }
            const double pad = 1e-5 * std::fmax(std::fabs(mid - half) + std::fabs(mid + half), reach) + 1e-20;
            b.lo[a] = std::nextafter((float)(mid - half - pad), -INFINITY);
            b.hi[a] = std::nextafter((float)(mid + half + pad), INFINITY);
        }
        iboxes.push_back(b);
    }
    const size_t tlas0 = nodes.size();
    const omv::Bvh4Result tl = omv::buildBvh4(iboxes, 1, 0, nodes, true);
    for (size_t n = tlas0; n < nodes.size(); ++n)
        for (int k = 0; k < 4; ++k)
            if (nodes[n].child[k] != OMV_EMPTY_CHILD && nodes[n].child[k] < 0)
                nodes[n].entry[k] = OMV_ENT(OMV_ENT_INST, tl.order[-(nodes[n].child[k] + 1)]);
    OmvSceneView S;
    std::memset(&S, 0, sizeof(S));
    S.nodes = nodes.data(); S.insts = insts.data(); S.tris = tris.data();
    S.pivots = anyPivot ? pivots.data() : nullptr;
    S.num_insts = (int)insts.size(); S.tlas_root = tl.root;

    std::vector<uint32_t> spill((size_t)(OMV_STACK_TOTAL - OMV_STACK_LDS) * OMV_BLOCK);
    Stack st;
    st.init(spill.data(), OMV_BLOCK);
    const int nray = rd<int32_t>();
    for (int i = 0; i < nray; ++i) {
        f3 o, d;
        o.x = rd<float>(); o.y = rd<float>(); o.z = rd<float>();
        d.x = rd<float>(); d.y = rd<float>(); d.z = rd<float>();
        const float tnear = rd<float>(), tfar = rd<float>();
        Counters c;
        c.zero();
        Hit h, g;
        const bool hit = traceClosest(S, o, d, tnear, tfar, h, st, c);
        if (c.overflow()) return 4;
        g.inst = -1; g.prim = 0; g.t = tfar; g.tie = false;
        if (std::fabs(d.x) > 0.0f || std::fabs(d.y) > 0.0f || std::fabs(d.z) > 0.0f)
            for (size_t k = 0; k < insts.size(); ++k) {
                const float* I = insts[k].inv;
                const f3 oo = mk3(I[0] * o.x + I[1] * o.y + I[2] * o.z + I[3], I[4] * o.x + I[5] * o.y + I[6] * o.z + I[7],
                                  I[8] * o.x + I[9] * o.y + I[10] * o.z + I[11]);
                const f3 od = mk3(I[0] * d.x + I[1] * d.y + I[2] * d.z, I[4] * d.x + I[5] * d.y + I[6] * d.z, I[8] * d.x + I[9] * d.y + I[10] * d.z);
                TriRay p;
                if (!rayPrep(oo, od, p)) continue;
                const Mesh& m = meshes[insts[k].mesh_id];
                for (int t = m.first; t < m.first + m.count; ++t) {
                    const float4* r = reinterpret_cast<const float4*>(tris.data()) + 3 * t;
                    float tt, u, v;
                    if (triIntersect(p, r[0], r[1], r[2], tnear, g.t, tt, u, v)) offer(g, tt, u, v, (int)k, __float_as_int(r[0].w));
                }
            }
        std::printf("%d %d %u %u %d %d %u\n", hit ? h.inst : -1, hit ? h.prim : 0, hit ? bitsOf(h.t) : 0u, c.nodes, g.inst, g.prim,
                    g.inst >= 0 ? bitsOf(g.t) : 0u);
    }
    return 0;
}
