// bvh.h -- host BVH builder: binned-SAH binary tree collapsed into 4-wide
// nodes (OmvNode4).  Replaces the Embree scene build of the reference
// (RenderScene::buildEmbreeScene, pathtracer/src/scene/RenderScene.cpp:225-272):
// one BLAS per mesh, one TLAS over the instances.
#ifndef OMV_BVH_H
#define OMV_BVH_H

#include <stddef.h>
#include <stdint.h>
#include <vector>

#include "omv_types.h"

namespace omv {

struct BuildBox { float lo[3], hi[3]; };

struct Bvh4Result {
    int root = -1;          // node index in the output pool
    int depth = 0;          // BVH4 levels on the longest root-to-leaf path
    std::vector<int> order; // primitive ids in leaf order
};

// The point that a mesh's boxes are built relative to: its origin, or for a
// mesh far from its origin the middle of the box of up to 64 corners spread
// over its faces; true when it is not the origin.  The traversal's slab test
// is off by a few ulps of plane and origin (BoxRay), which far away is more
// than a triangle: torus knot of 100 K triangles and size 2 at 0, 1e2, 1e3,
// 1e4, 1e5, 1e6 from its origin, 512^2 x 16 on MI355X, 1.49, 1.33, 1.42, 1.88,
// 11.6, 696 ms with boxes about the origin, 1.50, 1.32, 1.38, 1.33, 1.35, 1.62
// relative to its middle.  So the line lies at 256 times the size of the box.
bool meshPivot(const float* vertices, size_t stride, const uint32_t* faces, int fn, float pivot[3]);

// Builds over `boxes` (one per primitive), appending nodes to `pool`.
// Leaves hold up to leafMax primitives; leaf slots encode
// child = -(leafBase + first + 1), where first indexes `order`.  Entries:
// a BLAS (tlas = false) gets OMV_ENT_BLAS_NODE / OMV_ENT_BLAS_LEAF
// ((leafBase + first) << 3 | count - 1); a TLAS (leafMax 1) gets
// OMV_ENT_TLAS_NODE / OMV_ENT_INST (leafBase + first, an index into `order`
// that the caller replaces by the instance id).
Bvh4Result buildBvh4(const std::vector<BuildBox>& boxes, int leafMax, int leafBase, std::vector<OmvNode4>& pool, bool tlas);

}  // namespace omv
#endif
