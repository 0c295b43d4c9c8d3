// Device BVH8 builder (bvh_build.hip): the host builder's tree
// (host/bvh_build.cpp), built on the GPU from the scene's device arrays.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../device/bvh.h"
#include "../device/common.h"

namespace rm {

// Triangles of one instance (or of one shape, in its object space).
struct BvhSource {
    uint32_t first;          // its first triangle in the build's triangle order
    uint32_t vertex_offset;
    uint32_t face_offset;
    uint32_t inst;           // instance id stored with its triangles
    uint32_t transformed;    // 0: vertices are taken as they are stored
    mat4 transform;
};

enum BvhDeviceStatus { kBvhBuilt = 0, kBvhUnsupported = 1, kBvhTooDeep = 2, kBvhQuantisation = 3 };

// Bytes of scratch memory for n triangles.
size_t bvh_device_scratch_bytes(uint32_t n);

// Builds the tree over n >= 2 triangles: `nodes` receives up to n nodes (the
// caller copies the first `*num_nodes`), `tris` n triangles in leaf order.
// kBvhUnsupported: the geometry holds values that are not finite, or the
// splits go deeper than the level loop; the host builder takes such input.
hipError_t bvh_device_build(const float* vertices, const uint32_t* indices, const BvhSource* sources,
                            uint32_t num_sources, uint32_t n, uint32_t max_leaf, void* scratch, Bvh8Node* nodes,
                            BvhTri* tris, uint32_t* num_nodes, uint32_t* depth, BvhDeviceStatus* status,
                            hipStream_t stream);

}  // namespace rm
