// bvh_host.h — host BVH8 builder interface.
#pragma once

#include <hip/hip_runtime.h>

#include <functional>
#include <mutex>
#include <string>
#include <vector>

#include "rt_layout.h"

namespace rt {

struct Bvh8Result {
    std::vector<Bvh8Node> nodes;
    std::vector<float> tris;     // 12 floats per triangle (3 x float4), leaf order
    uint32_t max_depth = 0;
    float sah_cost = 0.0f;
};

// tri: 9 floats per triangle (world-space v0, v1, v2), flattened id = index.
bool build_bvh8_host(const float* tri, uint64_t ntri, Bvh8Result& out, std::string& err);

// The triangles of a scene on the device, instance by instance (arrays of the
// scene's arena). tri_inst, tri_prim: filled by the build, or by
// launch_triangle_ids alone.
struct DeviceMesh {
    const InstanceRec* inst = nullptr;
    const float4* vertices = nullptr;
    const uint32_t* indices = nullptr;
    uint32_t* tri_inst = nullptr;
    uint32_t* tri_prim = nullptr;
    uint32_t num_inst = 0, num_tris = 0;
};

// A tree in the scratch memory of its build: copied from there, then freed.
struct DeviceBvh {
    void* scratch = nullptr;
    const Bvh8Node* nodes = nullptr;
    const float4* tris = nullptr;    // 3 per triangle, leaf order
    uint32_t num_nodes = 0, max_depth = 0;
    float sah_cost = 0.0f;
    DeviceBvh() = default;
    DeviceBvh(const DeviceBvh&) = delete;
    DeviceBvh& operator=(const DeviceBvh&) = delete;
    ~DeviceBvh();
};

// The same build on the current HIP device: binned SAH, collapsed to BVH8 with
// the host builder's node and triangle format. flatten: the world-space
// triangles by the host's arithmetic (9 floats each), asked for only when a
// coordinate is not finite. On return the work is complete.
bool build_bvh8_device(const DeviceMesh& mesh, const std::function<void(std::vector<float>&)>& flatten, DeviceBvh& out,
                       std::string& err);

hipError_t launch_triangle_ids(const DeviceMesh& mesh, hipStream_t st);

// Surface-area-heuristic cost of a BVH8 (FP64 sum over the child boxes of
// every node, relative to the root's area; leaf boxes weighted by their
// triangle count).
float bvh8_sah_cost(const std::vector<Bvh8Node>& nodes);

// 8-bit quantized copy of a BVH8 (same topology, header and meta). Every
// decoded child box contains the FP32 child box. Fails only for non-finite
// or astronomically large boxes (grid step above 2^127).
bool quantize_bvh8(const std::vector<Bvh8Node>& nodes, std::vector<QBvh8Node>& out, std::string& err);

}  // namespace rt
