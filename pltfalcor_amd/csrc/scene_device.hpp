// Device-resident scene buffers (HBM). Owned by plt_scene; raw pointers are passed to kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <vector>
#include "../../include/plt_abi.h"
#include "scene_host.hpp"

namespace plt {

struct DeviceSceneBuffers {
    float4* nodes = nullptr;          // 8 x float4 per BVH node (BvhNode, 128 B)
    float4* tris = nullptr;           // 3 x float4 per triangle, leaf order (48 B)
    float* positions = nullptr;       // 3 floats per vertex
    float* normals = nullptr;         // 3 floats per vertex
    uint32_t* indices = nullptr;      // 3 per triangle
    uint32_t* tri_mesh = nullptr;     // mesh per triangle
    uint32_t* mesh_material = nullptr;
    plt_spectral_profile* profiles = nullptr;
    uint32_t n_tris = 0, n_nodes = 0;
    size_t nodes_cap = 0;  // nodes that `nodes` has room for
    std::vector<void*> owned;
};

// A tree built on the device (bvh_device.hip): nodes and leaf-order triangles in allocations the
// caller takes over.
struct DeviceBvh {
    float4* nodes = nullptr;
    float4* tris = nullptr;
    uint32_t n_nodes = 0;
    size_t nodes_cap = 0;  // nodes that `nodes` has room for
    int max_depth = 0;   // levels of 4-wide nodes (root = 1)
    int iterations = 0;  // clustering iterations
    float ms = 0.f;      // wall-clock build time
};
// What a scene that rebuilds its tree on the device keeps between builds: one scratch allocation (about
// 300 B per triangle) and the buffers of the tree before the current one, which the next build writes.
// Nothing reads that tree any more: a tree is replaced only after the device has been waited for.
struct BvhWork {
    void* scratch = nullptr;
    size_t scratch_bytes = 0;
    float4* nodes = nullptr;
    size_t nodes_cap = 0;  // nodes of 128 B
    float4* tris = nullptr;  // n_tris records
    void release();
};
// Builds the BVH of the scene's device triangles (positions, indices, n_tris) on `st` into buffers taken
// from `work` (allocated where it has none that fit); returns PLT_EINVAL, with `out` untouched, when the
// tree would be deeper than the traversal stack holds.
int build_bvh_device(const DeviceSceneBuffers& d, hipStream_t st, BvhWork& work, DeviceBvh& out);

}  // namespace plt

// Definition of the ABI's opaque scene handle.
struct plt_scene {
    plt_context* ctx = nullptr;
    plt::HostScene host;
    plt::DeviceSceneBuffers dev;
    plt_bvh_info bvh{};  // the tree the scene holds: builder, nodes, levels, build time
    plt::BvhWork work;     // of plt_scene_build_bvh's device builds
};
