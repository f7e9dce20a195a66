// rt_bvh_gpu.h -- the BVH builder that runs on the GPU (bvh_gpu.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <string>

#include "rt_internal.h"

namespace rt {

// A context's work space for builds: device memory grown on demand and kept
// for the next build (allocating and freeing ~130 B per triangle took longer
// than the kernels) up to kKeep bytes, and a pinned block for the read-backs.
// Builds of one context run one at a time under its lock, on its stream.
struct BvhBuildSpace {
    static constexpr size_t kKeep = (size_t)512 << 20, kPinned = 4096;
    void *dev = nullptr, *pinned = nullptr;
    size_t cap = 0;
    hipError_t reserve(size_t bytes, hipStream_t s);
    hipError_t reserve_pinned();
    void trim(hipStream_t s);  // gives back what is above kKeep
    void release();
};

// A tree built on the device: the two-wide nodes always (they are what
// rt_bvh_export copies), the four-wide nodes when the layout is four-wide,
// and the triangles in leaf order plus the degenerate sentinel; one
// allocation, at nodes2 (each hipFree of its own took 0.2 ms).
struct DeviceBvhBuild {
    Node2 *nodes2 = nullptr;
    Node4 *nodes4 = nullptr;
    Tri3 *tris = nullptr;
    void *extra = nullptr;    // the caller's bytes at the end of the allocation, 256-aligned
    uint32_t num_tris = 0, num_nodes2 = 0, num_nodes4 = 0, num_leaves = 0;
    uint32_t max_depth = 0;   // kept two-wide levels on the longest root-leaf path
    uint32_t depth4 = 0;      // levels of the four-wide tree
    uint32_t max_stack4 = 0;  // pending-entry bound of the four-wide traversal
    double sah_cost = 0.0, build_ms = 0.0;
};

// Builds from device-resident vertices (nv x 3 floats) and triangle indices
// (nt x 3) on stream s, with `extra` bytes for the caller behind the tree;
// synchronizes s.  On failure returns the HIP error
// (hipErrorInvalidValue for bad input) with err filled; what was allocated
// stays in out for free_bvh_device.
hipError_t build_bvh_device(const float *xyz, uint32_t nv, const uint32_t *idx, uint32_t nt, const rt_bvh_opts &o,
                            hipStream_t s, BvhBuildSpace &space, size_t extra, DeviceBvhBuild &out, std::string &err);
void free_bvh_device(DeviceBvhBuild &b);

// tris[k].flags = flags[tris[k].id] for the n real triangles (flags is a
// device array indexed by triangle id).
hipError_t set_transparent_device(Tri3 *tris, uint32_t n, const uint8_t *flags, hipStream_t s);

}  // namespace rt
