// bvh_gpu.hpp -- binned-SAH BVH construction on the GPU (bvh_gpu.hip).
#pragma once
#include <vector>

#include "../../include/barnacle_hip.h"

namespace bnx {

struct Ctx;

// Trees of a build, in the context's buffers until its next one.
struct GpuBvh {
    std::vector<int> counts, n_nodes;             // per set: items, nodes
    const bn_bvh_node* nodes = nullptr;           // set after set (device)
    const int32_t* perm = nullptr;                // set after set (device)
};
// Builds one BVH per item set in a single GPU pass over all sets: sets[s]
// holds counts[s] items of 6 floats (pmin xyz, pmax xyz), all finite.  The
// nodes and permutation of each set are those of bnh::build_bvh (the
// reference's BVHNode.Build), bit for bit.  Runs on the context's stream.
GpuBvh bvh_build_gpu(Ctx* c, const std::vector<const float*>& sets, const std::vector<int>& counts);
// The nodes and permutation of every set into the caller's arrays.
void bvh_fetch(Ctx* c, const GpuBvh& g, const std::vector<bn_bvh_node*>& nodes, const std::vector<int32_t*>& perms);

}  // namespace bnx
