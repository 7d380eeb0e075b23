// node_ref.hpp -- how far the indices reach with which a traversal finds nodes
// and items, for host and device.
#pragma once
#include <stddef.h>
#include <stdint.h>

#ifndef __host__
#define __host__
#define __device__
#endif

namespace bnd {

// What a node record's child is: an interior node (the index of its record) or
// a leaf (kRefLeaf, count in the seven bits below, first item in the low
// kRefBits).  A traversal finds a record by its offset of 32 bits.
constexpr uint32_t kRefLeaf = 0x80000000u;
constexpr int kRefBits = 24;
constexpr size_t kRecBytes = 64;

// Whether records can stand for two pools of nodes over so many items: every
// item has a number, and every node could have a record that an offset reaches
// (a tree with leaves of no items has more nodes than two an item).
inline bool records_reach(size_t n_tris, size_t n_blas_nodes, size_t n_insts, size_t n_tlas_nodes) {
    constexpr size_t items = ((size_t)1 << kRefBits) - 1, nodes = ((size_t)1 << 32) / kRecBytes;
    return n_tris < items && n_insts < items && n_blas_nodes <= nodes && n_tlas_nodes <= nodes;
}

// Where half `half` of node i lies in a pool of nodes, in 16-byte words.  A
// scene's BLAS share one pool, which may hold 2^30 nodes and more.
__host__ __device__ inline size_t node_at(int i, int half) { return 2 * (size_t)(uint32_t)i + (size_t)half; }

}  // namespace bnd
