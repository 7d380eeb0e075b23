// bvh_gpu.hip -- binned-SAH BVH construction on the GPU, node for node the
// build of BVHNode.Build (Util/BVH.fs:128-247): the same nodes in the same
// pre-order and the same item permutation as the recursive host build.
//
// What makes a parallel build exact:
//  * Every bound is a fold of MinNative/MaxNative over items in their order
//    (AABB.Union(acc, x): x wins ties, so of -0 and +0 the later one stays).
//    "Later wins ties" is associative, so the folds are evaluated as trees
//    that only ever join a range with the range right after it; with finite
//    inputs the result is bit-identical to the sequential fold.  Non-finite
//    bounds break associativity and are refused (the host build takes them).
//  * Bin counts, partition counts and positions are integers; the partition
//    is the reference's: left items in order from `first`, right items in
//    order from `last - 1` downwards (Util/BVH.fs:205-217).
//  * The SAH sweep of a node folds each prefix and suffix of its bins in a lane
//    of its own, in the reference's order.
//
// Schedule: a task is a node's item range.  Tasks of more than `small` items
// run level by level over chunks of kChunk items: bounds, bins and the scatter
// by one block per chunk, the decisions (split axis; split and children) by one
// wave or block per task.  Task and chunk counts stay on the device: the levels
// are launched for the most they can have, several levels at a time.  A task of
// at most `small` items (or at depth 64, where more than 127 are refused) is
// built whole by one wave into a node region of its own, of two nodes an item.
// One block numbers the upper nodes and regions in pre-order, and a last pass
// writes the flattened nodes.  A level takes 55 us for 240,000 items; with
// decisions by one thread per task, a copy of the counters and a host
// synchronisation it took 120, and with the decisions in the block that finishes
// a task's last chunk 90 (the fences).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "abi_internal.hpp"
#include "bvh_gpu.hpp"
#include "wave.hpp"

namespace bvhg {

constexpr int kBins = 12, kLeaf = 4, kMaxDepth = 64;        // BVHBuildConfig (Util/BVH.fs:99-107)
constexpr int kLeafMost = 127;                              // what a node's int8 count holds
constexpr int kThreads = 256, kIpt = 4;
constexpr int kChunk = kThreads * kIpt;                     // items per chunk block
constexpr int kWavesPerBlock = kThreads / 64;
constexpr float kInf = __builtin_huge_valf();

// 32-byte item: bounds and the item's index in its set.
struct alignas(16) Item { float lx, ly, lz; int32_t id; float hx, hy, hz; int32_t pad; };
struct DBox { float l[3], h[3]; };
struct BigTask { int first, last, depth, unode, set, chunk0, nchunks, pad; };
struct BigInfo { int mode, axis, best, pad; float lo_axis, extent, cb_area, pad1; };   // mode 0 bin, 1 middle
struct SmallTask { int first, last, depth, buf, set, pad0, pad1, pad2; };
struct UNode { DBox b; int axis, left, right, set; };      // child < 0: small task ~child
constexpr int kLevels = kMaxDepth + 1;
struct Ctl {
    int n_small, n_unodes, err, pad;
    int n_big[kLevels], n_chunks[kLevels];                 // tasks and chunks of each level
    int unode_end[kLevels];                                // end of the level's upper nodes (numbered level by level)
};
constexpr int kErrLeaf = 1, kErrCapacity = 2, kErrFinite = 4, kErrCount = 8;

__device__ __forceinline__ float omin(float a, float b) { return a < b ? a : b; }
__device__ __forceinline__ float omax(float a, float b) { return a > b ? a : b; }
__device__ __forceinline__ DBox empty_box() { return {{kInf, kInf, kInf}, {-kInf, -kInf, -kInf}}; }
// a covers items before b
__device__ __forceinline__ DBox join(const DBox& a, const DBox& b) {
    DBox r;
#pragma unroll
    for (int k = 0; k < 3; ++k) { r.l[k] = omin(a.l[k], b.l[k]); r.h[k] = omax(a.h[k], b.h[k]); }
    return r;
}
__device__ __forceinline__ Item load_item(const Item* p) {
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    Item it;
    it.lx = a.x; it.ly = a.y; it.lz = a.z; it.id = __float_as_int(a.w);
    it.hx = b.x; it.hy = b.y; it.hz = b.z; it.pad = 0;
    return it;
}
__device__ __forceinline__ void store_item(Item* p, const Item& it) {
    reinterpret_cast<float4*>(p)[0] = make_float4(it.lx, it.ly, it.lz, __int_as_float(it.id));
    reinterpret_cast<float4*>(p)[1] = make_float4(it.hx, it.hy, it.hz, 0.0f);
}
__device__ __forceinline__ DBox item_box(const Item& it) { return {{it.lx, it.ly, it.lz}, {it.hx, it.hy, it.hz}}; }
// AABB.Centroid = 0.5f * (pMin + pMax), as a point box for Union(acc, point)
__device__ __forceinline__ DBox centroid_box(const Item& it) {
    const float cx = 0.5f * (it.lx + it.hx), cy = 0.5f * (it.ly + it.hy), cz = 0.5f * (it.lz + it.hz);
    return {{cx, cy, cz}, {cx, cy, cz}};
}
__device__ __forceinline__ float centroid_on(const Item& it, int axis) {
    return axis == 0 ? 0.5f * (it.lx + it.hx) : axis == 1 ? 0.5f * (it.ly + it.hy) : 0.5f * (it.lz + it.hz);
}
// findBinIndex (Util/BVH.fs:163-168): int of (12 * (c - lo)) / extent, at most 11
__device__ __forceinline__ int bin_of(const Item& it, int axis, float lo, float extent) {
    const float v = (12.0f * (centroid_on(it, axis) - lo)) / extent;
    return min(kBins - 1, (int)v);
}
// AABB.SurfaceArea: 2 * (dx dy + dy dz + dz dx)
__device__ __forceinline__ float area(const DBox& b) {
    const float dx = b.h[0] - b.l[0], dy = b.h[1] - b.l[1], dz = b.h[2] - b.l[2];
    return 2.0f * (dx * dy + dy * dz + dz * dx);
}
// AABB.SplitAxis of the centroid bounds
__device__ __forceinline__ int split_axis(const DBox& b) {
    const float dx = b.h[0] - b.l[0], dy = b.h[1] - b.l[1], dz = b.h[2] - b.l[2];
    if (dx >= dy && dx >= dz) return 0;
    return dy >= dz ? 1 : 2;
}

// Ordered union over the lanes of a wave (lane i's items precede lane i+1's);
// the result is broadcast to every lane.
__device__ DBox wave_union(DBox v) {
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        DBox o;
#pragma unroll
        for (int k = 0; k < 3; ++k) { o.l[k] = __shfl_down(v.l[k], s); o.h[k] = __shfl_down(v.h[k], s); }
        v = join(v, o);                       // meaningful in lanes that are multiples of 2s
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) { v.l[k] = __shfl(v.l[k], 0); v.h[k] = __shfl(v.h[k], 0); }
    return v;
}
// Ordered union over a block (waves in order); every thread gets the result.
__device__ DBox block_union(DBox v, DBox* sh) {
    v = wave_union(v);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) sh[w] = v;
    __syncthreads();
    DBox r = sh[0];
    for (int k = 1; k < kWavesPerBlock; ++k) r = join(r, sh[k]);
    __syncthreads();
    return r;
}
__device__ int block_excl_scan(int x, int* sh) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int v = x;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const int y = __shfl_up(v, s);
        if (lane >= s) v += y;
    }
    if (lane == 63) sh[w] = v;
    __syncthreads();
    int off = 0;
    for (int k = 0; k < w; ++k) off += sh[k];
    __syncthreads();
    return off + v - x;
}

// A box as six maxima (-lo, hi): the negation is exact, and a min whose second
// operand wins ties is the negated max whose second operand wins them.
struct Box6 { float v[6]; };
__device__ __forceinline__ float later_max(float a, float b) { return a > b ? a : b; }
__device__ __forceinline__ Box6 empty6() { return {{-kInf, -kInf, -kInf, -kInf, -kInf, -kInf}}; }
__device__ __forceinline__ void join6(Box6& a, const Box6& b) {
#pragma unroll
    for (int c = 0; c < 6; ++c) a.v[c] = later_max(a.v[c], b.v[c]);
}
__device__ __forceinline__ DBox dbox(const Box6& b) { return {{-b.v[0], -b.v[1], -b.v[2]}, {b.v[3], b.v[4], b.v[5]}}; }

struct Bufs {
    Item* items[2];
    BigTask* big[2];         // by level parity
    BigInfo* info;
    SmallTask* small;
    int* chunk_task[2];      // by level parity
    int* chunk_start[2];
    DBox* part_b;            // per chunk: item bounds
    DBox* part_cb;           // per chunk: centroid bounds
    Box6* bin_b;             // per chunk x bin
    int* bin_n;
    int* chunk_lbase;
    int* chunk_rbase;
    UNode* unodes;
    int *udfs, *uright, *usize;   // per upper node: index, right child, subtree nodes
    bn_bvh_node* region;     // 2 * first: the region of the small task starting at `first`
    int* small_size;         // nodes of each small task's region
    int* small_base;         // the region's first node in its set
    int32_t* perm;           // per position: item id
    const int* set_off;      // first item of each set, and the end
    const int* root;         // root code of each set: an upper node, or ~(small task)
    int* set_nodes;          // nodes of each set
    int* set_base;           // first node of each set in the output
    Ctl* ctl;
    int n_sets, n_items, small_max, big_cap, small_cap, unode_cap, chunk_cap;
};

// The items of all sets from their bounds; their ids count within the set.
__global__ void __launch_bounds__(kThreads) k_items(Bufs B, const float* bounds) {
    bool finite = true;
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < B.n_items; i += gridDim.x * kThreads) {
        const float2* p = reinterpret_cast<const float2*>(bounds) + 3 * (size_t)i;
        const float2 a = p[0], b = p[1], c = p[2];
        int lo = 0, hi = B.n_sets - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (B.set_off[mid] <= i) lo = mid; else hi = mid - 1;
        }
        Item it;
        it.lx = a.x; it.ly = a.y; it.lz = b.x; it.id = i - B.set_off[lo];
        it.hx = b.y; it.hy = c.x; it.hz = c.y; it.pad = 0;
        finite = finite && isfinite(a.x) && isfinite(a.y) && isfinite(b.x) && isfinite(b.y) && isfinite(c.x) &&
                 isfinite(c.y);
        store_item(B.items[0] + i, it);
    }
    if (__ballot(!finite) != 0 && (threadIdx.x & 63) == 0) atomicOr(&B.ctl->err, kErrFinite);
}

// The thread's items of a chunk: [s + t * kIpt, ...) within [s, e).
__device__ __forceinline__ void thread_range(int s, int e, int& b, int& en) {
    b = min(s + (int)threadIdx.x * kIpt, e);
    en = min(b + kIpt, e);
}

// Bounds and counts of a node's twelve bins, for the sweep.
struct SplitLds {
    float bin_box[kBins][6];
    int bin_n[kBins];
};
// SAH sweep of a node of cnt items (Util/BVH.fs:183-203) by one wave, prefixes
// and suffixes of the bins side by side, each folded in the reference's order:
// the best split and the number of items left of it.
__device__ __forceinline__ void sah_sweep(const SplitLds& S, int cnt, float cb_area, int& best, int& n_left) {
    const int lane = threadIdx.x & 63;
    // lane s < 11: bins [0, s] in ascending order; lane 16 + s: bins [s + 1, 12) in descending order
    const bool right = (lane & 16) != 0;
    const int s = lane & 15;
    Box6 acc = empty6();
    int c = 0;
    for (int t = 0; t < kBins - 1; ++t) {
        const int q = right ? kBins - 1 - t : t;
        if (right ? t <= kBins - 2 - s : t <= s) {
#pragma unroll
            for (int w = 0; w < 6; ++w) acc.v[w] = later_max(acc.v[w], S.bin_box[q][w]);
            c += S.bin_n[q];
        }
    }
    const float cost1 = (float)c * area(dbox(acc));
    const float cost = (cost1 + __shfl(cost1, lane + 16)) + (float)cnt * cb_area;
    const bool valid = lane < kBins - 1 && cost < kInf;
    float m = valid ? cost : kInf;
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) m = fminf(m, __shfl_xor(m, o));
    const uint64_t at = __ballot(valid && cost == m);
    best = at ? __ffsll((unsigned long long)at) - 1 : 0;
    n_left = __builtin_amdgcn_readlane(c, best);
}

// Per chunk: item bounds and centroid bounds.
__global__ void __launch_bounds__(kThreads) k_chunk_bounds(Bufs B, int level) {
    __shared__ DBox sh[kWavesPerBlock];
    const int c = blockIdx.x, cur = level & 1;
    if (c == 0 && threadIdx.x == 0) B.ctl->unode_end[level] = B.ctl->n_unodes;
    if (c >= B.ctl->n_chunks[level] || (B.ctl->err & kErrFinite)) return;
    const BigTask t = B.big[cur][B.chunk_task[cur][c]];
    const int s = B.chunk_start[cur][c], e = min(s + kChunk, t.last);
    int b, en;
    thread_range(s, e, b, en);
    DBox bb = empty_box(), cb = empty_box();
    for (int i = b; i < en; ++i) {
        const Item it = load_item(B.items[cur] + i);
        bb = join(bb, item_box(it));
        cb = join(cb, centroid_box(it));
    }
    bb = block_union(bb, sh);
    cb = block_union(cb, sh);
    if (threadIdx.x == 0) { B.part_b[c] = bb; B.part_cb[c] = cb; }
}

// Per task (one wave): node bounds, split axis and mode.
__global__ void __launch_bounds__(64) k_task_bounds(Bufs B, int level) {
    const int ti = blockIdx.x, cur = level & 1;
    if (ti >= B.ctl->n_big[level] || (B.ctl->err & kErrFinite)) return;
    const BigTask t = B.big[cur][ti];
    const int run = (t.nchunks + 63) / 64;                          // chunks in order, a run per lane
    const int q0 = min((int)threadIdx.x * run, t.nchunks), q1 = min(q0 + run, t.nchunks);
    DBox bb = empty_box(), cb = empty_box();
    for (int q = t.chunk0 + q0; q < t.chunk0 + q1; ++q) { bb = join(bb, B.part_b[q]); cb = join(cb, B.part_cb[q]); }
    bb = wave_union(bb);
    cb = wave_union(cb);
    if (threadIdx.x != 0) return;
    const int axis = split_axis(cb);
    const float extent = cb.h[axis] - cb.l[axis];
    BigInfo inf{};
    inf.mode = extent == 0.0f ? 1 : 0;
    inf.axis = axis;
    inf.lo_axis = cb.l[axis];
    inf.extent = extent;
    inf.cb_area = area(cb);
    B.info[ti] = inf;
    UNode& u = B.unodes[t.unode];
    u.b = bb;
    u.axis = axis;
    u.set = t.set;
}

// Per chunk of a binned task: each bin's bounds (ordered) and count, by a
// thread per bin, side and run of items, then the runs in order.
constexpr int kRuns = kThreads / (2 * kBins);
__global__ void __launch_bounds__(kThreads) k_chunk_bins(Bufs B, int level) {
    __shared__ float f[6][kChunk + 4];
    __shared__ uint8_t bin[kChunk];
    __shared__ float run_box[kRuns][kBins][6];
    __shared__ int run_n[kRuns][kBins];
    const int c = blockIdx.x, cur = level & 1;
    if (c >= B.ctl->n_chunks[level] || (B.ctl->err & kErrFinite)) return;
    const int ti = B.chunk_task[cur][c];
    const BigInfo inf = B.info[ti];
    if (inf.mode != 0) return;                    // uniform per block
    const int s = B.chunk_start[cur][c], n = min(s + kChunk, B.big[cur][ti].last) - s;
    for (int i = threadIdx.x; i < n; i += kThreads) {
        const Item it = load_item(B.items[cur] + s + i);
        f[0][i] = -it.lx; f[1][i] = -it.ly; f[2][i] = -it.lz;
        f[3][i] = it.hx; f[4][i] = it.hy; f[5][i] = it.hz;
        bin[i] = (uint8_t)bin_of(it, inf.axis, inf.lo_axis, inf.extent);
    }
    __syncthreads();
    const int r = (int)threadIdx.x / (2 * kBins), j = (int)threadIdx.x % (2 * kBins);
    if (r < kRuns) {
        const int k = j >> 1, side = j & 1, len = (n + kRuns - 1) / kRuns;
        const int e = min((r + 1) * len, n);
        float x = -kInf, y = -kInf, z = -kInf;
        int m = 0;
        for (int i = min(r * len, n); i < e; ++i) {
            const bool in = bin[i] == k;
            const float a = f[3 * side][i], b = f[3 * side + 1][i], d = f[3 * side + 2][i];
            x = in ? later_max(x, a) : x;
            y = in ? later_max(y, b) : y;
            z = in ? later_max(z, d) : z;
            m += in ? 1 : 0;
        }
        float* o = &run_box[r][k][3 * side];
        o[0] = x; o[1] = y; o[2] = z;
        if (side == 0) run_n[r][k] = m;
    }
    __syncthreads();
    if (threadIdx.x < kBins * 6) {
        const int k = (int)threadIdx.x / 6, w = (int)threadIdx.x % 6;
        float v = -kInf;
        for (int q = 0; q < kRuns; ++q) v = later_max(v, run_box[q][k][w]);
        B.bin_b[(size_t)c * kBins + k].v[w] = v;
    } else if (threadIdx.x >= 128 && threadIdx.x < 128 + kBins) {
        int m = 0;
        for (int q = 0; q < kRuns; ++q) m += run_n[q][threadIdx.x - 128];
        B.bin_n[(size_t)c * kBins + (threadIdx.x - 128)] = m;
    }
}

// Per task (one block): the split, the chunks' scatter bases and the two
// children, each either a task of the next level or a small task.
__global__ void __launch_bounds__(kThreads) k_task_split(Bufs B, int level) {
    __shared__ int shn[kWavesPerBlock];
    __shared__ SplitLds sp;
    __shared__ float run_box[kRuns][kBins][6];
    __shared__ int run_n[kRuns][kBins];
    __shared__ int child_chunk0[2], child_task[2], pick[2];
    const int ti = blockIdx.x, cur = level & 1;
    if (ti >= B.ctl->n_big[level] || (B.ctl->err & kErrFinite)) return;
    const BigInfo inf = B.info[ti];
    const BigTask t = B.big[cur][ti];
    const int cnt = t.last - t.first;
    if (inf.mode == 0) {
        // the bins over all chunks: a thread per bin, side and run of chunks, then the runs in order
        const int j = (int)threadIdx.x % (2 * kBins), r = (int)threadIdx.x / (2 * kBins);
        const int k = j >> 1, side = j & 1;
        if (r < kRuns) {
            const int len = (t.nchunks + kRuns - 1) / kRuns;
            const int a = t.chunk0 + min(r * len, t.nchunks), z = t.chunk0 + min((r + 1) * len, t.nchunks);
            float v[3] = {-kInf, -kInf, -kInf};
            int n = 0;
            for (int q = a; q < z; ++q) {
                const Box6& x = B.bin_b[(size_t)q * kBins + k];
#pragma unroll
                for (int w = 0; w < 3; ++w) v[w] = later_max(v[w], x.v[3 * side + w]);
                n += B.bin_n[(size_t)q * kBins + k];
            }
#pragma unroll
            for (int w = 0; w < 3; ++w) run_box[r][k][3 * side + w] = v[w];
            if (side == 0) run_n[r][k] = n;
        }
        __syncthreads();
        if (threadIdx.x < kBins * 6) {
            const int kk = (int)threadIdx.x / 6, w = (int)threadIdx.x % 6;
            float v = -kInf;
            for (int q = 0; q < kRuns; ++q) v = later_max(v, run_box[q][kk][w]);
            sp.bin_box[kk][w] = v;
        }
        if (threadIdx.x < kBins) {
            int n = 0;
            for (int q = 0; q < kRuns; ++q) n += run_n[q][threadIdx.x];
            sp.bin_n[threadIdx.x] = n;
        }
        __syncthreads();
        if (threadIdx.x < 64) {
            int best, nl;
            sah_sweep(sp, cnt, inf.cb_area, best, nl);
            if (threadIdx.x == 0) { pick[0] = best; pick[1] = nl; }
        }
    } else if (threadIdx.x == 0) {
        pick[0] = 0;
        pick[1] = cnt / 2;                                          // equal centroids: split in the middle
    }
    __syncthreads();
    const int best = pick[0], nl = pick[1];
    const int run = (t.nchunks + kThreads - 1) / kThreads;
    const int q0 = t.chunk0 + min((int)threadIdx.x * run, t.nchunks);
    const int q1 = t.chunk0 + min(((int)threadIdx.x + 1) * run, t.nchunks);
    if (inf.mode == 0) {
        // scatter bases: lefts ascend from first, rights descend from last - 1
        int l = 0, all = 0;
        for (int q = q0; q < q1; ++q)
            for (int k = 0; k < kBins; ++k) {
                const int n = B.bin_n[(size_t)q * kBins + k];
                l += k <= best ? n : 0;
                all += n;
            }
        int lo = t.first + block_excl_scan(l, shn);
        int hi = t.last - 1 - block_excl_scan(all - l, shn);
        for (int q = q0; q < q1; ++q) {
            B.chunk_lbase[q] = lo;
            B.chunk_rbase[q] = hi;
            for (int k = 0; k < kBins; ++k) {
                const int n = B.bin_n[(size_t)q * kBins + k];
                if (k <= best) lo += n; else hi -= n;
            }
        }
    }
    if (threadIdx.x == 0) {
        B.info[ti].best = best;
        int code[2];
        for (int side = 0; side < 2; ++side) {
            const int f = side ? t.first + nl : t.first, l = side ? t.last : t.first + nl;
            child_task[side] = -1;
            code[side] = -1;
            if (l - f > B.small_max && t.depth + 1 < kMaxDepth) {
                const int nc = (l - f + kChunk - 1) / kChunk;
                const int u = atomicAdd(&B.ctl->n_unodes, 1);
                const int k = atomicAdd(&B.ctl->n_big[level + 1], 1);
                const int c0 = atomicAdd(&B.ctl->n_chunks[level + 1], nc);
                if (u >= B.unode_cap || k >= B.big_cap || c0 + nc > B.chunk_cap) {
                    atomicOr(&B.ctl->err, kErrCapacity);
                    continue;
                }
                B.big[cur ^ 1][k] = {f, l, t.depth + 1, u, t.set, c0, nc, 0};
                child_task[side] = k;
                child_chunk0[side] = c0;
                code[side] = u;
            } else if (t.depth + 1 >= kMaxDepth && l - f > kLeafMost) {
                // a leaf that its count cannot hold (and a task that k_small's
                // LDS may not): the host gives up before the subtrees are built
                atomicOr(&B.ctl->err, kErrLeaf);
            } else {
                const int k = atomicAdd(&B.ctl->n_small, 1);
                if (k >= B.small_cap) { atomicOr(&B.ctl->err, kErrCapacity); continue; }
                B.small[k] = {f, l, t.depth + 1, cur ^ 1, t.set, 0, 0, 0};
                code[side] = ~k;
            }
        }
        B.unodes[t.unode].left = code[0];
        B.unodes[t.unode].right = code[1];
    }
    __syncthreads();
    for (int side = 0; side < 2; ++side) {
        if (child_task[side] < 0) continue;
        const int f = side ? t.first + nl : t.first, l = side ? t.last : t.first + nl;
        const int nc = (l - f + kChunk - 1) / kChunk;
        for (int k = threadIdx.x; k < nc; k += kThreads) {
            B.chunk_task[cur ^ 1][child_chunk0[side] + k] = child_task[side];
            B.chunk_start[cur ^ 1][child_chunk0[side] + k] = f + k * kChunk;
        }
    }
}

// Per chunk: move the items to the next level's buffer, lefts and rights
// in order (a middle split keeps every item's position).
__global__ void __launch_bounds__(kThreads) k_scatter(Bufs B, int level) {
    __shared__ int sh[kWavesPerBlock];
    const int c = blockIdx.x, cur = level & 1;
    if (c >= B.ctl->n_chunks[level] || (B.ctl->err & kErrFinite)) return;
    const int ti = B.chunk_task[cur][c];
    const BigInfo inf = B.info[ti];
    const BigTask t = B.big[cur][ti];
    const int s = B.chunk_start[cur][c], e = min(s + kChunk, t.last);
    int b, en;
    thread_range(s, e, b, en);
    const Item* in = B.items[cur];
    Item* out = B.items[cur ^ 1];
    if (inf.mode != 0) {
        for (int i = b; i < en; ++i) store_item(out + i, load_item(in + i));
        return;
    }
    Item its[kIpt];
    bool left[kIpt];
    int nl = 0;
#pragma unroll
    for (int j = 0; j < kIpt; ++j) {
        left[j] = false;
        if (b + j < en) {
            its[j] = load_item(in + b + j);
            left[j] = bin_of(its[j], inf.axis, inf.lo_axis, inf.extent) <= inf.best;
            nl += left[j];
        }
    }
    const int nr = (en - b) - nl;
    const int pl = block_excl_scan(nl, sh);
    const int pr = block_excl_scan(nr, sh);
    int l = B.chunk_lbase[c] + pl, r = B.chunk_rbase[c] - pr;
#pragma unroll
    for (int j = 0; j < kIpt; ++j) {
        if (b + j >= en) break;
        if (left[j]) store_item(out + l++, its[j]);
        else store_item(out + r--, its[j]);
    }
}

__device__ __forceinline__ bn_bvh_node make_node(const DBox& b, int32_t word, bool leaf, int axis, int count) {
    bn_bvh_node n;
    n.pmin[0] = b.l[0]; n.pmin[1] = b.l[1]; n.pmin[2] = b.l[2];
    n.pmax[0] = b.h[0]; n.pmax[1] = b.h[1]; n.pmax[2] = b.h[2];
    n.right_or_offset = word;
    n.is_leaf = leaf ? 1 : 0;
    n.split_axis = (int8_t)axis;
    n.count = (int8_t)count;
    n.mask = 0;
    return n;
}

// One wave builds the whole subtree of a small task (Tree.Build, recursive,
// left first) into the task's node region, numbered in pre-order from 0.
//
// The task's items live in LDS; a lane holds its run of at most kPer
// consecutive ones in registers while they are moved.  Most nodes hold a
// few items, so a node's cost has to follow its item count: the bins are
// folded by 48 lanes, one per bin, side and half of the items, each walking
// the items in order (24 x 7 values through six lane-reduction steps took the
// same time for every node: the kernel ran 2.6 ms for 240,000 items, 0.50 ms
// like this, 0.26 ms for tasks of up to 128 items), and the SAH sweep runs in 22
// lanes, one per prefix and suffix.
constexpr int kPer = 4;
constexpr int kSmallMax = 64 * kPer;
static_assert(kSmallMax >= kLeafMost, "a task at the depth limit fits, whatever the option says");
constexpr int kRow = kSmallMax + 4;               // the two sides' rows start in different banks
struct SmallLds {
    float f[6][kRow];
    int id[kSmallMax];
    uint8_t bin[kSmallMax];
    SplitLds split;
    int4 frames[kMaxDepth + 2];                   // first, last (in the task), depth, parent
};
// Ordered union over the first `lanes` lanes, in lane 0; broadcast.
__device__ __forceinline__ void wave_union6(Box6& b, int lanes) {
    for (int s = 1; s < lanes; s <<= 1) {
        Box6 o;
#pragma unroll
        for (int c = 0; c < 6; ++c) o.v[c] = __shfl_down(b.v[c], s);
        join6(b, o);                              // meaningful in lanes that are multiples of 2s
    }
#pragma unroll
    for (int c = 0; c < 6; ++c) b.v[c] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(b.v[c])));
}
__device__ __forceinline__ int sreg(int v) { return __builtin_amdgcn_readfirstlane(v); }

// The best split of the binned items [0, cnt) of a node (Util/BVH.fs:183-203)
// and the number of items left of it.
__device__ __forceinline__ void small_split(SmallLds& S, int first, int cnt, float cb_area, int& best, int& n_left) {
    const int lane = threadIdx.x & 63;
    const int half = lane >= 24 ? 1 : 0, j = lane - 24 * half;
    const int k = j >> 1, side = j & 1;
    const int mid = (cnt + 1) >> 1;
    float x = -kInf, y = -kInf, z = -kInf;
    int n = 0;
    if (lane < 48) {
        const float* fx = S.f[3 * side];
        const int e = first + (half ? cnt : mid);
        for (int i = first + (half ? mid : 0); i < e; ++i) {
            const bool in = S.bin[i] == k;
            const float a = fx[i], b = fx[kRow + i], c = fx[2 * kRow + i];
            x = in ? later_max(x, a) : x;
            y = in ? later_max(y, b) : y;
            z = in ? later_max(z, c) : z;
            n += in ? 1 : 0;
        }
    }
    const float ox = __shfl(x, lane + 24), oy = __shfl(y, lane + 24), oz = __shfl(z, lane + 24);
    const int on = __shfl(n, lane + 24);
    if (lane < 24) {
        float* o = &S.split.bin_box[k][3 * side];
        o[0] = later_max(x, ox);
        o[1] = later_max(y, oy);
        o[2] = later_max(z, oz);
        S.split.bin_n[k] = n + on;
    }
    bnd::wave_sync();
    sah_sweep(S.split, cnt, cb_area, best, n_left);
}

__global__ void __launch_bounds__(kThreads) k_small(Bufs B, int n_small) {
    __shared__ SmallLds lds[kWavesPerBlock];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int ti = sreg(blockIdx.x * kWavesPerBlock + w);
    if (ti >= n_small) return;
    SmallLds& S = lds[w];
    const SmallTask task = B.small[ti];
    const int off = B.set_off[task.set];
    bn_bvh_node* region = B.region + 2 * (size_t)task.first;
    const int total = task.last - task.first;
    for (int i = lane; i < total; i += 64) {
        const Item it = load_item(B.items[task.buf] + task.first + i);
        S.f[0][i] = -it.lx; S.f[1][i] = -it.ly; S.f[2][i] = -it.lz;
        S.f[3][i] = it.hx; S.f[4][i] = it.hy; S.f[5][i] = it.hz;
        S.id[i] = it.id;
    }
    if (lane == 0) S.frames[0] = make_int4(0, total, task.depth, -1);
    bnd::wave_sync();
    int sp = 1, nodes = 0;
    while (sp > 0) {
        // nodes without items are the only way past the region's 2 * total
        if (nodes >= 2 * total) {
            if (lane == 0) atomicOr(&B.ctl->err, kErrCount);
            break;
        }
        const int4 f = S.frames[--sp];
        const int first = sreg(f.x), last = sreg(f.y), depth = sreg(f.z), parent = sreg(f.w);
        const int me = nodes++;
        if (parent >= 0 && lane == 0) region[parent].right_or_offset = me;
        const int cnt = last - first;
        // at most kPer; a node has no items where the centroids' extent is
        // infinite, which puts all of its parent's in bin 0
        const int per = max(1, (cnt + 63) >> 6);
        const int lanes = (cnt + per - 1) / per;          // lanes with items
        const int b = min(first + lane * per, last), n = min(b + per, last) - b;
        Box6 its[kPer], bb = empty6(), cb = empty6();
        int ids[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            if (j >= per) break;
            if (j < n) {
#pragma unroll
                for (int c = 0; c < 6; ++c) its[j].v[c] = S.f[c][b + j];
                ids[j] = S.id[b + j];
                join6(bb, its[j]);
                Box6 ce;                                  // the centroid 0.5 * (lo + hi), as a point
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const float m = 0.5f * (-its[j].v[c] + its[j].v[3 + c]);
                    ce.v[c] = -m;
                    ce.v[3 + c] = m;
                }
                join6(cb, ce);
            }
        }
        wave_union6(bb, lanes);
        if (cnt <= kLeaf || depth >= kMaxDepth) {
            if (cnt > kLeafMost) {
                if (lane == 0) atomicOr(&B.ctl->err, kErrLeaf);
            } else if (lane == 0) {
                region[me] = make_node(dbox(bb), task.first + first - off, true, 0, cnt);
            }
#pragma unroll
            for (int j = 0; j < kPer; ++j)
                if (j < n) B.perm[task.first + b + j] = ids[j];
            continue;
        }
        wave_union6(cb, lanes);
        const DBox cbox = dbox(cb);
        const int axis = sreg(split_axis(cbox));
        const float lo = axis == 0 ? cbox.l[0] : axis == 1 ? cbox.l[1] : cbox.l[2];
        const float extent = (axis == 0 ? cbox.h[0] : axis == 1 ? cbox.h[1] : cbox.h[2]) - lo;
        if (lane == 0) region[me] = make_node(dbox(bb), 0, false, axis, 0);
        int n_left;
        if (extent == 0.0f) {
            n_left = cnt / 2;                              // items stay where they are
        } else {
            int bin[kPer];
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                bin[j] = -1;
                if (j >= per) break;
                if (j < n) {
                    const Box6& q = its[j];
                    const float l = axis == 0 ? q.v[0] : axis == 1 ? q.v[1] : q.v[2];
                    const float h = axis == 0 ? q.v[3] : axis == 1 ? q.v[4] : q.v[5];
                    const float v = (12.0f * (0.5f * (-l + h) - lo)) / extent;
                    bin[j] = min(kBins - 1, (int)v);       // findBinIndex, as bin_of
                    S.bin[b + j] = (uint8_t)bin[j];
                }
            }
            bnd::wave_sync();
            int best;
            small_split(S, first, cnt, area(cbox), best, n_left);
            // partition: lefts in order from first, rights in order from last - 1 down
            int before = 0;                                // lefts before this lane's items
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                if (j >= per) break;
                before += (int)bnd::mbcnt(__ballot(j < n && bin[j] <= best));
            }
            int l = first + before, r = last - 1 - (b - first - before);
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                if (j >= per) break;
                if (j < n) {
                    const int to = bin[j] <= best ? l++ : r--;
#pragma unroll
                    for (int c = 0; c < 6; ++c) S.f[c][to] = its[j].v[c];
                    S.id[to] = ids[j];
                }
            }
        }
        const int mid = first + n_left;
        if (lane == 0) {
            S.frames[sp] = make_int4(mid, last, depth + 1, me);
            S.frames[sp + 1] = make_int4(first, mid, depth + 1, -1);
        }
        sp += 2;
        bnd::wave_sync();
    }
    if (lane == 0) B.small_size[ti] = nodes;
}

// Pre-order numbering (one block): subtree sizes from the deepest level up,
// the sets' places in the output, then indices from the roots down.
constexpr int kNumThreads = 1024;
__global__ void __launch_bounds__(kNumThreads) k_number(Bufs B, int levels) {
    __shared__ int sh[kNumThreads / 64], carry;
    auto size_of = [&](int code) { return code < 0 ? B.small_size[~code] : B.usize[code]; };
    auto place = [&](int code, int idx) { if (code < 0) B.small_base[~code] = idx; else B.udfs[code] = idx; };
    for (int d = levels - 1; d >= 0; --d) {
        const int u0 = d > 0 ? B.ctl->unode_end[d - 1] : 0, u1 = B.ctl->unode_end[d];
        for (int u = u0 + threadIdx.x; u < u1; u += kNumThreads)
            B.usize[u] = 1 + size_of(B.unodes[u].left) + size_of(B.unodes[u].right);
        __syncthreads();
    }
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < B.n_sets; base += kNumThreads) {
        const int s = base + threadIdx.x;
        int n = 0;
        if (s < B.n_sets) {
            n = size_of(B.root[s]);
            if (n <= 0 || n > 2 * (B.set_off[s + 1] - B.set_off[s])) {
                atomicOr(&B.ctl->err, kErrCount);
                n = 0;
            }
            place(B.root[s], 0);
            B.set_nodes[s] = n;
        }
        int v = n;                                        // inclusive scan over the block
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(v, o);
            if (lane >= o) v += y;
        }
        if (lane == 63) sh[w] = v;
        __syncthreads();
        int before = carry;
        for (int k = 0; k < w; ++k) before += sh[k];
        if (s < B.n_sets) B.set_base[s] = before + v - n;
        __syncthreads();
        if (threadIdx.x == kNumThreads - 1) carry = before + v;
        __syncthreads();
    }
    for (int d = 0; d < levels; ++d) {
        const int u0 = d > 0 ? B.ctl->unode_end[d - 1] : 0, u1 = B.ctl->unode_end[d];
        for (int u = u0 + threadIdx.x; u < u1; u += kNumThreads) {
            const UNode n = B.unodes[u];
            const int idx = B.udfs[u], r = idx + 1 + size_of(n.left);
            place(n.left, idx + 1);
            place(n.right, r);
            B.uright[u] = r;
        }
        __syncthreads();
    }
}

__global__ void k_write_upper(Bufs B, int n_unodes, bn_bvh_node* out) {
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= n_unodes) return;
    const UNode n = B.unodes[u];
    out[(size_t)B.set_base[n.set] + B.udfs[u]] = make_node(n.b, B.uright[u], false, n.axis, 0);
}

// Copy each region to its place in its set's node array; right-child indices
// move with the region's base.
__global__ void __launch_bounds__(kThreads) k_write_regions(Bufs B, int n_small, bn_bvh_node* out) {
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int ti = blockIdx.x * kWavesPerBlock + w;
    if (ti >= n_small) return;
    const SmallTask t = B.small[ti];
    const int base = B.small_base[ti], n = B.small_size[ti];
    const bn_bvh_node* src = B.region + 2 * (size_t)t.first;
    bn_bvh_node* dst = out + (size_t)B.set_base[t.set] + base;
    for (int k = lane; k < n; k += 64) {
        bn_bvh_node x = src[k];
        if (!x.is_leaf) x.right_or_offset += base;
        dst[k] = x;
    }
}

}  // namespace bvhg

namespace bnx {

using namespace bvhg;
using bnh::Error;

namespace {
// Page-locked staging memory of the context, grown on demand.
void* pinned(Ctx* c, size_t bytes) {
    if (c->g_pinned_bytes < bytes) {
        if (c->g_pinned) (void)hipHostFree(c->g_pinned);
        c->g_pinned = nullptr;
        c->g_pinned_bytes = 0;
        hip_check(hipHostMalloc(&c->g_pinned, bytes, hipHostMallocDefault), "hipHostMalloc");
        c->g_pinned_bytes = bytes;
    }
    return c->g_pinned;
}
size_t up16(size_t n) { return (n + 15) / 16 * 16; }
}  // namespace

GpuBvh bvh_build_gpu(Ctx* c, const std::vector<const float*>& sets, const std::vector<int>& counts) {
    const int S = (int)sets.size();
    GpuBvh g;
    g.counts = counts;
    if (S == 0) return g;
    std::vector<int> off(S + 1, 0);
    for (int s = 0; s < S; ++s) {
        if (counts[s] <= 0) throw Error(BN_E_INVALID, "BVH build of an empty item set");
        if ((int64_t)off[s] + counts[s] > (1 << 28)) throw Error(BN_E_CAPACITY, "GPU BVH build: more than 2^28 items");
        off[s + 1] = off[s] + counts[s];
    }
    const int N = off[S];
    const int small = std::min(c->bvh_small, kSmallMax);
    const size_t item_bytes = (size_t)N * sizeof(Item);
    const int big_cap = N / small + S + 1;
    const int unode_cap = kMaxDepth * big_cap;
    const int small_cap = (int)std::min((int64_t)N + S, 2 * (int64_t)unode_cap + S) + 1;
    const int chunk_cap = 2 * (N / kChunk + big_cap) + 1;
    // the level-0 tasks
    std::vector<BigTask> big0;
    std::vector<SmallTask> small0;
    std::vector<int> root(S), ctask, cstart;
    int largest = 0;
    for (int s = 0; s < S; ++s) {
        largest = std::max(largest, counts[s]);
        if (counts[s] > small) {
            const int u = (int)big0.size();
            const int nc = (counts[s] + kChunk - 1) / kChunk;
            big0.push_back({off[s], off[s + 1], 0, u, s, (int)ctask.size(), nc, 0});
            for (int k = 0; k < nc; ++k) { ctask.push_back(u); cstart.push_back(off[s] + k * kChunk); }
            root[s] = u;
        } else {
            root[s] = ~(int)small0.size();
            small0.push_back({off[s], off[s + 1], 0, 0, s, 0, 0, 0});
        }
    }
    // device memory (grow-only buffers of the context)
    c->g_items.ensure(2 * std::max(item_bytes, (size_t)N * sizeof(bn_bvh_node)));   // A | B, then the nodes
    c->g_region.ensure(2 * (size_t)N * sizeof(bn_bvh_node));                        // the bounds, then the regions
    c->g_perm.ensure((size_t)N * 4);
    c->g_rsize.ensure((size_t)small_cap * 4 * 2);         // region sizes, region bases (by small task)
    c->g_big.ensure(2 * (size_t)big_cap * sizeof(BigTask));
    c->g_info.ensure((size_t)big_cap * sizeof(BigInfo));
    c->g_small.ensure((size_t)small_cap * sizeof(SmallTask));
    c->g_chunks.ensure(4 * (size_t)chunk_cap * 4);
    c->g_part.ensure((size_t)chunk_cap * (2 * sizeof(DBox) + kBins * sizeof(Box6)) + (size_t)chunk_cap * (kBins + 2) * 4);
    c->g_unodes.ensure((size_t)unode_cap * (sizeof(UNode) + 3 * 4));
    // what the host sets up, in one block: counters, set offsets, roots, the
    // level-0 tasks; then what it reads back: the sets' nodes and places
    const size_t o_off = up16(sizeof(Ctl)), o_root = o_off + up16(((size_t)S + 1) * 4);
    const size_t o_nodes = o_root + up16((size_t)S * 4), o_base = o_nodes + up16((size_t)S * 4);
    c->g_misc.ensure(o_base + (size_t)S * 4);
    hipStream_t st = c->stream;
    char* items_base = (char*)c->g_items.p;
    char* misc = (char*)c->g_misc.p;
    Bufs B{};
    B.items[0] = (Item*)items_base;
    B.items[1] = (Item*)(items_base + item_bytes);
    B.info = (BigInfo*)c->g_info.p;
    B.small = (SmallTask*)c->g_small.p;
    for (int k = 0; k < 2; ++k) {
        B.big[k] = (BigTask*)c->g_big.p + (size_t)k * big_cap;
        B.chunk_task[k] = (int*)c->g_chunks.p + (size_t)(2 * k) * chunk_cap;
        B.chunk_start[k] = (int*)c->g_chunks.p + (size_t)(2 * k + 1) * chunk_cap;
    }
    B.part_b = (DBox*)c->g_part.p;
    B.part_cb = B.part_b + chunk_cap;
    B.bin_b = (Box6*)(B.part_cb + chunk_cap);
    B.bin_n = (int*)(B.bin_b + (size_t)chunk_cap * kBins);
    B.chunk_lbase = B.bin_n + (size_t)chunk_cap * kBins;
    B.chunk_rbase = B.chunk_lbase + chunk_cap;
    B.unodes = (UNode*)c->g_unodes.p;
    B.udfs = (int*)(B.unodes + unode_cap);
    B.uright = B.udfs + unode_cap;
    B.usize = B.uright + unode_cap;
    B.region = (bn_bvh_node*)c->g_region.p;
    B.small_size = (int*)c->g_rsize.p;
    B.small_base = B.small_size + small_cap;
    B.perm = (int32_t*)c->g_perm.p;
    B.ctl = (Ctl*)misc;
    B.set_off = (const int*)(misc + o_off);
    B.root = (const int*)(misc + o_root);
    B.set_nodes = (int*)(misc + o_nodes);
    B.set_base = (int*)(misc + o_base);
    B.n_sets = S; B.n_items = N; B.small_max = small;
    B.big_cap = big_cap; B.small_cap = small_cap; B.unode_cap = unode_cap; B.chunk_cap = chunk_cap;

    // The bounds go up a piece at a time through page-locked memory, each
    // piece copied in while the one before is on its way.
    const size_t bounds_bytes = (size_t)N * 24;
    char* host = (char*)pinned(c, std::max(bounds_bytes, o_base + (size_t)S * 4) + o_nodes);
    char* head = host;                                     // the block above, then the bounds
    char* stage = host + o_nodes;
    Ctl ctl{};
    ctl.n_small = (int)small0.size();
    ctl.n_unodes = (int)big0.size();
    ctl.n_big[0] = (int)big0.size();
    ctl.n_chunks[0] = (int)ctask.size();
    std::memcpy(head, &ctl, sizeof(ctl));
    std::memcpy(head + o_off, off.data(), ((size_t)S + 1) * 4);
    std::memcpy(head + o_root, root.data(), (size_t)S * 4);
    hip_check(hipMemcpyAsync(misc, head, o_nodes, hipMemcpyHostToDevice, st), "bvh ctl");
    if (!big0.empty()) {
        hip_check(hipMemcpyAsync(B.big[0], big0.data(), big0.size() * sizeof(BigTask), hipMemcpyHostToDevice, st), "bvh tasks");
        hip_check(hipMemcpyAsync(B.chunk_task[0], ctask.data(), ctask.size() * 4, hipMemcpyHostToDevice, st), "bvh chunks");
        hip_check(hipMemcpyAsync(B.chunk_start[0], cstart.data(), cstart.size() * 4, hipMemcpyHostToDevice, st), "bvh chunks");
    }
    if (!small0.empty())
        hip_check(hipMemcpyAsync(B.small, small0.data(), small0.size() * sizeof(SmallTask), hipMemcpyHostToDevice, st),
                  "bvh small tasks");
    constexpr size_t kUp = (size_t)1 << 20;
    size_t sent = 0, filled = 0;
    for (int s = 0; s < S; ++s)
        for (size_t a = 0, n = (size_t)counts[s] * 24; a < n;) {
            const size_t m = std::min(n - a, kUp - (filled - sent));
            std::memcpy(stage + filled, (const char*)sets[s] + a, m);
            a += m;
            filled += m;
            if (filled - sent == kUp || filled == bounds_bytes) {
                hip_check(hipMemcpyAsync((char*)c->g_region.p + sent, stage + sent, filled - sent, hipMemcpyHostToDevice, st),
                          "bvh bounds");
                sent = filled;
            }
        }
    k_items<<<std::min((N + kThreads - 1) / kThreads, 8 * c->n_cu), kThreads, 0, st>>>(B, (const float*)c->g_region.p);
    hip_check(hipGetLastError(), "bvh items launch");
    auto read_ctl = [&] {
        hip_check(hipMemcpyAsync(&ctl, B.ctl, sizeof(Ctl), hipMemcpyDeviceToHost, st), "bvh ctl");
        hip_check(hipStreamSynchronize(st), "bvh level");
        if (ctl.err & kErrFinite) throw Error(BN_E_INVALID, "GPU BVH build needs finite bounds (bn_bvh_build takes any)");
        if (ctl.err & kErrCapacity) throw Error(BN_E_CAPACITY, "GPU BVH build: task capacity exceeded");
        if (ctl.err & kErrLeaf) throw Error(BN_E_CAPACITY, "BVH leaf larger than the int8 count field");
    };
    // Levels: as many as an even tree has and three more, then four at a time
    // while there are tasks left.  A level holds at most twice the tasks of
    // the one before, and a chunk more than its items fill per task.
    int level = 0;
    if (big0.empty()) read_ctl();
    for (int todo = 3 + (int)std::ceil(std::log2(std::max(2.0, (double)largest / small)));
         !big0.empty() && (level == 0 || ctl.n_big[level] > 0); todo = 4) {
        for (int k = 0; k < todo && level < kMaxDepth; ++k, ++level) {
            const int64_t tasks = std::min<int64_t>((int64_t)big0.size() << std::min(level, 30), big_cap);
            const int grid = (int)std::min<int64_t>(N / kChunk + tasks + 1, chunk_cap);
            k_chunk_bounds<<<grid, kThreads, 0, st>>>(B, level);
            k_task_bounds<<<(int)tasks, 64, 0, st>>>(B, level);
            k_chunk_bins<<<grid, kThreads, 0, st>>>(B, level);
            k_task_split<<<(int)tasks, kThreads, 0, st>>>(B, level);
            k_scatter<<<grid, kThreads, 0, st>>>(B, level);
        }
        hip_check(hipGetLastError(), "bvh level launch");
        read_ctl();
        if (level >= kMaxDepth && ctl.n_big[kMaxDepth] > 0)
            throw Error(BN_E_INVALID, "GPU BVH build: deeper than the depth limit");
    }
    const int n_small = ctl.n_small, n_unodes = ctl.n_unodes;
    bn_bvh_node* out = (bn_bvh_node*)items_base;                // the item buffers are done with after k_small
    if (n_small > 0) k_small<<<(n_small + kWavesPerBlock - 1) / kWavesPerBlock, kThreads, 0, st>>>(B, n_small);
    k_number<<<1, kNumThreads, 0, st>>>(B, level);
    if (n_unodes) k_write_upper<<<(n_unodes + 255) / 256, 256, 0, st>>>(B, n_unodes, out);
    if (n_small > 0) k_write_regions<<<(n_small + kWavesPerBlock - 1) / kWavesPerBlock, kThreads, 0, st>>>(B, n_small, out);
    hip_check(hipGetLastError(), "bvh flatten launch");
    hip_check(hipMemcpyAsync(host, misc, o_base, hipMemcpyDeviceToHost, st), "bvh sizes");
    hip_check(hipStreamSynchronize(st), "bvh subtrees");
    std::memcpy(&ctl, host, sizeof(ctl));
    if (ctl.err & kErrLeaf) throw Error(BN_E_CAPACITY, "BVH leaf larger than the int8 count field");
    if (ctl.err & kErrCount) throw Error(BN_E_DEVICE, "GPU BVH build: inconsistent node count");
    g.n_nodes.assign((const int*)(host + o_nodes), (const int*)(host + o_nodes) + S);
    g.nodes = out;
    g.perm = B.perm;
    return g;
}

void bvh_fetch(Ctx* c, const GpuBvh& g, const std::vector<bn_bvh_node*>& nodes, const std::vector<int32_t*>& perms) {
    std::vector<HostCopy::Part> pn, pp;
    for (size_t s = 0; s < g.counts.size(); ++s) {
        pn.push_back({nodes[s], (size_t)g.n_nodes[s] * sizeof(bn_bvh_node)});
        pp.push_back({perms[s], (size_t)g.counts[s] * 4});
    }
    c->host_copy.download(g.nodes, pn, c->stream);
    c->host_copy.download(g.perm, pp, c->stream);
}

}  // namespace bnx
