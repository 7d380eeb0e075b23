// traverse.hpp -- persistent, lane-refilling BVH traversal for gfx950.
//
// Semantics are those of BVHAggregate.Intersect (Extensions/Aggregate/BVH.fs:
// 11-58) over PrimitiveInstance.Intersect (Base/Primitive.fs:111-129) and
// MeshPrimitive.Intersect (Extensions/Primitive/Mesh.fs:188-242): the same
// items are visited in the same order with the same current t, so hit
// (instance, triangle, t) and the traversal counters are identical to the
// reference's.  The schedule differs: in every loop iteration a lane processes
// at most one item of each sort that it comes to,
//
//    instance of a TLAS leaf, then TLAS or BLAS node, then triangle of a leaf
//
// (the counting traversal: one item), and lanes whose ray finished are refilled
// from the work queue in batches (one atomic per wave).
#pragma once
#include "device.hpp"
#include "wave.hpp"

namespace bnd {

// Slab test with hardware min/max.  Equal in outcome to the exact test when
// the ray origin and 1/d are finite and the box is finite: then no t0/t1 is
// NaN, and min/max results can differ only in the sign of a zero, which the
// final comparison does not see.
__device__ __forceinline__ bool slab_fast(V3 lo, V3 hi, V3 o, V3 inv, float t) {
    const float t0x = (lo.x - o.x) * inv.x, t1x = (hi.x - o.x) * inv.x;
    const float t0y = (lo.y - o.y) * inv.y, t1y = (hi.y - o.y) * inv.y;
    const float t0z = (lo.z - o.z) * inv.z, t1z = (hi.z - o.z) * inv.z;
    const float tmin = fmaxf(fmaxf(1e-3f, fminf(t0x, t1x)), fmaxf(fminf(t0y, t1y), fminf(t0z, t1z)));
    const float tmax = fminf(fminf(t, fmaxf(t0x, t1x)), fminf(fmaxf(t0y, t1y), fmaxf(t0z, t1z)));
    return tmin <= tmax;
}
// Three-way min / max in one instruction.  Used only on the finite path, where
// they agree with the compare-and-select Vector3.Min/Max up to the sign of a
// zero, which no slab comparison can see.
__device__ __forceinline__ float min3f(float a, float b, float c) {
    float r;
    asm volatile("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float max3f(float a, float b, float c) {
    float r;
    asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ bool finite3(V3 v) {
    return __builtin_isfinite(v.x) && __builtin_isfinite(v.y) && __builtin_isfinite(v.z);
}

enum : int { kItemNone = 0, kItemTNode = 1, kItemBNode = 2, kItemTri = 3, kItemInst = 4 };
constexpr uint32_t kNoNode = 0xffffffffu;
constexpr uint32_t kNeedTest = 0x80000000u;   // node whose box is still to be tested
constexpr uint32_t kNodeMask = 0x7fffffffu;

// The geometry a lane traverses (per lane, so a batched launch can mix scenes).
struct TraceScene {
    const float4* tlas;
    const float4* blas;
    const float* tris;
    const DevInst* insts;
    const FlatScene* flat;
    const NodeRec *trecs, *recs;
    int n_insts, n_tlas;
    __device__ __forceinline__ void set(const DevScene& S) {
        tlas = S.tlas; blas = S.blas; tris = S.tris; insts = S.insts;
        flat = S.flat; trecs = S.trecs; recs = S.recs; n_insts = S.n_insts; n_tlas = S.n_tlas;
    }
};

// Read through the scalar cache: the same address in all lanes, memory that no
// kernel writes.
template <typename T>
using Scalar = const T __attribute__((address_space(4)));
template <typename T>
__device__ __forceinline__ Scalar<T>* scalar(const T* p) { return (Scalar<T>*)(uintptr_t)p; }

// FLAT: for scenes of at most kFlatMax instances (DevScene::flat).  A ray meets
// all instance bounds when it starts, and the ones it hits become the bits of
// `left`, in the order in which the reference's TLAS walk reaches them (each
// octant of ray directions has one order, known on the host; an any-hit query
// takes them as they are).  An instance is tested again when it is taken, with
// the t of that moment, as the reference does; a TLAS node contains the bounds
// below it, so a ray that meets an instance has met the nodes above it.
// The start costs about 27 instructions an instance, which all lanes of a
// refill share; the walk was the larger part of the steps: with 9 instances 18
// of 38 busy lanes of a wave step stood at a TLAS node or at an instance they
// then missed, and the traversal is bound by instruction issue.  Config-1 frame
// 109 -> 89 ms, 1024x768 frame of analytic spheres 11.7 -> 8.8 ms.
template <int K, int MODE, int PITCH = 256>
struct Traversal {
    static constexpr bool FLAT = MODE == kList, RECS = MODE != kNodes;
    TraceScene G;
    // world ray and the ray of the current space (world, or object inside a BLAS)
    V3 wo, wd, winv;
    V3 co, cd, cinv;
    float t;
    int hit_inst, hit_prim;   // hit_prim: triangle of the pool, or the branch of a sphere
    bool exact;          // take the NaN-exact slab path
    // traversal position
    LaneStack<K, PITCH> st;
    uint32_t nxt;        // node to take before the stack (kNoNode: none); kNeedTest: box not tested yet
    int blas_base;       // stack depth at BLAS entry, -1 in the TLAS
    int tl_cur, tl_end;  // instances left in the current TLAS leaf
    uint32_t left;       // FLAT: places of the instances still to be taken
    int bl_cur, bl_end;  // triangles left in the current BLAS leaf
    int cur_inst;
    const uint8_t* order;   // FLAT: FlatScene::order (a copy in LDS, but in batches)

    // The primitive of the hit as the reference numbers it: a mesh's triangle.
    __device__ __forceinline__ int prim_of(int4 info) const { return hit_prim - (info.x >= 0 ? info.y : 0); }

    // Half of a node.  With records the pools have less than 4 GiB: an offset of
    // 32 bits to a base in scalar registers takes no 64-bit address arithmetic.
    // (With indices into the pools in the nodes, so that a lane holds no BLAS
    // root or first triangle, and the order in LDS: config-1 frame 89 -> 84 ms.)
    __device__ __forceinline__ static float4 node_half(const float4* nodes, int i, int half) {
        if (RECS) return *(const float4*)((const char*)nodes + ((uint32_t)i * 32u + 16u * half));
        return nodes[node_at(i, half)];
    }
    __device__ __forceinline__ static Tri load_tri32(const float* tris, int i) {
        const float* p = (const float*)((const char*)tris + ((uint32_t)i * 32u + (uint32_t)i * 4u));
        return {{p[0], p[1], p[2]}, {p[3], p[4], p[5]}, {p[6], p[7], p[8]}};
    }

    // A new ray over the geometry already in G (set once per launch for a
    // single scene, per ray in a batch).
    __device__ __forceinline__ void start(const Ray& r, float tmax, bool exact_scene) {
        wo = r.o; wd = r.d;
        winv = {1.0f / r.d.x, 1.0f / r.d.y, 1.0f / r.d.z};
        co = wo; cd = wd; cinv = winv;
        t = tmax;
        hit_inst = -1; hit_prim = -1;
        exact = exact_scene || !finite3(wo) || !finite3(winv);
        st.sp = 0;
        nxt = kNeedTest;                 // the TLAS root
        blas_base = -1;
        tl_cur = tl_end = 0;
        bl_cur = bl_end = 0;
        cur_inst = 0;
        if (FLAT) { left = 0; nxt = kNoNode; }
    }

    // No traversal at all (placeholder rays, NaN t max).
    __device__ __forceinline__ void empty() {
        st.sp = 0;
        nxt = kNoNode;
        tl_cur = tl_end = 0;
        if (FLAT) left = 0;
    }
    // FLAT: the instances the ray of start() meets.
    __device__ __forceinline__ uint32_t octant_shift() const {
        return (wd.x > 0.0f ? 8u : 0u) + (wd.y > 0.0f ? 16u : 0u) + (wd.z > 0.0f ? 32u : 0u);
    }
    // LANE: each lane has a scene of its own (a batch; 48 thumbnails of four
    // scenes 6.2 -> 5.45 ms).
    template <bool LANE>
    __device__ __forceinline__ void take_instances(bool any) {
        if (LANE) take_instances_of(G.flat, any);
        else take_instances_of(scalar(G.flat), any);
        if (exact) take_instances_exact(any);
    }
    template <typename P>
    __device__ __forceinline__ void take_instances_of(P F, bool any) {
        const uint32_t oct = octant_shift();
        for (int i = 0; i < G.n_insts; ++i) {
            const auto& f = F->inst[i];
            const uint64_t place = (uint64_t)f.place[1] << 32 | f.place[0];
            const bool h = slab_fast(mk(f.lo[0], f.lo[1], f.lo[2]), mk(f.hi[0], f.hi[1], f.hi[2]), wo, winv, t);
            const uint32_t bit = 1u << (any ? (uint32_t)i : (uint32_t)(place >> oct) & 31u);
            left |= h ? bit : 0u;
        }
    }
    // A wave whose lanes all hold the same ray: a lane for each place (1024
    // Metropolis chains of a wave each: 52.9 -> 41.5 ms).
    __device__ __forceinline__ void take_instances_wave(bool any) {
        const int p = (int)lane_id();
        bool h = false;
        if (p < G.n_insts) {
            const FlatScene::Inst& f = G.flat->inst[any ? p : (int)order[(octant_shift() << 2) + p]];
            h = slab_fast(mk(f.lo[0], f.lo[1], f.lo[2]), mk(f.hi[0], f.hi[1], f.hi[2]), wo, winv, t);
        }
        left = (uint32_t)__ballot(h);
        if (exact) take_instances_exact(any);
    }
    // A ray whose slab test can see a NaN meets what the walk lets through:
    // the node tests have NaNs of their own.
    __device__ __forceinline__ void take_instances_exact(bool any) {
        const uint32_t oct = octant_shift() >> 3;
        left = 0;
        for (int i = 0; i < G.n_tlas;) {
            const NodeView n = load_node(G.tlas, i);
            if (!slab(n.lo, n.hi, wo, winv, t)) {
                i = G.flat->after[i];
                continue;
            }
            if (n.leaf)
                for (int k = 0; k < G.n_insts; ++k) {
                    const int inst = any ? k : (int)order[oct * kFlatMax + k];
                    if (inst >= n.word && inst < n.word + n.count) left |= 1u << k;
                }
            ++i;
        }
    }
    // The fast traversal tests a root when it is reached: the TLAS root when
    // the ray starts, a BLAS root when its instance is entered.  A failing
    // root leaves nothing to do, a leaf root hands over its items at once,
    // and an interior root is expanded next without a second test.  (The
    // counting traversal leaves the TLAS root to step(), which tests and
    // counts it.)
    __device__ __forceinline__ void take_tlas_root() { take_root(G.tlas, 0, false); }
    __device__ __forceinline__ void take_root(const float4* nodes, int root, bool in_blas) {
        const float4 a = node_half(nodes, root, 0), b = node_half(nodes, root, 1);
        nxt = kNoNode;
        if (!box(mk(a.x, a.y, a.z), mk(a.w, b.x, b.y))) return;
        const uint32_t f = __float_as_uint(b.w);
        if (f & 0xff) {
            const int cnt = (int)(int8_t)((f >> 16) & 0xff);
            const int w = __float_as_int(b.z);
            if (in_blas) { bl_cur = w; bl_end = w + cnt; }
            else { tl_cur = w; tl_end = w + cnt; }
        } else {
            nxt = (uint32_t)root;
        }
    }
    // An idle lane: no item left anywhere, so a step does nothing.
    __device__ __forceinline__ void clear() {
        st.sp = 0;
        nxt = kNoNode;
        blas_base = -1;
        tl_cur = tl_end = 0;
        bl_cur = bl_end = 0;
        if (FLAT) left = 0;
    }

    // The fast test is evaluated first, in the block that computes its
    // products, so its min/max need no operand canonicalisation; the exact
    // test replaces it on the rare non-finite rays.
    __device__ __forceinline__ bool box(V3 lo, V3 hi) const {
        bool r = slab_fast(lo, hi, co, cinv, t);
        if (exact) r = slab(lo, hi, co, cinv, t);
        return r;
    }
    // A triangle's bounding-box pre-test (Mesh.fs:204).
    __device__ __forceinline__ bool box_tri(const Tri& tr) const {
        if (!exact)
            return slab_fast(mk(min3f(tr.p0.x, tr.p1.x, tr.p2.x), min3f(tr.p0.y, tr.p1.y, tr.p2.y),
                                min3f(tr.p0.z, tr.p1.z, tr.p2.z)),
                             mk(max3f(tr.p0.x, tr.p1.x, tr.p2.x), max3f(tr.p0.y, tr.p1.y, tr.p2.y),
                                max3f(tr.p0.z, tr.p1.z, tr.p2.z)),
                             co, cinv, t);
        return slab(vmin(vmin(tr.p0, tr.p1), tr.p2), vmax(vmax(tr.p0, tr.p1), tr.p2), co, cinv, t);
    }

    // One item.  Returns false when the traversal has finished (no items left,
    // or an any-hit query found its hit); `found` reports an any-hit.
    // The reference's visit sequence item by item (every popped node is
    // tested); the counting kernels use it, so the counters are the
    // reference's.
    template <bool ANY, bool COUNT>
    __device__ __forceinline__ bool step(TraceCount& cnt, bool& found) {
        // leave a finished BLAS
        if (blas_base >= 0 && bl_cur >= bl_end && nxt == kNoNode && st.sp == blas_base) {
            blas_base = -1;
            co = wo; cd = wd; cinv = winv;
        }
        int kind;
        int idx = 0;
        if (blas_base >= 0) {
            if (bl_cur < bl_end) { kind = kItemTri; idx = bl_cur++; }
            else if (nxt != kNoNode) { kind = kItemBNode; idx = (int)(nxt & kNodeMask); nxt = kNoNode; }
            else { kind = kItemBNode; idx = (int)st.pop(); }
        } else if (tl_cur < tl_end) {
            kind = kItemInst; idx = tl_cur++;
        } else if (nxt != kNoNode) {
            kind = kItemTNode; idx = (int)(nxt & kNodeMask); nxt = kNoNode;
        } else if (st.sp > 0) {
            kind = kItemTNode; idx = (int)st.pop();
        } else {
            return false;
        }
        V3 lo, hi;
        Tri tr;
        NodeView n;
        if (kind == kItemTri) {
            tr = load_tri(G.tris, idx);
            lo = vmin(vmin(tr.p0, tr.p1), tr.p2);
            hi = vmax(vmax(tr.p0, tr.p1), tr.p2);
            if (COUNT) cnt.tris++;
        } else if (kind == kItemInst) {
            const float4 a = G.insts[idx].lo, b = G.insts[idx].hi;
            lo = xyz(a); hi = xyz(b);
        } else {
            n = load_node(kind == kItemTNode ? G.tlas : G.blas, idx);
            lo = n.lo; hi = n.hi;
            if (COUNT) cnt.nodes++;
        }
        if (!box(lo, hi)) return true;
        if (kind == kItemTri) {
            float tt;
            if (tri_hit(tr, co, cd, t, tt)) {
                if (ANY) { found = true; return false; }
                t = tt;
                hit_inst = cur_inst;
                hit_prim = idx;
            }
        } else if (kind == kItemInst) {
            if (COUNT) cnt.insts++;
            const DevInst& I = G.insts[idx];
            const Xf w2o = I.w2o;
            const V3 oo = xf_point(w2o, wo), od = xf_dir(w2o, wd);
            const int4 info = I.info;
            if (info.x < 0) {
                float tt;
                int br;
                if (sphere_hit(I.lo.w, oo, od, t, tt, br)) {
                    if (ANY) { found = true; return false; }
                    t = tt;
                    hit_inst = idx;
                    hit_prim = br;
                }
            } else {
                co = oo; cd = od;
                cinv = {1.0f / od.x, 1.0f / od.y, 1.0f / od.z};
                exact = exact || !finite3(co) || !finite3(cinv);
                cur_inst = idx;
                blas_base = st.sp;
                nxt = (uint32_t)info.x | kNeedTest;   // the BLAS root
            }
        } else if (n.leaf) {
            if (kind == kItemTNode) { tl_cur = n.word; tl_end = n.word + n.count; }
            else { bl_cur = n.word; bl_end = bl_cur + n.count; }
        } else if (comp(cd, n.axis) > 0.0f) {
            st.push((uint32_t)n.word); st.push((uint32_t)(idx + 1));
        } else {
            st.push((uint32_t)(idx + 1)); st.push((uint32_t)n.word);
        }
        return true;
    }

    // The fast traversal (do_tri / do_inst / do_node): the same hits with
    // fewer iterations.  An interior node tests both children when it is
    // expanded, with the t of that moment, and only the children that pass
    // are kept.  A kept child is not re-tested when it is taken later with a
    // smaller t.  That changes no hit:
    // if its box would fail then, the box lies beyond the current t, and so do
    // the boxes of every triangle and instance below it, which are still
    // tested (Mesh.fs:204,231 pre-test every triangle; instances have their
    // world bounds); a box that passes with the current t passed with the
    // larger one too.  Every triangle the reference tests is tested, in the
    // same order, so ties resolve alike.
    // One triangle of the current BLAS leaf.
    __device__ __forceinline__ void do_tri(bool any, bool& found) {
        const int idx = bl_cur++;
        const Tri tr = RECS ? load_tri32(G.tris, idx) : load_tri(G.tris, idx);
        if (box_tri(tr)) {
            float tt;
            if (tri_hit(tr, co, cd, t, tt)) {
                if (any) found = true;
                else { t = tt; hit_inst = cur_inst; hit_prim = idx; }
            }
        }
    }

    // One instance of the current TLAS leaf (FLAT: the next of the ray's): a
    // sphere is intersected, a mesh BLAS is entered.
    __device__ __forceinline__ void do_inst(bool any, bool& found) {
        int idx;
        if (FLAT) {
            idx = __ffs((int)left) - 1;
            left &= left - 1;
            if (!any) idx = order[(octant_shift() << 2) + idx];
        } else {
            idx = tl_cur++;
        }
        const DevInst& I = G.insts[idx];
        bool in;
        if (FLAT) {
            in = any || slab_fast(xyz(I.lo), xyz(I.hi), wo, winv, t);   // t as in take_instances
            if (exact) in = slab(xyz(I.lo), xyz(I.hi), wo, winv, t);
        } else {
            in = box(xyz(I.lo), xyz(I.hi));
        }
        if (!in) return;
        const int4 info = I.info;
        const int4 aux = I.aux;
        if (!FLAT && info.x >= 0) blas_base = st.sp;
        if (info.x >= 0) cur_inst = idx;
        // Identity world-to-object map on a finite ray: Transform gives o but
        // for the signs of zeros and d unchanged (no component of d is 0 when
        // 1/d is finite), so the object ray's 1/d is the world one.  The sign
        // of a zero coordinate changes no test: it is subtracted from box and
        // triangle coordinates, and no comparison sees the sign of a zero
        // difference.  The instance's bounds are its root's, so the root is
        // not tested again, and one that is a leaf is not even read (frame of
        // instances 17.1 -> 16.8 ms, 2^20 Metropolis chains 123 -> 120).
        const bool same = info.x >= 0 && aux.x != 0 && !exact;
        if (same) {
            co = wo;
            cd = wd;
            cinv = winv;
            if (RECS) {
                take_ref((uint32_t)aux.w);
            } else {
                if (aux.y >= 0) { bl_cur = aux.y; bl_end = aux.z; }
                nxt = aux.y >= 0 ? kNoNode : (uint32_t)info.x;
            }
        }
        if (opaque(same)) return;
        const Xf w2o = I.w2o;
        const V3 oo = xf_point(w2o, wo), od = xf_dir(w2o, wd);
        if (info.x < 0) {
            float tt;
            int br;
            if (sphere_hit(I.lo.w, oo, od, t, tt, br)) {
                if (any) found = true;
                else { t = tt; hit_inst = idx; hit_prim = br; }
            }
        }
        if (opaque(info.x) >= 0) {
            // its root is tested at once, as the reference pops and tests it
            // first (Mesh.fs:217-242); a lane whose root fails leaves the
            // BLAS in its next step
            co = oo; cd = od;
            cinv = {1.0f / od.x, 1.0f / od.y, 1.0f / od.z};
            exact = exact || !finite3(co) || !finite3(cinv);
            if (RECS) {
                const float4 a = I.rlo, b = I.rhi;
                if (box(xyz(a), xyz(b))) take_ref((uint32_t)aux.w);
            } else {
                take_root(G.blas, info.x, true);
            }
        }
    }

    // Expand the next node (RECS: record): a leaf sets its item range; an interior node
    // tests both children with the current t and keeps those that pass (the
    // near one in `nxt`, the far one on the stack, near first as in
    // Extensions/Aggregate/BVH.fs:47-56 and Mesh.fs:233-240).  A child taken
    // next that is a leaf hands over its items at once (same items, same
    // order), without being popped first.
    __device__ __forceinline__ void do_node(bool any) {
        uint32_t e = nxt;
        if (e == kNoNode) e = st.pop();
        nxt = kNoNode;
        if (RECS) {
            do_rec(e, any);
            return;
        }
        const bool in_blas = blas_base >= 0;
        const float4* base = in_blas ? G.blas : G.tlas;
        const int node = (int)e;
        const float4 b = node_half(base, node, 1);
        int word = __float_as_int(b.z);
        uint32_t f = __float_as_uint(b.w);
        bool leaf = (f & 0xff) != 0;
        if (!leaf) {
            const int axis = (int)(int8_t)((f >> 8) & 0xff);
            const int l = node + 1, r = word;
            const float4 la = node_half(base, l, 0), lb = node_half(base, l, 1);
            const float4 ra = node_half(base, r, 0), rb = node_half(base, r, 1);
            const bool hl = box(mk(la.x, la.y, la.z), mk(la.w, lb.x, lb.y));
            const bool hr = box(mk(ra.x, ra.y, ra.z), mk(ra.w, rb.x, rb.y));
            // An any-hit query finds the same in any order, and t does not
            // change on the way: left first saves it the axis (preview 1.02
            // -> 0.97 ms, adjoint step 44.9 -> 43.0).
            const bool left_near = any || comp(cd, axis) > 0.0f;
            if (hl && hr) st.push((uint32_t)(left_near ? r : l));
            const bool take_left = hl && (left_near || !hr);
            f = __float_as_uint(take_left ? lb.w : rb.w);
            word = __float_as_int(take_left ? lb.z : rb.z);
            const bool any_child = hl || hr;
            leaf = any_child && (f & 0xff) != 0;
            if (any_child && !leaf) nxt = (uint32_t)(take_left ? l : r);
        }
        if (leaf) {
            const int end = word + (int)(int8_t)((f >> 16) & 0xff);
            if (in_blas) { bl_cur = word; bl_end = end; }
            if (!in_blas) { tl_cur = word; tl_end = end; }
        }
    }

    // RECS: the reference of a record's child, or of a root (nxt == kNoNode).
    // (Adjoint step over 8000 instances: 43.3 ms by nodes, 41.7 by records.)
    __device__ __forceinline__ void take_ref(uint32_t e) {
        const int first = (int)(e & ((1u << kRefBits) - 1)), end = first + (int)((e & ~kRefLeaf) >> kRefBits);
        const bool in_blas = FLAT || blas_base >= 0;
        if ((e & kRefLeaf) && in_blas) { bl_cur = first; bl_end = end; }
        if ((e & kRefLeaf) && !in_blas) { tl_cur = first; tl_end = end; }
        nxt = e & kRefLeaf ? kNoNode : e;
    }
    __device__ __forceinline__ void do_rec(uint32_t e, bool any) {
        if (!(e & kRefLeaf)) {
            const NodeRec* base = FLAT || blas_base >= 0 ? G.recs : G.trecs;
            const NodeRec& n = *(const NodeRec*)((const char*)base + e * (uint32_t)sizeof(NodeRec));
            const float4 la = n.llo, lb = n.lhi, ra = n.rlo, rb = n.rhi;
            const bool hl = box(mk(la.x, la.y, la.z), mk(la.w, lb.x, lb.y));
            const bool hr = box(mk(ra.x, ra.y, ra.z), mk(ra.w, rb.x, rb.y));
            const bool left_near = any || comp(cd, __float_as_int(lb.w)) > 0.0f;
            const uint32_t l = __float_as_uint(lb.z), r = __float_as_uint(rb.z);
            if (hl && hr) st.push(left_near ? r : l);
            e = hl && (left_near || !hr) ? l : r;
            if (!hl && !hr) e = kRefLeaf;            // a leaf of no triangles
        }
        take_ref(e);
    }

    // One step of the fast traversal: an instance, then a node, then a
    // triangle, each if it is what the lane has next at that moment, so one
    // step can take a lane from an instance through its root to the first
    // triangle of a leaf (each lane's items in its own order).  Returns false
    // when the traversal has finished or an any-hit query (`any`, per lane)
    // found its hit.
    //
    // The three run one behind the other, each updating the lane's state in
    // place under the mask of its lanes.  As branches of one choice they cost
    // two copies of the state: the compiler lets the branches write a second
    // set of registers, which lanes of the other branches fill by moves (14
    // for each branch and 18 at the end of a step, of about 330 instructions).
    // Config-1 frame 82.0 -> 77.1 ms, preview 1.18 -> 1.03, adjoint step
    // 51.6 -> 45.6 ms; 64 VGPRs hold both kinds of scene.
    __device__ __forceinline__ bool step_fast(bool any, bool& found) {
        if (!FLAT) {
            // leave a finished BLAS; selects, so that the ray's registers are
            // updated in place
            const bool leave = blas_base >= 0 && bl_cur >= bl_end && nxt == kNoNode && st.sp == blas_base;
            blas_base = leave ? -1 : blas_base;
            co = sel(leave, wo, co);
            cd = sel(leave, wd, cd);
            cinv = sel(leave, winv, cinv);
        }
        if (FLAT ? left != 0 && nothing_in_blas() : blas_base < 0 && tl_cur < tl_end) do_inst(any, found);
        if (wants_node()) do_node(any);
        if (bl_cur < bl_end) do_tri(any, found);
        if (FLAT) return !found && (left != 0 || !nothing_in_blas());
        return !found && (tl_cur < tl_end || !nothing_in_blas());
    }
    __device__ __forceinline__ bool wants_node() const {
        if (FLAT) return bl_cur >= bl_end && (nxt != kNoNode || st.sp > 0);
        return bl_cur >= bl_end && (blas_base >= 0 || tl_cur >= tl_end) &&
               (nxt != kNoNode || st.sp > (blas_base >= 0 ? blas_base : 0));
    }
    // The any-hit query of a ray that all lanes of the wave hold (kList, after
    // start() and take_instances_wave()).  It finds the same in any order, so
    // the lanes take up to 64 of the open nodes at a time: a ray needs about
    // as many steps as a BLAS has levels, not as many as it visits nodes.
    // The open references are a stack of `cap` words in LDS; a step takes m of
    // them and puts back at most 2 m, and only one at a time (a depth-first
    // walk, which adds one a level) when fewer than 64 + 64 would stay free.
    // 300 mutations of 1024 Metropolis chains: 39.8 -> 35.4 ms.
    __device__ __forceinline__ bool any_hit_wave(uint32_t* open, int cap) {
        const int lane = (int)lane_id();
        bool found = false;
        while (left != 0 && !found) {
            bl_cur = bl_end = 0;
            nxt = kNoNode;
            do_inst(true, found);
            if (found) break;
            // the triangles of a BLAS of one leaf
            for (int k = bl_cur + lane; k < bl_end; k += 64) found = found || hits(k);
            if (nxt != kNoNode) {
                int n = 1;
                if (lane == 0) open[0] = nxt;
                wave_sync();
                while (n > 0 && __ballot(found) == 0) {
                    const int m = min(min(n, 64), max(1, cap - 128 - n));
                    n -= m;
                    uint32_t l = 0, r = 0;
                    bool hl = false, hr = false;
                    if (lane < m) {
                        const uint32_t e = open[n + lane];
                        if (e & kRefLeaf) {
                            const int first = (int)(e & ((1u << kRefBits) - 1));
                            const int end = first + (int)((e & ~kRefLeaf) >> kRefBits);
                            for (int k = first; k < end; ++k) found = found || hits(k);
                        } else {
                            const NodeRec& rec = *(const NodeRec*)((const char*)G.recs + e * (uint32_t)sizeof(NodeRec));
                            const float4 la = rec.llo, lb = rec.lhi, ra = rec.rlo, rb = rec.rhi;
                            hl = box(mk(la.x, la.y, la.z), mk(la.w, lb.x, lb.y));
                            hr = box(mk(ra.x, ra.y, ra.z), mk(ra.w, rb.x, rb.y));
                            l = __float_as_uint(lb.z);
                            r = __float_as_uint(rb.z);
                        }
                    }
                    const uint64_t ml = __ballot(hl), mr = __ballot(hr);
                    wave_sync();
                    if (hl) open[n + (int)mbcnt(ml)] = l;
                    n += __popcll(ml);
                    if (hr) open[n + (int)mbcnt(mr)] = r;
                    n += __popcll(mr);
                    wave_sync();
                }
            }
            found = __ballot(found) != 0;
        }
        clear();
        return found;
    }
    __device__ __forceinline__ bool hits(int triangle) const {
        const Tri tr = load_tri32(G.tris, triangle);
        float tt;
        return box_tri(tr) && tri_hit(tr, co, cd, t, tt);
    }
    // FLAT: also no BLAS is being traversed; otherwise the TLAS stack is empty as well.
    __device__ __forceinline__ bool nothing_in_blas() const {
        return bl_cur >= bl_end && nxt == kNoNode && st.sp == 0;
    }
};

}  // namespace bnd
