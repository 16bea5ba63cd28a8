// Device traversal routines shared by the ray-query kernels and the
// wavefront renderer's extension kernel.
//
// Two engines answer SceneAcceleration::hit (core/scene.rs:182-185):
//
//  * wide  — SAH 8-wide BVH with 8-bit outward-rounded child boxes, one ray
//            per lane, a short LDS stack, nearest-child-first order and t_max
//            shrinking.  Box tests are conservative (padded boxes, a relative
//            slack on the slab exit, a relative slack on the cull distance), so
//            every triangle the reference could return is reached.  Equal-t
//            hits go to the smaller prim id (see below).  The winner is
//            then confirmed to be a triangle the reference reaches: its
//            top-level ancestors must pass the exact reference slab test, and
//            so must its mesh-tree ancestors — taken as passed when the hit
//            point lies strictly inside the eps-expanded triangle box by a
//            margin that dominates the slab test's rounding, walked exactly
//            otherwise.  Winners the reference does not reach and stack
//            overflows go to the exact engine.
//  * exact — the flattened reference trees walked exactly as BvhNode::hit
//            (core/bvh.rs:132-181): both children, unshrunk t_max, no box test
//            at leaves, brute force for meshes of <= 4 triangles
//            (core/mesh.rs:125-138), with the same slab arithmetic
//            (util/aabb.rs:86-148).
//
// Ties.  merge_optionals (bvh.rs:164-181) compares Option<(HitRecord, usize)>
// tuples, and HitRecord orders by t alone (ray.rs:52-62), so on equal t the
// smaller handle wins: the smaller surface index at the top level
// (scene.rs:182-185), then the smaller triangle index inside the mesh
// (mesh.rs:269-279; the brute-force loop of mesh.rs:125-138 keeps the earlier
// triangle, the same rule).  Prim ids are numbered surface by surface in
// triangle order, so both engines keep the lexicographic minimum of (t, prim).
//
// Instances (template flag INST, scenes with vr_instance surfaces; no
// counterpart in the reference): an instance is one record of the top-level
// wide BVH holding its world box (kInstanceMarker in p2.x).  A ray that meets
// one pushes an "enter" entry at the box's entry distance; popping it pushes an
// "exit" entry, maps the ray into the instance's object space (t is unchanged:
// the direction is mapped, not renormalised) and walks the shared object-space
// BVH of its mesh; popping the exit entry restores the world ray.  Hits inside
// an instance carry the instance's prim base and need no confirmation.
//
// Watertight mode (template flag WT, engine VR_ENGINE_WATERTIGHT): the same
// traversal with the watertight ray/triangle test of vrmath.h in place of
// Moller-Trumbore and no reference semantics: every candidate the
// conservative boxes reach counts (no ancestor confirmation), and the exact
// fallback walks the median-split trees with slab tests that never reject a
// ray crossing the box.  For the extended estimator only.
#pragma once
#include "internal.h"

namespace vr {

struct HitOut {
    float t, u, v;
    uint32_t prim;  // 0xFFFFFFFF: miss
};

// The scene, for code that rarely runs in a kernel whose first argument starts
// with a SceneView (TraceArgs): read through a pointer the compiler cannot see
// through, so that it loads what the code needs there and then.  Through the
// argument itself it keeps all of it in scalar registers across the traversal
// loop, spills them and reads them back, lane by lane, in every step.
VR_HD const SceneView& cold_scene(const SceneView& sv) {
#ifdef __HIP_DEVICE_COMPILE__
    auto p = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const SceneView*)p;
#else
    return sv;
#endif
}

constexpr float kSlabSlack = 1.0f + 1.0f / 131072.0f;  // 2^-17 relative on the slab exit
constexpr float kCullSlack = 1.0f + 1.0f / 65536.0f;   // 2^-16 relative on t_best
constexpr float kRobustRel = 1.0f / 1048576.0f;        // 2^-20 interior margin


// Geometry of a triangle record: two 16-byte loads + one 4-byte load, all
// float.  The integer words (prim = 9, flags = 11) are read with their own
// loads, only when a hit needs them.
VR_HD void load_tri_geom(const TriRec* tris, uint32_t slot, vf3& p0, vf3& p1, vf3& p2) {
    const f32x4* q = (const f32x4*)(tris + slot);
    f32x4 a = q[0], b = q[1];
    float c = ((const float*)(tris + slot))[8];
    p0 = mk3(a.x, a.y, a.z);
    p1 = mk3(a.w, b.x, b.y);
    p2 = mk3(b.z, b.w, c);
}
VR_HD uint32_t tri_word(const TriRec* tris, uint32_t slot, int w) { return ((const uint32_t*)(tris + slot))[w]; }

// The ray (o, d) in an instance's object space: o' = M^-1 o + c', d' = M^-1 d
// (not renormalised, so a hit's t is the world t), f32, the same operation
// order in every engine.
VR_HD void instance_ray(const InstanceDev& x, vf3 o, vf3 d, vf3& oo, vf3& dd) {
    const float* m = x.inv;
    oo = mk3(((m[0] * o.x + m[1] * o.y) + m[2] * o.z) + m[3], ((m[4] * o.x + m[5] * o.y) + m[6] * o.z) + m[7],
             ((m[8] * o.x + m[9] * o.y) + m[10] * o.z) + m[11]);
    dd = mk3((m[0] * d.x + m[1] * d.y) + m[2] * d.z, (m[4] * d.x + m[5] * d.y) + m[6] * d.z,
             (m[8] * d.x + m[9] * d.y) + m[10] * d.z);
}

// Exact membership of a triangle in the reference's candidate set within its
// mesh: BvhNode::hit (core/bvh.rs:132-181) descends into a child only after
// the parent's box passes the slab test, and tests leaves without a box, so
// the triangle is reached iff every inner ancestor of its leaf passes
// AABB::hit with the unshrunk t_max.  Walks leaf parent -> mesh root with the
// reference's own slab arithmetic, so the answer is the reference's.
VR_HD bool mesh_ancestors_pass(const SceneView& sv, vf3 o, vf3 d, float tmin, uint32_t prim) {
    int32_t nd = sv.prim_anc[prim];
    while (nd >= 0) {
        const RefNode& n = sv.ref_nodes[nd];
        int32_t up = sv.ref_parent[nd];
        Box3 b{mk3(n.lo[0], n.lo[1], n.lo[2]), mk3(n.hi[0], n.hi[1], n.hi[2])};
        if (!ref_slab_hit(b, o, d, tmin, kInf)) return false;
        nd = up;
    }
    return true;
}

// Confirms that the reference would consider this hit (see header comment).
VR_HD bool confirm_winner(const SceneView& sv, vf3 o, vf3 d, float tmin, float t, vf3 p0, vf3 p1,
                                               vf3 p2, uint32_t flags, uint32_t prim) {
    uint32_t surf = flags >> 1;
    if (sv.num_surfaces > 1) {
        SurfaceInfo si = sv.surfaces[surf];
        for (uint32_t k = 0; k < si.path_len; ++k) {
            const RefNode& nd = sv.top_nodes[sv.top_path[si.path_off + k]];
            Box3 b{mk3(nd.lo[0], nd.lo[1], nd.lo[2]), mk3(nd.hi[0], nd.hi[1], nd.hi[2])};
            if (!ref_slab_hit(b, o, d, tmin, kInf)) return false;
        }
    }
    if (flags & 1u) {
        // fast path: a hit point inside the eps-expanded triangle box by a
        // margin that dominates the slab test's rounding passes every
        // ancestor box; otherwise walk the ancestors exactly
        vf3 P = o + d * t;  // Ray::at (ray.rs:19-21)
        Box3 bb = tri_box_eps(p0, p1, p2);
        bool inside = true;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            float pa = comp(P, a);
            float delta = kRobustRel * (t + fabsf(pa) + fabsf(comp(o, a)));
            inside = inside && pa - comp(bb.lo, a) > delta && comp(bb.hi, a) - pa > delta;
        }
        if (!inside) return mesh_ancestors_pass(sv, o, d, tmin, prim);
    }
    return true;
}


// ---- analytic surfaces -------------------------------------------------------
// AnalyticSurface::hit with t_max = inf, as SceneAcceleration::hit passes it:
// Sphere::hit (voidray_common/src/surfaces.rs:46-78) and GroundPlane::hit
// (surfaces.rs:88-104), same f32 operations.  Out: t and the hit record's uv.
// A ray lying exactly in a ground plane (t = 0/0) counts as a miss.
VR_HD bool analytic_hit(const AnalyticDev& a, vf3 o, vf3 d, float tmin, float& t, float& u, float& v) {
    if (a.kind == VR_ANALYTIC_SPHERE) {
        const vf3 oc = o - mk3(a.c[0], a.c[1], a.c[2]);
        const float aa = mag2(d);
        const float half_b = dot3(oc, d);
        const float c = mag2(oc) - a.r * a.r;
        const float disc = half_b * half_b - aa * c;
        if (disc < 0.0f) return false;
        const float sqrtd = sqrtf(disc);
        float root = (-half_b - sqrtd) / aa;
        if (root < tmin || kInf < root) {
            root = (-half_b + sqrtd) / aa;
            if (root < tmin || kInf < root) return false;
        }
        t = root;
        u = v = 0.0f;
        return true;
    }
    const float tt = (a.h - o.y) / d.y;
    if (tt <= tmin || tt >= kInf || tt != tt) return false;
    const vf3 p = o + d * tt;  // Ray::at
    t = tt;
    u = p.x;
    v = p.z;
    return true;
}

// Every top-level ancestor of `surf` passes the reference slab test.
VR_HD bool top_path_pass(const SceneView& sv, uint32_t surf, vf3 o, vf3 d, float tmin) {
    const SurfaceInfo& si = sv.surfaces[surf];
    for (uint32_t k = 0; k < si.path_len; ++k) {
        const RefNode& nd = sv.top_nodes[sv.top_path[si.path_off + k]];
        Box3 b{mk3(nd.lo[0], nd.lo[1], nd.lo[2]), mk3(nd.hi[0], nd.hi[1], nd.hi[2])};
        if (!ref_slab_hit(b, o, d, tmin, kInf)) return false;
    }
    return true;
}

// Closest analytic surface the reference reaches (lexicographic min of (t,
// prim), like the triangles); with `first_below` set, the first one found
// with t < first_below.  Returns its index or -1.  WT: every analytic
// surface counts (no top-level reach test).
template <bool WT = false>
VR_HD int analytic_best(const SceneView& sv, vf3 o, vf3 d, float tmin, float first_below, float& bt, uint32_t& bprim,
                        float& bu, float& bv) {
    int best = -1;
    for (uint32_t k = 0; k < sv.num_analytic; ++k) {
        const AnalyticDev& a = sv.analytic[k];
        float t, u, v;
        if (!analytic_hit(a, o, d, tmin, t, u, v)) continue;
        if (best >= 0 && !(t < bt || (t == bt && a.prim < bprim))) continue;
        if (!WT && !top_path_pass(sv, a.surface, o, d, tmin)) continue;
        best = (int)k;
        bt = t;
        bprim = a.prim;
        bu = u;
        bv = v;
        if (t < first_below) break;
    }
    return best;
}

constexpr uint32_t kAnalyticSlot = 0x40000000u;  // best_slot of an analytic winner (triangle slots < 2^27)

// ---- wide engine as a resumable per-lane state machine ----------------------
// A ray holds the node it visits next and a triangle group (the records of
// the hit leaves of one wide node); a step visits a node (wide_node_step) or
// tests one record (wide_tri_step).  A node's nearest hit inner child is
// visited next; the others go on the stack together as one 8-byte entry: the
// node's first child, the mask of the hit children and a lower bound of their
// entry distances, so a pop skips the group when all of it lies beyond the
// best hit.  One entry per level at most.  The stack's first LDS_STACK entries
// live in LDS (strided by `stride`), deeper ones in a per-lane global region
// (`spill`, strided by `spill_stride`, `spill_cap` entries).
struct WideState {
    vf3 o, d;  // the ray as the current BVH sees it (object space inside an instance)
    WTRay wt;  // watertight mode: the ray's shear (unused otherwise)
    float idx, idy, idz;
    float tbest, bu, bv;
    uint32_t best_prim, best_slot;
    uint32_t cur;  // node to visit next, kNoNode: the stack decides
    // triangle group: first record, the positions (QNode::leaf_bits) of the
    // records to test and of the node's records
    uint32_t tg_base, tg_mask, tg_all;
    int sp;
    // 0 or 1.  As words they live in vector registers; as bools the compiler
    // keeps each as a lane mask in scalar registers, which the persistent
    // kernel runs out of (spilled masks cost readlanes in every node step).
    uint32_t unconfirmed, found;
    // INST only: the instance being walked (kNoInstance: none), its prim
    // base and triangle determinant threshold, the instance of the best hit
    // (the world ray is the caller's)
    uint32_t inst, inst_base, best_inst;
    float inst_eps;
};
constexpr uint32_t kNoInstance = 0xFFFFFFFFu;
// First words of instance stack entries (INST): bit 30 set.  Node indices
// stay below 2^29 (the scene build checks it).
constexpr uint32_t kInstEntry = 0x40000000u;            // | instance index: enter
constexpr uint32_t kInstExit = kInstEntry | 0x3FFFFFFFu;  // leave the current instance
// Group entries: x = first child | kDescend, y = bits 16..31 of the bound's
// float bits (rounded down) | hit children by slot.
constexpr uint32_t kDescend = 0x80000000u;  // the far slots come first (the ray runs against the node's axis)
constexpr uint32_t kNoNode = 0xFFFFFFFFu;

// On the device the stack's LDS part is addressed through an LDS pointer: with
// a generic one the compiler merges the two stores of a push (and the two
// loads of a pop) into one flat access through a selected pointer, which
// takes the slower path and waits for both memories.
#ifdef __HIP_DEVICE_COMPILE__
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
#else
typedef u32x2 lds_u32x2;
#endif
struct WideStack {
    lds_u32x2* lds;
    int stride;
    u32x2* spill;
    int spill_stride, spill_cap;
};

enum : int { kStepContinue = 0, kStepDone = 1, kStepFallback = 2 };

template <bool WT = false>
VR_HD void wide_set_ray(WideState& st, vf3 o, vf3 d) {
    const float kTiny = 1e-20f;
    st.o = o;
    st.d = d;
    if (WT) st.wt = wt_prepare(d);
    st.idx = 1.0f / (fabsf(d.x) > kTiny ? d.x : copysignf(kTiny, d.x));
    st.idy = 1.0f / (fabsf(d.y) > kTiny ? d.y : copysignf(kTiny, d.y));
    st.idz = 1.0f / (fabsf(d.z) > kTiny ? d.z : copysignf(kTiny, d.z));
}

template <bool WT = false>
VR_HD void wide_init(WideState& st, vf3 o, vf3 d, bool nonempty) {
    wide_set_ray<WT>(st, o, d);
    st.inst = kNoInstance;
    st.inst_base = 0;
    st.best_inst = kNoInstance;
    st.tbest = kInf;
    st.bu = st.bv = 0.f;
    st.best_prim = 0xFFFFFFFFu;
    st.best_slot = 0xFFFFFFFFu;
    st.cur = nonempty ? 0u : kNoNode;
    st.tg_base = 0;
    st.tg_mask = 0;
    st.tg_all = 0;
    st.sp = 0;
    st.unconfirmed = false;
    st.found = false;
}

// Analytic surfaces are few and not in the wide BVH: each ray tests them all
// up front, and the best one seeds the closest hit (so the triangle walk culls
// against it and ties resolve by prim id as usual).  An any-hit ray that hits
// one below tmax_any is finished.
template <bool ANY, bool WT = false>
VR_HD void wide_seed_analytic(const SceneView& sv, WideState& st, float tmin, float tmax_any) {
    float t = kInf, u = 0.f, v = 0.f;
    uint32_t prim = 0xFFFFFFFFu;
    const int k = analytic_best<WT>(sv, st.o, st.d, tmin, ANY ? tmax_any : -kInf, t, prim, u, v);
    if (k < 0) return;
    if (ANY) {
        if (!(t < tmax_any)) return;
        st.found = true;
        st.cur = kNoNode;
    }
    st.tbest = t;
    st.best_prim = prim;
    st.best_slot = kAnalyticSlot | (uint32_t)k;
    st.bu = u;
    st.bv = v;
}

template <int LDS_STACK>
VR_HD bool wide_push(WideState& st, const WideStack& ws, u32x2 e) {
    if (st.sp < LDS_STACK) {
        ws.lds[st.sp * ws.stride] = e;
    } else {
        if (st.sp - LDS_STACK >= ws.spill_cap) return false;
        ws.spill[(st.sp - LDS_STACK) * ws.spill_stride] = e;
    }
    ++st.sp;
    return true;
}

// The stack's top entry (sp > 0), which stays there.
template <int LDS_STACK>
VR_HD u32x2 wide_top(const WideState& st, const WideStack& ws) {
    const int i = st.sp - 1;
    if (i >= LDS_STACK) return ws.spill[(i - LDS_STACK) * ws.spill_stride];
    return ws.lds[i * ws.stride];
}
template <int LDS_STACK>
VR_HD void wide_set_top(const WideState& st, const WideStack& ws, u32x2 e) {
    const int i = st.sp - 1;
    if (i >= LDS_STACK) ws.spill[(i - LDS_STACK) * ws.spill_stride] = e;
    else ws.lds[i * ws.stride] = e;
}

// Tests one record of the triangle group (tg_mask != 0).  Returns
// kStepContinue, kStepDone when an any-hit query has its confirmed hit, or
// kStepFallback when an instance entry finds the stack exhausted (INST).
template <int LDS_STACK, bool ANY, bool WT = false, bool INST = false>
VR_HD int wide_tri_step(const SceneView& sv, WideState& st, const WideStack& ws, float tmin, float tmax_any) {
    const vf3 o = st.o, d = st.d;
    const bool in_inst = INST && st.inst != kNoInstance;
    const uint32_t bit = st.tg_mask & (0u - st.tg_mask);
    const uint32_t entry = st.tg_base + (uint32_t)__builtin_popcount(st.tg_all & (bit - 1u));
    st.tg_mask ^= bit;
    // the record's index (best_slot keeps it, not the leaf entry)
    const uint32_t slot = sv.tri_ref ? sv.tri_ref[entry] : entry;
    vf3 p0, p1, p2;
    load_tri_geom(sv.tris, slot, p0, p1, p2);
    if (INST && f2u(p2.x) == kInstanceMarker) {
        // an instance: its world box is [p0, p1]; entered when its stack entry is popped
        const float tcull = ANY ? tmax_any : st.tbest * kCullSlack;
        const float ax = (p0.x - o.x) * st.idx, bx = (p1.x - o.x) * st.idx;
        const float ay = (p0.y - o.y) * st.idy, by = (p1.y - o.y) * st.idy;
        const float az = (p0.z - o.z) * st.idz, bz = (p1.z - o.z) * st.idz;
        const float tnear = fmaxf(fmaxf(fminf(ax, bx), fminf(ay, by)), fmaxf(fminf(az, bz), tmin));
        const float tfar = fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fminf(fmaxf(az, bz), tcull));
        if (tnear <= tfar * kSlabSlack && !wide_push<LDS_STACK>(st, ws, u32x2{kInstEntry | f2u(p2.y), f2u(tnear)}))
            return kStepFallback;
        return kStepContinue;
    }
    MTResult r;
    if (WT ? !wt_hit(st.wt, o, p0, p1, p2, tmin, r) : !mt_hit(o, d, p0, p1, p2, tmin, r, in_inst ? st.inst_eps : -1.0f))
        return kStepContinue;
    if (ANY) {
        if (!(r.t < tmax_any)) return kStepContinue;
        if (WT || in_inst ||
            confirm_winner(cold_scene(sv), o, d, tmin, r.t, p0, p1, p2, tri_word(sv.tris, slot, 11),
                           tri_word(sv.tris, slot, 9))) {
            st.found = true;
            st.tbest = r.t;
            st.best_slot = slot;
            st.bu = r.u;
            st.bv = r.v;
            if (INST) {
                st.best_inst = st.inst;
                st.best_prim = st.inst_base + tri_word(sv.tris, slot, 9);
            }
            return kStepDone;
        }
        st.unconfirmed = true;
        return kStepContinue;
    }
    if (r.t > st.tbest) return kStepContinue;
    const uint32_t prim = (in_inst ? st.inst_base : 0u) + tri_word(sv.tris, slot, 9);
    if (r.t < st.tbest || prim < st.best_prim) {
        st.tbest = r.t;
        st.best_prim = prim;
        st.best_slot = slot;
        st.bu = r.u;
        st.bv = r.v;
        if (INST) st.best_inst = st.inst;
    }
    return kStepContinue;
}

// Pops of instance entries (INST).  Enter (code kInstEntry | k, popped in
// world space): push the exit entry, map the ray into object space
// (instance_ray) and continue at the mesh BVH's root; returns kStepFallback
// when the exit entry does not fit on the stack.  Exit (kInstExit): the caller
// hands back the world ray (the state does not keep it, to save registers).
template <int LDS_STACK, bool WT = false>
VR_HD int wide_instance_enter(const SceneView& sv, WideState& st, const WideStack& ws, uint32_t code, float tmin) {
    const uint32_t k = code & ~kInstEntry;
    if (!wide_push<LDS_STACK>(st, ws, u32x2{kInstExit, 0u})) return kStepFallback;
    const InstanceDev& x = cold_scene(sv).instances[k];
    vf3 oo, dd;
    instance_ray(x, st.o, st.d, oo, dd);
    wide_set_ray<WT>(st, oo, dd);
    st.inst = k;
    st.inst_base = x.prim_base;
    st.inst_eps = tmin * x.det_inv;
    st.cur = x.blas_root;
    return kStepContinue;
}

template <bool WT = false>
VR_HD void wide_instance_exit(WideState& st, vf3 world_o, vf3 world_d) {
    wide_set_ray<WT>(st, world_o, world_d);
    st.inst = kNoInstance;
}

VR_HD uint32_t min_u(uint32_t a, uint32_t b) { return a < b ? a : b; }
// Median of three.
VR_HD uint32_t med3_u(uint32_t a, uint32_t b, uint32_t c) {
#ifdef __HIP_DEVICE_COMPILE__
    uint32_t r;
    asm("v_med3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
#else
    const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
    return c < lo ? lo : c > hi ? hi : c;
#endif
}

// Tests the 8 child boxes of node `node`.  The hit leaves' records become the
// triangle group, the nearest hit inner child (any hit: the first along the
// node's axis) st.cur, and the other hit inner children are pushed.  Returns
// kStepContinue, or kStepFallback when the stack is exhausted.
template <int LDS_STACK, bool ANY>
VR_HD int wide_node(const SceneView& sv, WideState& st, const WideStack& ws, uint32_t node, float tmin,
                    float tmax_any) {
    const u32x4* qp = (const u32x4*)(sv.qnodes + node);
    const u32x4 w0 = qp[0], w1 = qp[1], w2 = qp[2], w3 = qp[3], w4 = qp[4];
    const uint32_t e = w0.w;
    const float sx = u2f((e & 0xFFu) << 23) * st.idx;
    const float sy = u2f(((e >> 8) & 0xFFu) << 23) * st.idy;
    const float sz = u2f(((e >> 16) & 0xFFu) << 23) * st.idz;
    const uint32_t num_inner = e >> 24;
    const float bx = (u2f(w0.x) - st.o.x) * st.idx;
    const float by = (u2f(w0.y) - st.o.y) * st.idy;
    const float bz = (u2f(w0.z) - st.o.z) * st.idz;
    // Near and far planes chosen once per node from the ray's direction signs
    // (four children's bytes at once): with s > 0, fma(lo, s, b) <=
    // fma(hi, s, b), so this equals taking min/max per child and axis.
    const bool negx = st.idx < 0.f, negy = st.idy < 0.f, negz = st.idz < 0.f;
    const float tcull = ANY ? tmax_any : st.tbest * kCullSlack;
    uint32_t hits = 0;
    // the two smallest (entry distance, slot) keys of the hit inner children:
    // the distance's float bits with the slot in the lowest three
    uint32_t m1 = 0xFFFFFFFFu, m2 = 0xFFFFFFFFu;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        // words: lo x, y, z at 0..5, hi x, y, z at 6..11 of w2, w3, w4
        const uint32_t lx = h ? w2.y : w2.x, ly = h ? w2.w : w2.z, lz = h ? w3.y : w3.x;
        const uint32_t hx = h ? w3.w : w3.z, hy = h ? w4.y : w4.x, hz = h ? w4.w : w4.z;
        const uint32_t qnx = negx ? hx : lx, qfx = negx ? lx : hx;
        const uint32_t qny = negy ? hy : ly, qfy = negy ? ly : hy;
        const uint32_t qnz = negz ? hz : lz, qfz = negz ? lz : hz;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int s = 4 * h + c;
            const float nx = fmaf((float)((qnx >> (8 * c)) & 0xFFu), sx, bx), fx = fmaf((float)((qfx >> (8 * c)) & 0xFFu), sx, bx);
            const float ny = fmaf((float)((qny >> (8 * c)) & 0xFFu), sy, by), fy = fmaf((float)((qfy >> (8 * c)) & 0xFFu), sy, by);
            const float nz = fmaf((float)((qnz >> (8 * c)) & 0xFFu), sz, bz), fz = fmaf((float)((qfz >> (8 * c)) & 0xFFu), sz, bz);
            const float tnear = fmaxf(fmaxf(nx, ny), fmaxf(nz, tmin));
            const float tfar = fminf(fminf(fx, fy), fminf(fz, tcull));
            const bool hit = tnear <= tfar * kSlabSlack;
            hits |= hit ? 1u << s : 0u;
            if (!ANY) {
                const uint32_t key = hit && (uint32_t)s < num_inner ? (f2u(tnear) & ~7u) | (uint32_t)s : 0xFFFFFFFFu;
                m2 = med3_u(m1, m2, key);
                m1 = min_u(m1, key);
            }
        }
    }
    // empty slots (lo 255, hi 0) can pass within the slack, or where a
    // direction component is zero: only the node's own slots count
    const uint32_t inner = (1u << num_inner) - 1u;
    uint32_t leaves = hits & ~inner;
    leaves = (leaves | (leaves << 8)) & 0x00F00Fu;
    leaves = (leaves | (leaves << 4)) & 0x0C30C3u;
    leaves = (leaves | (leaves << 2)) & 0x249249u;
    st.tg_all = w1.z & 0xFFFFFFu;
    st.tg_mask = ((leaves << 3) - leaves) & st.tg_all;
    st.tg_base = w1.y;
    hits &= inner;
    st.cur = kNoNode;
    if (hits) {
        const uint32_t axis = (w1.z >> 24) & 3u;
        const bool neg = axis == 0u ? negx : axis == 1u ? negy : negz;
        uint32_t slot;
        if (ANY) slot = neg ? 31u - (uint32_t)__builtin_clz(hits) : (uint32_t)__builtin_ctz(hits);
        else slot = m1 & 7u;
        st.cur = w1.x + slot;
        hits &= ~(1u << slot);
        if (hits) {
            // (a negative t_min, whose keys do not order as integers, makes
            // the bound a NaN: nothing is skipped)
            const uint32_t bound = ANY ? 0u : (m2 & 0xFFFF0000u) | (tmin < 0.0f ? 0xFFFF0000u : 0u);
            if (!wide_push<LDS_STACK>(st, ws, u32x2{w1.x | (neg ? kDescend : 0u), bound | hits})) return kStepFallback;
        }
    }
    return kStepContinue;
}

// One node step (tg_mask == 0): visits st.cur, or the next child of the
// stack's top group (entering or leaving an instance: INST).  Returns
// kStepContinue, kStepDone when nothing is left (result ready for
// wide_finish), or kStepFallback when the stack is exhausted (the exact engine
// answers).  world_ray(o, d): the query's world ray, for leaving an instance
// (a functor, so that only that reads it).
template <int LDS_STACK, bool ANY, bool WT = false, bool INST = false, class WorldRay>
VR_HD int wide_node_step(const SceneView& sv, WideState& st, const WideStack& ws, float tmin, float tmax_any,
                         WorldRay world_ray) {
    while (st.cur == kNoNode) {
        if (st.sp == 0) return kStepDone;
        const u32x2 e = wide_top<LDS_STACK>(st, ws);
        if (INST && (e.x & kInstEntry)) {
            --st.sp;
            if (e.x == kInstExit) {
                vf3 wo, wd;
                world_ray(wo, wd);
                wide_instance_exit<WT>(st, wo, wd);
            } else if (ANY || !(u2f(e.y) > st.tbest * kCullSlack)) {  // (else the box lies beyond the best hit)
                return wide_instance_enter<LDS_STACK, WT>(sv, st, ws, e.x, tmin);
            }
            continue;
        }
        if (!ANY && u2f(e.y & 0xFFFF0000u) > st.tbest * kCullSlack) {
            --st.sp;
            continue;
        }
        const uint32_t hits = e.y & 0xFFu;
        const uint32_t slot = (e.x & kDescend) ? 31u - (uint32_t)__builtin_clz(hits) : (uint32_t)__builtin_ctz(hits);
        st.cur = (e.x & ~kDescend) + slot;
        if (hits & (hits - 1u)) wide_set_top<LDS_STACK>(st, ws, u32x2{e.x, e.y & ~(1u << slot)});
        else --st.sp;
    }
    const uint32_t node = st.cur;
    return wide_node<LDS_STACK, ANY>(sv, st, ws, node, tmin, tmax_any);
}

// Result of a finished query (after kStepDone).  Returns kStepDone or
// kStepFallback (winner not confirmed / any-hit candidates unconfirmed).
template <bool ANY, bool WT = false, bool INST = false>
VR_HD int wide_finish(const SceneView& sv, const WideState& st, float tmin, HitOut& out) {
    out.t = 0.f;
    out.u = 0.f;
    out.v = 0.f;
    out.prim = 0xFFFFFFFFu;
    if (ANY) {
        if (st.found) {
            out.t = st.tbest;
            out.u = st.bu;
            out.v = st.bv;
            out.prim = (st.best_slot & kAnalyticSlot) ? sv.analytic[st.best_slot & ~kAnalyticSlot].prim
                       : (INST && st.best_inst != kNoInstance) ? st.best_prim
                                                                : tri_word(sv.tris, st.best_slot, 9);
            return kStepDone;
        }
        return st.unconfirmed ? kStepFallback : kStepDone;
    }
    if (st.best_slot == 0xFFFFFFFFu) return kStepDone;
    if ((st.best_slot & kAnalyticSlot) || (INST && st.best_inst != kNoInstance)) {
        // analytic: confirmed when it was seeded; instance: nothing to confirm
        out.t = st.tbest;
        out.u = st.bu;
        out.v = st.bv;
        out.prim = st.best_prim;
        return kStepDone;
    }
    vf3 p0, p1, p2;
    load_tri_geom(sv.tris, st.best_slot, p0, p1, p2);
    // (a finished query is back in world space: every exit entry was popped)
    if (!WT && !confirm_winner(sv, st.o, st.d, tmin, st.tbest, p0, p1, p2, tri_word(sv.tris, st.best_slot, 11),
                               tri_word(sv.tris, st.best_slot, 9)))
        return kStepFallback;
    out.t = st.tbest;
    out.u = st.bu;
    out.v = st.bv;
    out.prim = tri_word(sv.tris, st.best_slot, 9);
    return kStepDone;
}

// Whole query for one ray (used by the host-side checks and simple kernels).
template <int LDS_STACK, bool ANY, bool WT = false, bool INST = false>
VR_HD int trace_wide(const SceneView& sv, vf3 o, vf3 d, float tmin, float tmax_any, const WideStack& ws,
                     HitOut& out) {
    WideState st;
    wide_init<WT>(st, o, d, sv.num_qnodes > 0);
    if (sv.num_analytic) wide_seed_analytic<ANY, WT>(sv, st, tmin, tmax_any);
    int rc;
    do {
        rc = st.tg_mask ? wide_tri_step<LDS_STACK, ANY, WT, INST>(sv, st, ws, tmin, tmax_any)
                        : wide_node_step<LDS_STACK, ANY, WT, INST>(sv, st, ws, tmin, tmax_any, [&](vf3& wo, vf3& wd) {
                              wo = o;
                              wd = d;
                          });
    } while (rc == kStepContinue);
    if (rc == kStepFallback) {
        out.prim = 0xFFFFFFFFu;
        return kStepFallback;
    }
    return wide_finish<ANY, WT, INST>(sv, st, tmin, out);
}

// Exact reference engine for one ray (closest hit).  The two traversal
// stacks (64 entries each, element k at [k * stride]) are the caller's: local
// arrays, or a lane's slice of LDS.  WT: the watertight engine's fallback
// (conservative slab tests, watertight triangle test).
template <bool WT = false>
__host__ __device__ inline void trace_exact_stk(const SceneView& sv, vf3 o, vf3 d, float tmin, HitOut& out,
                                                int32_t* tstack, int32_t* mstack, int stride) {
    out.prim = 0xFFFFFFFFu;
    out.t = out.u = out.v = 0.f;
    if (!sv.top_root_valid) return;
    WTRay wt{};
    if (WT) wt = wt_prepare(d);
    bool have = false;
    float bt = 0.f;
    int tsp = 0;
    tstack[tsp++ * stride] = 0;
    while (tsp) {
        int32_t ni = tstack[--tsp * stride];
        RefNode tn = sv.top_nodes[ni];
        if (tn.obj < 0) {
            Box3 b{mk3(tn.lo[0], tn.lo[1], tn.lo[2]), mk3(tn.hi[0], tn.hi[1], tn.hi[2])};
            if (WT ? wt_slab_hit(b, o, d, tmin, kInf) : ref_slab_hit(b, o, d, tmin, kInf)) {
                tstack[tsp++ * stride] = tn.right;
                tstack[tsp++ * stride] = ni + 1;
            }
            continue;
        }
        uint32_t surf = (uint32_t)tn.obj;
        SurfaceInfo si = sv.surfaces[surf];
        if (si.analytic >= 0) {
            float t, u, v;
            if (analytic_hit(sv.analytic[si.analytic], o, d, tmin, t, u, v) &&
                (!have || t < bt || (t == bt && si.prim_base < out.prim))) {
                have = true;
                bt = t;
                out.t = t;
                out.u = u;
                out.v = v;
                out.prim = si.prim_base;
            }
            continue;
        }
        MeshInfo mi = sv.meshes[si.mesh];
        // an instance's mesh is walked with the ray in its object space
        vf3 mo = o, md = d;
        WTRay mwt = wt;
        float meps = -1.0f;
        if (si.instance >= 0) {
            instance_ray(sv.instances[si.instance], o, d, mo, md);
            if (WT) mwt = wt_prepare(md);
            meps = tmin * sv.instances[si.instance].det_inv;
        }
        auto test = [&](uint32_t tri) {
            const uint32_t* ix = sv.mesh_idx + 3 * (size_t)(mi.tri_base + tri);
            const float* vp = sv.vpos + 3 * (size_t)mi.vert_base;
            vf3 p0 = mk3(vp[3 * ix[0]], vp[3 * ix[0] + 1], vp[3 * ix[0] + 2]);
            vf3 p1 = mk3(vp[3 * ix[1]], vp[3 * ix[1] + 1], vp[3 * ix[1] + 2]);
            vf3 p2 = mk3(vp[3 * ix[2]], vp[3 * ix[2] + 1], vp[3 * ix[2] + 2]);
            MTResult r;
            if (WT ? !wt_hit(mwt, mo, p0, p1, p2, tmin, r) : !mt_hit(mo, md, p0, p1, p2, tmin, r, meps)) return;
            const uint32_t prim = si.prim_base + tri;
            if (!have || r.t < bt || (r.t == bt && prim < out.prim)) {
                have = true;
                bt = r.t;
                out.t = r.t;
                out.u = r.u;
                out.v = r.v;
                out.prim = prim;
            }
        };
        if (mi.root < 0) {
            for (uint32_t k = 0; k < mi.num_tris; ++k) test(k);
            continue;
        }
        int msp = 0;
        mstack[msp++ * stride] = mi.root;
        while (msp) {
            int32_t mj = mstack[--msp * stride];
            RefNode nd = sv.ref_nodes[mj];
            if (nd.obj >= 0) {
                test((uint32_t)nd.obj);
                continue;
            }
            Box3 b{mk3(nd.lo[0], nd.lo[1], nd.lo[2]), mk3(nd.hi[0], nd.hi[1], nd.hi[2])};
            if (!(WT ? wt_slab_hit(b, mo, md, tmin, kInf) : ref_slab_hit(b, mo, md, tmin, kInf))) continue;
            mstack[msp++ * stride] = nd.right;
            mstack[msp++ * stride] = mj + 1;
        }
    }
}

template <bool WT = false>
__host__ __device__ inline void trace_exact(const SceneView& sv, vf3 o, vf3 d, float tmin, HitOut& out) {
    int32_t tstack[64], mstack[64];
    trace_exact_stk<WT>(sv, o, d, tmin, out, tstack, mstack, 1);
}

}  // namespace vr
