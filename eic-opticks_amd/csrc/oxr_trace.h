// oxr_trace.h -- two-level BVH closest-hit traversal, the engine's replacement for the
// OptiX IAS/GAS traversal behind optixTrace (CSGOptiX/CSGOptiX7.cu:110-216) together
// with __intersection__is, __closesthit__ch and __miss__ms (CSGOptiX7.cu:655-940).
//
// Layout in HBM:
//   tlas[]  BNode 64 B: both child boxes + child refs; BFS order so the top levels are
//           the first nodes and a workgroup can stage them in LDS. The two-level form's array
//           holds the instance tree, then every solid's tree over its prim AABBs.
//   inst[]  InstD 64 B: world-to-object columns + (solid, iindex|identity, flags, root of the
//           solid's tree).
//   prim[]  int2 (nodeOffset, globalPrimIdx<<16|boundary).
//   flat[]  int4 per leaf when the geometry is flattened: one BVH over every placed prim's
//           world box, no second level. trace<..., FLAT=true> walks that tree.
// A child ref is a node (>= 0), a prim leaf ~k (k: the prim's place in prim[], or the leaf's
// in flat[]; at most 2^30 of them) or an instance leaf 0x80000000 + instance (two-level
// form), so one unsigned comparison tells what a lane has to do next. The traversal stack
// lives in LDS, one column per lane, its first entry the end mark.
#pragma once
#include "oxr_device.h"

namespace oxd {

struct BNode { float4 a, b, c; int4 ch; };
// A staged node is read through an LDS-typed pointer, so it loads with ds_read; a load
// through one pointer that may address either LDS or global memory compiles to a flat load,
// which takes the vector-memory path for both.
typedef float LdsF4 __attribute__((ext_vector_type(4)));
typedef int LdsI4 __attribute__((ext_vector_type(4)));
struct LdsNode { LdsF4 a, b, c; LdsI4 ch; };
typedef __attribute__((address_space(3))) const LdsNode LdsNodeL;
OXD BNode lds_node(const BNode* top, int i) {
    LdsNodeL* p = (LdsNodeL*)top + i;
    const LdsF4 a = p->a, b = p->b, c = p->c;
    const LdsI4 ch = p->ch;
    BNode n;
    n.a = make_float4(a.x, a.y, a.z, a.w);
    n.b = make_float4(b.x, b.y, b.z, b.w);
    n.c = make_float4(c.x, c.y, c.z, c.w);
    n.ch = make_int4(ch.x, ch.y, ch.z, ch.w);
    return n;
}
struct InstD { float4 c0, c1, c2; int4 info; };   // info: prim offset, ii_id, flags (bit 0 identity,
                                                  // bits 8-15 visibility mask), blas_root
// an instance takes part in a trace when its visibility mask shares a bit with the ray's
// (OptixInstance::visibilityMask against optixTrace's visibilityMask, SBT.cc:538-545)
OXD bool visible(const InstD& in, unsigned vizmask) { return ((unsigned(in.info.z) >> 8) & vizmask) != 0u; }

struct Geom {
    const float4* node;    // two float4 per CSG node (load_node)
    const float4* plan;
    const float4* itra;    // three float4 per inverse CSG transform, its rows (intersect_leaf)
    const int2* prim;
    const BNode* tlas;
    const InstD* inst;
    const int4* flat;      // flattened leaves {instance, prim's place, its node offset, InstD flags}, or null
    int tlas_root;
    int num_inst;
    unsigned vizmask;      // ray visibility mask against InstD flag bits 8-15
    // radial bounds, two float4 per node of tlas {centre, (r_in0, r_out0, r_in1, r_out1)}
    const float4* rad;
    // far_pad's: the longest distance of a point of the scene from its origin, and the pad per distance
    float far_extent, far_scale;
};

struct Hit {
    float t;
    f3 n;          // world normal (not normalised)
    f3 lpos;       // object-frame hit position
    uint32_t ii_id, gpbd;
};

// Slab-test helpers. These only decide which boxes are entered, never a hit's value:
// the reciprocal is the hardware approximation (v_rcp_f32, 1 ulp) and the slab
// distances are fma(bound, inv, -origin*inv). The host widens every stored box by more
// than the resulting rounding for ray origins anywhere in the scene.
OXD f3 safe_inv(f3 d) {
    const float e = 1e-20f;
    return mk(__builtin_amdgcn_rcpf(fabsf(d.x) > e ? d.x : copysignf(e, d.x)),
              __builtin_amdgcn_rcpf(fabsf(d.y) > e ? d.y : copysignf(e, d.y)),
              __builtin_amdgcn_rcpf(fabsf(d.z) > e ? d.z : copysignf(e, d.z)));
}
OXD f3 neg_oi(f3 o, f3 inv) { return mk(-(o.x * inv.x), -(o.y * inv.y), -(o.z * inv.z)); }
// A box holds what the single-precision tests of its prims may report from origins within the
// scene (oxr_boxes.h). The error of a test grows with the origin's distance D: for a ray from
// outside, a box has to reach sqrt(2e-6) D further, times the worst stretch of a leaf's
// transform. far_scale holds both; nothing is added for an origin within the scene. In the
// frame of an instance the pad is as much longer as its transform may stretch it (in_frame).
OXD bool far_away(const Geom& g, f3 pos) { return dot(pos, pos) > g.far_extent * g.far_extent; }
OXD float far_pad(const Geom& g, f3 pos) {
    return far_away(g, pos) ? g.far_scale * (__builtin_amdgcn_sqrtf(dot(pos, pos)) + g.far_extent) : 0.f;
}
OXD float in_frame(const InstD& in, float pad) {
    const float n2 = in.c0.x * in.c0.x + in.c0.y * in.c0.y + in.c0.z * in.c0.z + in.c1.x * in.c1.x + in.c1.y * in.c1.y +
                     in.c1.z * in.c1.z + in.c2.x * in.c2.x + in.c2.y * in.c2.y + in.c2.z * in.c2.z;
    return 1.7321f * pad * __builtin_amdgcn_sqrtf(n2);
}
// slab test of one child box (noi_lo, noi_hi: -origin*inv for its low and high planes, which
// differ by what the box is widened by)
OXD bool box_hit(float lx, float ly, float lz, float hx, float hy, float hz, f3 noi_lo, f3 noi_hi, f3 inv, float tbest, float& tn) {
    float tx0 = fmaf(lx, inv.x, noi_lo.x), tx1 = fmaf(hx, inv.x, noi_hi.x);
    float ty0 = fmaf(ly, inv.y, noi_lo.y), ty1 = fmaf(hy, inv.y, noi_hi.y);
    float tz0 = fmaf(lz, inv.z, noi_lo.z), tz1 = fmaf(hz, inv.z, noi_hi.z);
    float n = fmaxf(fmaxf(fminf(tx0, tx1), fminf(ty0, ty1)), fminf(tz0, tz1));
    float f = fminf(fminf(fmaxf(tx0, tx1), fmaxf(ty0, ty1)), fmaxf(tz0, tz1));
    tn = n;
    return n <= f && f >= 0.f && n <= tbest;
}

// world -> object frame of one instance (rows c0..c2 hold the world-to-object 3x4)
OXD void to_object(const InstD& in, f3 pos, f3 mom, f3& o, f3& d) {
    o = mk(in.c0.x * pos.x + in.c0.y * pos.y + in.c0.z * pos.z + in.c0.w,
           in.c1.x * pos.x + in.c1.y * pos.y + in.c1.z * pos.z + in.c1.w,
           in.c2.x * pos.x + in.c2.y * pos.y + in.c2.z * pos.z + in.c2.w);
    d = mk(in.c0.x * mom.x + in.c0.y * mom.y + in.c0.z * mom.z,
           in.c1.x * mom.x + in.c1.y * mom.y + in.c1.z * mom.z,
           in.c2.x * mom.x + in.c2.y * mom.y + in.c2.z * mom.z);
}

// Closest hit in (tmin, tmax]; ties in t go to the smaller (instance, local prim) key.
//
// A traversal is a resumable state (Trav) moved on by two steps: trav_node visits one BVH
// node (in the two-level form also enters or leaves an instance), trav_leaf tests one prim.
// The simulate kernels hold 64 of these in a wave and choose which step runs by how many
// lanes wait for it; trace() runs one traversal to its end. The order of a lane's own steps
// is the same in both.
//
// Template flags: SHALLOW: every CSG tree of the geometry has height <= 2 (register-resident
// CSG stacks). RADIAL: besides its box, each child must pass its radial bound: its surfaces
// lie between r_in and r_out from the node's centre c, so along a ray from o (direction
// length |d|) they are no nearer than max(r_in - |o - c|, |o - c| - r_out) / |d|; a child
// whose bound lies beyond the best hit is skipped, and the bound orders the children and
// fills the distance stack. Concentric shells, whose boxes all hold the ray origin, are
// culled this way. TN: a second column of cap floats follows the stack (at stk + stride*cap)
// holding each pushed node's box entry distance, and a popped node whose entry lies beyond
// the best hit so far is dropped without loading it: the same cull the box test applies, so
// the hit found is the same.
//
// Only (t, instance, local prim, object-frame normal) of the best hit and the stack position
// live between steps: the ray in the current frame and its reciprocals are formed again
// where a run of steps begins (ray_of, from the photon and the instance record), and the
// best hit's world normal, local position and identity words after the end (trav_hit), all
// with the same arithmetic.
//
// What a lane waits for, as ranges of the unsigned ref: [0, TRAV_WAIT_END) a node step,
// from PRIM_LEAVES on a leaf step, and between the two a lane whose traversal has ended or
// that holds no photon.
constexpr uint32_t INST_LEAVES = 0x80000000u;
constexpr uint32_t TRAV_BACK = 0xbffffff0u;       // leave the instance's tree
constexpr uint32_t TRAV_WAIT_END = 0xbffffff1u;
constexpr uint32_t TRAV_DONE = 0xbffffff8u;       // the traversal has ended (best_inst < 0: a miss)
constexpr uint32_t TRAV_IDLE = 0xbffffff9u;       // the lane holds no photon
constexpr uint32_t PRIM_LEAVES = 0xc0000000u;
constexpr int INST_IDENT = 1 << 30;               // Trav::inst: the instance's transform is the identity
struct Trav {
    float best;
    uint32_t cur;
    int sp;                     // the free stack entry's offset: entry k of a lane lies at k*stride
    int inst;                   // two-level form: the instance being walked, -1 in the instance tree
    int best_inst, best_item;   // (instance, prim's place), or (flat leaf, 0): leaves are numbered in that order
    f3 bn;
};
OXD bool at_node(const Trav& v) { return v.cur < TRAV_WAIT_END; }
OXD bool at_leaf(const Trav& v) { return v.cur >= PRIM_LEAVES; }
OXD void trav_begin(Trav& v, const Geom& g, float tmax, int* stk, int stride, int cap, bool tn) {
    v.best = tmax;
    v.cur = uint32_t(g.tlas_root);
    stk[0] = int(TRAV_DONE);
    if (tn) reinterpret_cast<float*>(stk)[stride * cap] = -INFINITY;
    v.sp = stride;
    v.inst = -1;
    v.best_inst = -1;
    v.best_item = 0;
    v.bn = mk(0.f, 0.f, 0.f);
}

// the ray in the frame of the current tree, and what the slab tests need of it
// WIDE: the boxes are widened for origins outside the scene (far_pad); the high planes
// then have their own product, and a radial bound lies off, sqrt(3) of the pad, nearer
template <bool WIDE> struct RayF {
    f3 o, inv, noi;
    float ilen;
    OXD f3 noi_high() const { return noi; }
    OXD float bound(float x) const { return x * ilen; }
    OXD void widen(float) {}
};
template <> struct RayF<true> {
    f3 o, inv, noi, noi_hi;
    float ilen, off;
    OXD f3 noi_high() const { return noi_hi; }
    OXD float bound(float x) const { return fmaf(x, ilen, -off); }
    OXD void widen(float pad) {
        noi_hi = mk(fmaf(pad, inv.x, noi.x), fmaf(pad, inv.y, noi.y), fmaf(pad, inv.z, noi.z));
        noi = mk(fmaf(-pad, inv.x, noi.x), fmaf(-pad, inv.y, noi.y), fmaf(-pad, inv.z, noi.z));
        off = 1.7321f * pad * ilen;
    }
};
template <bool RADIAL, bool WIDE>
OXD void ray_frame(RayF<WIDE>& r, f3 o, f3 d, float pad) {
    r.o = o;
    r.inv = safe_inv(d);
    r.noi = neg_oi(o, r.inv);
    r.ilen = RADIAL ? __builtin_amdgcn_rsqf(dot(d, d)) : 1.f;
    r.widen(pad);
}
template <bool RADIAL, bool WIDE>
OXD void ray_world(RayF<WIDE>& r, const Geom& g, f3 pos, f3 mom) { ray_frame<RADIAL>(r, pos, mom, WIDE ? far_pad(g, pos) : 0.f); }
template <bool RADIAL, bool WIDE>
OXD void ray_inst(RayF<WIDE>& r, const Geom& g, const InstD& in, f3 pos, f3 mom) {
    f3 o, d;
    to_object(in, pos, mom, o, d);
    ray_frame<RADIAL>(r, o, d, WIDE ? in_frame(in, far_pad(g, pos)) : 0.f);
}
template <bool FLAT, bool RADIAL, bool WIDE>
OXD void ray_of(RayF<WIDE>& r, const Geom& g, const Trav& v, f3 pos, f3 mom) {
    if (FLAT || v.inst < 0 || (v.inst & INST_IDENT)) ray_world<RADIAL>(r, g, pos, mom);
    else ray_inst<RADIAL>(r, g, g.inst[v.inst], pos, mom);
}

// the next stack entry worth visiting; the first one is the end mark
template <bool TN>
OXD void trav_pop(Trav& v, const int* stk, int stride, int cap) {
    v.sp -= stride;
    if (TN) {
        const float* stkt = reinterpret_cast<const float*>(stk + stride * cap);
        while (stkt[v.sp] > v.best) v.sp -= stride;
    }
    v.cur = uint32_t(stk[v.sp]);
}

struct TraceCount { uint32_t visits, tests, csgb, ivis; };

template <bool COUNT, bool TN, bool FLAT, bool RADIAL, bool WIDE>
OXD void trav_node(Trav& v, const Geom& g, RayF<WIDE>& r, f3 pos, f3 mom, int* stk, int stride, int cap, const BNode* top, int ntop,
                   uint32_t& err, TraceCount& cnt) {
    float* stkt = reinterpret_cast<float*>(stk + stride * cap);
    if (FLAT || v.cur < INST_LEAVES) {
        const int cur = int(v.cur);
        float4 rc, rr;
        // first, so that they are under way while the node comes and its boxes are tested (left
        // where they are used, thin shells took 11.6 ms and not 11.1)
        if (RADIAL) { rc = g.rad[2 * cur]; rr = g.rad[2 * cur + 1]; }
        BNode nd;
        if (cur < ntop) nd = lds_node(top, cur);
        else nd = g.tlas[cur];
        if (COUNT) cnt.visits++;
        float tn0, tn1;
        bool h0 = box_hit(nd.a.x, nd.a.y, nd.a.z, nd.a.w, nd.b.x, nd.b.y, r.noi, r.noi_high(), r.inv, v.best, tn0);
        bool h1 = box_hit(nd.b.z, nd.b.w, nd.c.x, nd.c.y, nd.c.z, nd.c.w, r.noi, r.noi_high(), r.inv, v.best, tn1);
        if (RADIAL) {
            const float dx = r.o.x - rc.x, dy = r.o.y - rc.y, dz = r.o.z - rc.z;
            const float dist = __builtin_amdgcn_sqrtf(dx * dx + dy * dy + dz * dz);
            const float lb0 = r.bound(fmaxf(rr.x - dist, dist - rr.y));
            const float lb1 = r.bound(fmaxf(rr.z - dist, dist - rr.w));
            h0 = h0 && lb0 <= v.best;
            h1 = h1 && lb1 <= v.best;
            tn0 = fmaxf(tn0, lb0);
            tn1 = fmaxf(tn1, lb1);
        }
        if (h0 || h1) {
            const bool first0 = h0 && !(h1 && tn1 < tn0);   // the nearer child, child 0 in a tie
            v.cur = uint32_t(first0 ? nd.ch.x : nd.ch.y);
            if (h0 && h1) {
                if (v.sp < stride * cap) {
                    stk[v.sp] = first0 ? nd.ch.y : nd.ch.x;
                    if (TN) stkt[v.sp] = first0 ? tn1 : tn0;
                    v.sp += stride;
                } else {
                    err |= 1u;
                }
            }
        } else {
            trav_pop<TN>(v, stk, stride, cap);
        }
        return;
    }
    if constexpr (!FLAT) {
        if (v.cur == TRAV_BACK) {      // the instance's tree is done: back to the world frame
            v.inst = -1;
            ray_world<RADIAL>(r, g, pos, mom);
            trav_pop<TN>(v, stk, stride, cap);
            return;
        }
        const int item = int(v.cur - INST_LEAVES);
        const InstD in = g.inst[item];
        if (COUNT) cnt.ivis++;
        if (!visible(in, g.vizmask)) {
            trav_pop<TN>(v, stk, stride, cap);
            return;
        }
        const bool ident = (in.info.z & 1) != 0;
        v.inst = item | (ident ? INST_IDENT : 0);
        if (!ident) ray_inst<RADIAL>(r, g, in, pos, mom);
        if (v.sp < stride * cap) {
            stk[v.sp] = int(TRAV_BACK);
            if (TN) stkt[v.sp] = -INFINITY;
            v.sp += stride;
        } else {
            err |= 1u;
        }
        v.cur = uint32_t(in.info.w);
    }
}

template <bool FP64, bool COUNT, bool LIST, bool TN, bool FLAT, bool SHALLOW, bool SIMPLE>
OXD void trav_leaf(Trav& v, const Geom& g, f3 pos, f3 mom, float tmin, const int* stk, int stride, int cap, TraceCount& cnt) {
    const int leaf = int(~v.cur);
    f3 o = pos, d = mom;
    int nodeOffset;
    if (FLAT) {
        const int4 fi = g.flat[leaf];
        if (COUNT) cnt.ivis++;
        if (((unsigned(fi.w) >> 8) & g.vizmask) == 0u) {
            trav_pop<TN>(v, stk, stride, cap);
            return;
        }
        if ((fi.w & 1) == 0) to_object(g.inst[fi.x], pos, mom, o, d);
        nodeOffset = fi.z;
    } else {
        if (!(v.inst & INST_IDENT)) to_object(g.inst[v.inst], pos, mom, o, d);
        nodeOffset = g.prim[leaf].x;
    }
    if (COUNT) {
        cnt.tests++;
        const unsigned nn = node_type(g.node, nodeOffset) >= CSG_LEAF ? 1u : node_word0(g.node, nodeOffset);
        for (unsigned k = 0; k < nn; k++) {   // 64 B per CSGNode and per transform it carries
            const float4 q1 = g.node[2 * (nodeOffset + int(k)) + 1];
            cnt.csgb += 64u;
            if (__float_as_uint(q1.z) >= CSG_LEAF && (__float_as_uint(q1.w) & 0x7fffffffu) != 0u) cnt.csgb += 64u;
        }
    }
    Is is;
    if (intersect_prim<FP64, LIST, SHALLOW, SIMPLE>(is, g.node, nodeOffset, g.plan, g.itra, tmin, o, d)) {
        // a reported distance outside the ray interval is ignored, as by
        // optixReportIntersection (CSGOptiX/CSGOptiX7.cu:912): a convex polyhedron
        // wholly behind the ray reports valid with the zeroed isect
        const float t = is.w;
        // ties go to the smaller (instance, prim)
        const int ki = FLAT ? leaf : (v.inst & ~INST_IDENT), kp = FLAT ? 0 : leaf;
        const bool before = v.best_inst >= 0 && t == v.best && (ki < v.best_inst || (ki == v.best_inst && kp < v.best_item));
        if (t >= tmin && (t < v.best || before)) {
            v.best = t; v.best_inst = ki; v.best_item = kp;
            v.bn = mk(is.x, is.y, is.z);
        }
    }
    trav_pop<TN>(v, stk, stride, cap);
}

// the ended traversal's hit; false for a miss
template <bool FLAT>
OXD bool trav_hit(const Trav& v, const Geom& g, f3 pos, f3 mom, Hit& hit) {
    if (v.best_inst < 0) {
        hit.t = 0.f; hit.n = mk(0.f, 0.f, 0.f); hit.lpos = mk(0.f, 0.f, 0.f);
        hit.ii_id = 0xffffffffu; hit.gpbd = 0xffffffffu;
        return false;
    }
    int bi = v.best_inst, bp = v.best_item;
    if (FLAT) {
        const int4 fi = g.flat[bi];
        bi = fi.x; bp = fi.y;
    }
    const InstD in = g.inst[bi];
    f3 bo = pos, bd = mom;
    bool ident = (in.info.z & 1) != 0;
    if (!ident) to_object(in, pos, mom, bo, bd);
    hit.t = v.best;
    hit.lpos = mk(bo.x + v.best * bd.x, bo.y + v.best * bd.y, bo.z + v.best * bd.z);
    hit.ii_id = uint32_t(in.info.y);
    hit.gpbd = uint32_t(g.prim[bp].y);
    if (!ident) {
        hit.n = mk(in.c0.x * v.bn.x + in.c1.x * v.bn.y + in.c2.x * v.bn.z,
                   in.c0.y * v.bn.x + in.c1.y * v.bn.y + in.c2.y * v.bn.z,
                   in.c0.z * v.bn.x + in.c1.z * v.bn.y + in.c2.z * v.bn.z);
    } else {
        hit.n = v.bn;
    }
    return true;
}

// one ray to its end (the query kernels)
template <bool FP64, bool LIST, bool FLAT>
OXD bool trace(const Geom& g, f3 pos, f3 mom, float tmin, float tmax, Hit& hit, int* stk, int stride, int cap,
               const BNode* top, int ntop) {
    Trav v;
    RayF<true> r;
    TraceCount cnt;
    uint32_t err = 0;
    trav_begin(v, g, tmax, stk, stride, cap, false);
    ray_world<false>(r, g, pos, mom);
    while (v.cur != TRAV_DONE) {
        if (at_leaf(v)) trav_leaf<FP64, false, LIST, false, FLAT, false, false>(v, g, pos, mom, tmin, stk, stride, cap, cnt);
        else trav_node<false, false, FLAT, false>(v, g, r, pos, mom, stk, stride, cap, top, ntop, err, cnt);
    }
    return trav_hit<FLAT>(v, g, pos, mom, hit);
}

} // namespace oxd
