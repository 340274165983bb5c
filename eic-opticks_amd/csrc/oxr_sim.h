// oxr_sim.h -- the per-photon pieces and the two simulate kernels (plain and persistent
// form), templated on root precision (FP64), counting (COUNT), debug outputs (DBG), list-node
// support (LIST) and the traversal mode TM (bit 0: stack entries carry box entry distances;
// bit 1: the flattened BVH; bit 2: every CSG tree has height <= 2, so the CSG evaluation
// stacks live in registers, production kernels without list nodes only; bit 3: nodes also
// cull by their radial bounds, production and counting kernels). k_generate
// (oxr_kernels.hip) uses the per-photon pieces; the kernels are instantiated by the
// oxr_sim_*.hip units, one per (FP64, LIST) pair and two for simple leaves, which compile in
// parallel.
#pragma once
#include "oxr_kernels.h"
#include "oxr_steps.h"

// Minimum waves per SIMD the simulate kernels are compiled for (VGPR budget 512/N per
// lane). 4 beat 3 and 5 on MI355X: with 5 the spilled registers cost more than the wave
// brings, with 3 the loop waits more for memory (kernel ms with 4, 3 and 5: instanced CSG 5.95,
// 6.73, 7.17; calorimeter 2.39, 2.93, 2.76; thin shells, 500k, 11.1, 13.7, 11.5).
#ifndef OXR_PERSIST_WAVES
#define OXR_PERSIST_WAVES 4
#endif
#ifndef OXR_PLAIN_WAVES
#define OXR_PLAIN_WAVES 4
#endif

namespace oxd {

// ------------------------------------------------------------------ seeding
// genstep g with offsets[g] <= i < offsets[g+1] (offsets non-decreasing, i < offsets[num_gs])
OXD int genstep_of(const long long* __restrict__ offsets, int num_gs, long long i) {
    int lo = 0, hi = num_gs - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (offsets[mid] <= i) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// ------------------------------------------------------------------ per-photon pieces
struct Lane {
    Ph p;
    Rng r;
    unsigned long long sh0, sh1, sb0, sb1;   // seqhis / seqbnd
    float lc, lf;                            // lposcost, lposfphi of the last trace (photonlite)
    long long idx;
    int bounce;
};

template <bool DBG>
OXD void point(const Params& P, Lane& L) {
    if (!DBG) return;
    if (P.record && L.bounce < P.max_record) store_photon(P.record + 4 * (L.idx * P.max_record + L.bounce), L.p);
    if (P.rec && L.bounce < P.max_rec) P.rec[L.idx * P.max_rec + L.bounce] = rec_pack(L.p, P.extent_domain, P.time_domain);
    if (P.seq) {
        unsigned slot = unsigned(L.bounce);
        if (slot < 32) {
            unsigned shift = 4u * (slot & 15u);
            unsigned long long his = (unsigned long long)(unsigned(__ffs(int(ph_flag(L.p)))) & 0xfu) << shift;
            unsigned long long bnd = (unsigned long long)(ph_boundary(L.p) & 0xfu) << shift;
            if (slot < 16) { L.sh0 |= his; L.sb0 |= bnd; } else { L.sh1 |= his; L.sb1 |= bnd; }
        }
    }
}

// the LDS copy of the node and itra arrays and the prim table (TM bit 5): after the P.ntop
// staged top nodes
// and the traversal stacks (blockDim.x lanes x P.stack_cap entries of 4 B, 8 B with
// distances), the layout simulate_smem sizes
OXD const float4* csg_copy(const Params& P) {
    extern __shared__ int4 smem4[];
    return reinterpret_cast<const float4*>(smem4) + 4 * P.ntop + (blockDim.x * unsigned(P.stack_cap) * (P.tn_stack ? 2u : 1u)) / 4u;
}

// returns false for padding indices of a batched step
template <bool DBG>
OXD bool begin_photon(const Params& P, Lane& L, long long idx) {
    L.idx = idx;
    const float4* gsb = P.gs;
    unsigned long long pidx;
    int gsi;
    int evt = P.event_index;
    if (P.segs) {
        int lo = 0, hi = P.nseg - 1;
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (P.segs[mid].start <= idx) lo = mid; else hi = mid - 1;
        }
        const Seg sg = P.segs[lo];
        long long li = idx - sg.start;
        if (li >= sg.count) return false;
        pidx = sg.photon0 + (unsigned long long)li;
        gsb = sg.gs;
        gsi = genstep_of(sg.off, sg.num_gs, (long long)pidx);   // served events carry no seed array
        evt = sg.event_index;
    } else {
        pidx = P.slot_offset + (unsigned long long)idx;
        gsi = P.seed[idx];
    }
    const float4* gs = gsb + 6 * gsi;
    rng_init(L.r, P.rng_seed, P.rng_offset, P.skip, (unsigned long long)evt, pidx);
    if (DBG && P.pre) { L.r.pre = P.pre + (size_t)idx * P.npre; L.r.npre = P.npre; }
    rng_rest(L.r);
    uint32_t gencode = __float_as_uint(gs[0].x);
    // the photon starts zeroed (sctx ctx = {}, CSGOptiX7.cu:432): a generator that leaves a
    // field unset (T_RECTANGLE beyond its fourth side sets no position or direction,
    // sysrap/storch.h:460-512) leaves it zero
    L.p = Ph{};
    if (gencode == 6) gen_torch(L.p, gs, pidx, L.r);
    else if (gencode == 15 || gencode == 18) gen_cerenkov(L.p, gs, L.r, P.t);
    else if (gencode == 16 || gencode == 5) gen_scint(L.p, gs, L.r, P.t);
    else if (gencode == 19) { load_photon(L.p, P.input + 4 * pidx); set_flag(L.p, TORCH); }
    else { zero_flags(L.p); }
    set_index(L.p, pidx);
    L.sh0 = L.sh1 = L.sb0 = L.sb1 = 0ull;
    if (DBG) { L.lc = 0.f; L.lf = 0.f; }
    L.bounce = 0;
    point<DBG>(P, L);
    return true;
}

// the geometry as the kernel reads it: with CSGL the node and itra arrays and the prim table
// come from the LDS copy stage_csg made
template <bool CSGL>
OXD Geom geom_of(const Params& P) {
    Geom g = P.g;
    if constexpr (CSGL) {
        g.node = csg_copy(P);
        g.itra = g.node + P.csg_node4;
        g.prim = reinterpret_cast<const int2*>(g.itra + P.csg_itra4);
    }
    return g;
}

// trace<refine> (CSGOptiX7.cu:110-216): with PropagateRefine, when 0.99 of the distance
// found lies beyond the refine distance, the ray is traced again from that point and the
// 0.99 part added back, so a far surface is intersected from close by. A miss reports
// distance 1, as the miss program writes it (CSGOptiX7.cu:666-670), so h.t is the
// reference's prd distance in every case. t_approx holds the part already covered,
// NOT_REFINED before the second trace.
constexpr float NOT_REFINED = -1e38f;
OXD f3 ray_origin(f3 pos, f3 mom, float t_approx) {
    if (t_approx == NOT_REFINED) return pos;
    return mk(pos.x + t_approx * mom.x, pos.y + t_approx * mom.y, pos.z + t_approx * mom.z);
}
// true when the ended trace (distance h.t) has to run again from t_approx, which is set
OXD bool refine_again(const Params& P, const Hit& h, float& t_approx) {
    if (!P.refine || t_approx != NOT_REFINED) return false;
    const float ta = 0.99f * h.t;
    if (!(ta > P.refine_distance)) return false;
    t_approx = ta;
    return true;
}

// the photon goes on to another trace (loop condition of CSGOptiX7.cu:450-482)
OXD bool goes_on(const Params& P, const Lane& L) { return L.bounce < P.max_bounce && L.p.time < P.max_time; }
OXD float photon_tmin(const Params& P, const Lane& L) { return (L.p.obf & P.eps0_mask) ? P.tmin0 : P.tmin; }

// what one loop iteration of CSGOptiX7.cu:450-482 does with its trace; returns false when the
// photon is done
template <bool DBG>
OXD bool shade(const Params& P, Lane& L, const Hit& h, bool found) {
    if (!found) {
        if (DBG) { L.lc = 0.f; L.lf = 0.f; }   // __miss__ms sets lposcost = lposfphi = 0
        return false;
    }
    // normalize(n) is n * (1 / sqrt(dot(n, n))): when that dot rounds to exactly 1 it
    // returns n itself, so an already unit normal (boxes, polyhedra) skips the arithmetic
    const float nn = dot(h.n, h.n);
    f3 normal = nn == 1.f ? h.n : normalize(h.n);
    if (DBG && (P.lite || P.prd)) {
        L.lc = lpos_cost(h.lpos);
        L.lf = (xatan2(h.lpos.y, h.lpos.x) + PIf) / (2.0f * PIf);   // normalize_fphi, sysrap/scuda.h:653
    }
    // sctx::trace (sysrap/sctx.h:170-173): the trace result of this bounce, normal normalised
    // (CSGOptiX7.cu:466-474), in the quad2 layout of sysrap/squad.h:95-112
    if (DBG && P.prd && L.bounce < P.max_prd) {
        float4* q = P.prd + 2 * (L.idx * P.max_prd + L.bounce);
        q[0] = make_float4(normal.x, normal.y, normal.z, h.t);
        q[1] = make_float4(L.lc, L.lf, __uint_as_float(h.ii_id), __uint_as_float(h.gpbd));
    }
    int command = propagate(L.p, h, normal, L.r, P.t, P.aligned);
    L.bounce++;
    point<DBG>(P, L);
    return command != BREAK;
}

// production launches: pick up a photon that k_generate wrote (false for padding)
OXD bool resume_photon(const Params& P, Lane& L, long long idx) {
    const ulonglong2 st = P.rstate[idx];
    if (st.x == ~0ull) return false;
    L.idx = idx;
    load_photon(L.p, P.photon + 4 * idx);
    rng_resume(L.r, P.rng_seed, st.x, st.y);
    rng_rest(L.r);
    L.bounce = 0;
    return true;
}

template <bool DBG>
OXD bool start_photon(const Params& P, Lane& L, long long idx) {
    if (DBG) return begin_photon<true>(P, L, idx);
    if (P.gen_inplace) return begin_photon<false>(P, L, idx);
    return resume_photon(P, L, idx);
}

template <bool DBG>
OXD void end_photon(const Params& P, const Lane& L) {
    if (DBG && P.seq) {
        ulonglong2* s = P.seq + 2 * L.idx;
        s[0] = make_ulonglong2(L.sh0, L.sh1);
        s[1] = make_ulonglong2(L.sb0, L.sb1);
    }
    store_photon(P.photon + 4 * L.idx, L.p);
    // all bits of the hit mask must be set (sphoton_selector, sysrap/sphoton.h:1219-1225)
    if (P.hitflag) P.hitflag[L.idx] = (L.p.flagmask & P.hitmask) == P.hitmask ? 1 : 0;
    if (DBG && P.lite) P.lite[L.idx] = lite_pack(L.p, L.lc, L.lf);
    if (DBG && P.bounce_out) P.bounce_out[L.idx] = uint32_t(L.bounce);
    if (DBG && P.overflow_out) P.overflow_out[L.idx] = L.r.overflow;
}

OXD void stage_top(const Params& P, BNode* top, int ntop) {
    for (int i = threadIdx.x; i < ntop; i += blockDim.x) top[i] = P.g.tlas[i];
}

// TM bit 5 (32): the node and itra arrays and the prim table are copied into LDS after the
// top nodes and the traversal stacks, and the trace reads them there. The copy's address derives from the
// LDS array alone, so its reads compile to ds_read.
template <int TM>
OXD void stage_csg(const Params& P) {
    if constexpr ((TM & 32) != 0) {
        float4* l = const_cast<float4*>(csg_copy(P));
        for (int i = threadIdx.x; i < P.csg_node4; i += blockDim.x) l[i] = P.g.node[i];
        for (int i = threadIdx.x; i < P.csg_itra4; i += blockDim.x) l[P.csg_node4 + i] = P.g.itra[i];
        int2* lp = reinterpret_cast<int2*>(l + P.csg_node4 + P.csg_itra4);
        for (int i = threadIdx.x; i < P.csg_prim; i += blockDim.x) lp[i] = P.g.prim[i];
    }
}

OXD unsigned long long wave_sum(unsigned long long v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

OXD void flush_counters(const Params& P, unsigned long long steps, unsigned long long visits,
                        unsigned long long tests, uint32_t err, bool count,
                        unsigned long long csgb = 0, unsigned long long ivis = 0) {
    steps = wave_sum(steps);
    if (count) { visits = wave_sum(visits); tests = wave_sum(tests); csgb = wave_sum(csgb); ivis = wave_sum(ivis); }
    uint64_t anyerr = __ballot(err != 0u);
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(P.counters + 0, steps);
        if (count) {
            atomicAdd(P.counters + 2, visits); atomicAdd(P.counters + 3, tests);
            atomicAdd(P.counters + 5, csgb); atomicAdd(P.counters + 6, ivis);
        }
        if (anyerr) atomicAdd(P.counters + 4, 1ull);
    }
}


// ------------------------------------------------------------------ the wave's loop
// A wave holds up to 64 photons, each at its own place: at a BVH node, at a prim to test, or
// at the end of its trace with a bounce to compute. A turn of the loop runs one of the three
// for the lanes that wait for it. The loop is bound by vector issue under divergence: when a
// bounce waited for every lane's trace and a prim was tested as soon as one lane reached it,
// 18-37% of the lanes of an issued instruction were active, now 38-42%.
//   * Nodes run while NODE_LEAST/64 of the wave's photons are at one: a visit costs a tenth to
//     a fiftieth of a prim test or a bounce and brings lanes on to those. With radial bounds a
//     visit costs a third more and is most of the time, so it wants more lanes
//     (NODE_LEAST_RADIAL).
//   * Prims are tested before bounces are computed unless LEAF_WEIGHT times as many lanes wait
//     for a bounce, the dearer step. Choosing by the steps' measured clocks was slower on every
//     event but the calorimeter.
// The plain form has no photons to refill idle lanes with, and in a small launch a wave alone on
// its SIMD pays every turn in full: it runs each step to the last lane.
// Kernel times on MI355X with the settings of tuning_gfx950.json (ms): instanced CSG (10M
// photons) 5.95, with NODE_LEAST 3 5.88, with 12 6.27; with LEAF_WEIGHT 2 6.52, with 32 5.95.
// Thin shells (500k) 11.1, with NODE_LEAST_RADIAL 6 12.3, with 20 10.7. Calorimeter (2.07M) 2.39
// whichever, 2.44 with LEAF_WEIGHT 2; plain form, 62k photons, 0.71, with the persistent form's
// two values 0.77. The bounce-by-bounce loop took 9.5 (instanced CSG), 20.9 (thin shells) and
// 2.9 ms (calorimeter) with its own settings.
constexpr int NODE_LEAST = 6, NODE_LEAST_RADIAL = 12, LEAF_WEIGHT = 16;
constexpr int NODE_LEAST_PLAIN = 1, LEAF_WEIGHT_PLAIN = 64;

template <bool FP64, bool COUNT, bool DBG, bool LIST, int TM, bool REFILL>
OXD void run_wave(const Params& P, int* stk, int stride, const BNode* top) {
    constexpr bool TN = (TM & 1) != 0, FLAT = (TM & 2) != 0, SHALLOW = (TM & 4) != 0, RADIAL = (TM & 8) != 0,
                   SIMPLE = (TM & 16) != 0, CSGL = (TM & 32) != 0;
    const Geom g = geom_of<CSGL>(P);
    const int lane = threadIdx.x & 63;
    Lane L;
    Trav v;
    float t_approx = NOT_REFINED;
    uint32_t steps = 0;
    uint32_t err = 0;
    TraceCount cnt = {0, 0, 0, 0};
    v.cur = TRAV_IDLE;
    bool first = true, drained = false;
    // When the wave last took photons, one it held was outside the scene (far_pad). A bounce takes
    // it to a surface, inside, or so little beyond that the stored margins, twice the errors'
    // bound, hold it; looking after every bounce too spills four registers more.
    bool far_wave = false;
    unsigned long long pool = 0;   // photons the wave has claimed and not yet started: [pool, pool + pooled)
    int pooled = 0;
    for (;;) {
        int nnode = __popcll(__ballot(at_node(v)));
        const int nleaf = __popcll(__ballot(at_leaf(v)));
        const int nend = __popcll(__ballot(v.cur == TRAV_DONE));
        const int least = max(1, ((nnode + nleaf + nend) * (!REFILL ? NODE_LEAST_PLAIN : RADIAL ? NODE_LEAST_RADIAL : NODE_LEAST)) >> 6);   // lanes that keep the nodes running
        if (nnode >= least) {
            const f3 org = P.refine ? ray_origin(L.p.pos, L.p.mom, t_approx) : L.p.pos;
            auto visit = [&](auto r) __attribute__((always_inline)) {
                if (at_node(v)) ray_of<FLAT, RADIAL>(r, g, v, org, L.p.mom);
                do {
                    if (at_node(v)) trav_node<COUNT, TN, FLAT, RADIAL>(v, g, r, org, L.p.mom, stk, stride, P.stack_cap, top, P.ntop, err, cnt);
                    nnode = __popcll(__ballot(at_node(v)));
                } while (nnode >= least);
            };
            // in a loop of its own: one for both takes three registers more and 1-4% on every event
            if (__builtin_expect(far_wave, 0)) visit(RayF<true>());
            else visit(RayF<false>());
            continue;
        }
        if (nleaf > 0 && nleaf * (REFILL ? LEAF_WEIGHT : LEAF_WEIGHT_PLAIN) >= nend) {
            if (at_leaf(v))
                trav_leaf<FP64, COUNT, LIST, TN, FLAT, SHALLOW, SIMPLE>(v, g, P.refine ? ray_origin(L.p.pos, L.p.mom, t_approx) : L.p.pos,
                                                                       L.p.mom, photon_tmin(P, L), stk, stride, P.stack_cap, cnt);
            continue;
        }
        if (nend > 0 && v.cur == TRAV_DONE) {
            Hit h;
            const bool found = trav_hit<FLAT>(v, g, ray_origin(L.p.pos, L.p.mom, t_approx), L.p.mom, h);
            if (!found) h.t = 1.f;
            if (refine_again(P, h, t_approx)) {
                trav_begin(v, g, P.tmax, stk, stride, P.stack_cap, TN);
            } else {
                if (t_approx != NOT_REFINED) h.t = h.t + t_approx;
                t_approx = NOT_REFINED;
                if (shade<DBG>(P, L, h, found) && goes_on(P, L)) {
                    trav_begin(v, g, P.tmax, stk, stride, P.stack_cap, TN);
                } else {
                    end_photon<DBG>(P, L);
                    add_steps(steps, L.bounce, [&](uint32_t n) __attribute__((always_inline)) { atomicAdd(P.counters + 0, (unsigned long long)n); });
                    v.cur = TRAV_IDLE;
                }
            }
        }
        const uint64_t idle = __ballot(v.cur == TRAV_IDLE);
        const int nidle = __popcll(idle);
        if (drained) {
            if (nidle == 64) break;
            continue;
        }
        if (nidle > 0 && (nidle >= P.refill_threshold || nidle == 64)) {
            // The wave's idle lanes take the next photons: the first time those of the lanes'
            // numbers in the grid, then photons the wave has claimed with an add on the queue
            // counter (which counts on from the first ones), 64 at a time while the queue holds
            // many, else just what the lanes need. The adds of all waves meet at one address:
            // with one per refill (177,000 in the calorimeter event) they bound that event,
            // 3.03 against 2.35 ms.
            const unsigned long long nfirst = (unsigned long long)gridDim.x * blockDim.x;
            unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
            if (first) {
                first = false;
                drained = !REFILL || nfirst >= (unsigned long long)P.num_photon;
            } else {
                const int rank = int(__builtin_amdgcn_mbcnt_hi(uint32_t(idle >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(idle), 0u)));
                const int more = nidle - pooled;
                i = pool + (unsigned long long)rank;
                if (more > 0) {
                    const bool many = pool + 2ull * nfirst < (unsigned long long)P.num_photon;
                    const int take = many ? max(more, 64) : more;
                    unsigned long long base = 0;
                    if (lane == 0) base = atomicAdd(P.counters + 1, (unsigned long long)take);
                    base = __shfl(base, 0, 64) + nfirst;
                    if (rank >= pooled) i = base + (unsigned long long)(rank - pooled);
                    pool = base + (unsigned long long)more;
                    pooled = take - more;
                } else {
                    pool += (unsigned long long)nidle;
                    pooled -= nidle;
                }
                drained = pool >= (unsigned long long)P.num_photon;
            }
            if (v.cur == TRAV_IDLE && i < (unsigned long long)P.num_photon) {
                const long long pi = REFILL && P.perm ? (long long)P.perm[i] : (long long)i;
                if (start_photon<DBG>(P, L, pi)) {
                    if (goes_on(P, L)) { trav_begin(v, g, P.tmax, stk, stride, P.stack_cap, TN); t_approx = NOT_REFINED; }
                    else end_photon<DBG>(P, L);
                } else {
                    P.hitflag[pi] = 0;
                }
            }
            far_wave = __ballot(v.cur != TRAV_IDLE && far_away(g, L.p.pos)) != 0ull;
        }
    }
    flush_counters(P, steps, cnt.visits, cnt.tests, err, COUNT, cnt.csgb, cnt.ivis);
}

// ------------------------------------------------------------------ plain form
// one lane per photon, no refill
template <bool FP64, bool COUNT, bool DBG, bool LIST, int TM>
__global__ void __launch_bounds__(256, OXR_PLAIN_WAVES) k_simulate(Params P) {
    extern __shared__ int4 smem4[];
    BNode* top = reinterpret_cast<BNode*>(smem4);
    int* stk = reinterpret_cast<int*>(top + P.ntop) + threadIdx.x;
    stage_top(P, top, P.ntop);
    stage_csg<TM>(P);
    __syncthreads();
    run_wave<FP64, COUNT, DBG, LIST, TM, false>(P, stk, blockDim.x, top);
}

// ------------------------------------------------------------------ persistent form
// A fixed grid whose lanes take photons from a queue: the first by their number in the grid
// (an add on the queue counter by every wave at once takes tens of microseconds), later
// ones when at least refill_threshold lanes of a wave are idle (or all are), claimed with one
// atomicAdd on counters[1]; with P.perm the k-th claim is photon P.perm[k] (a sorted
// order), else photon k. Every wave leaves the loop once the queue has passed num_photon
// and its lanes are idle.
template <bool FP64, bool DBG, bool LIST, int TM>
__global__ void __launch_bounds__(256, OXR_PERSIST_WAVES) k_simulate_persist(Params P) {
    extern __shared__ int4 smem4[];
    BNode* top = reinterpret_cast<BNode*>(smem4);
    int* stk = reinterpret_cast<int*>(top + P.ntop) + threadIdx.x;
    stage_top(P, top, P.ntop);
    stage_csg<TM>(P);
    __syncthreads();
    run_wave<FP64, false, DBG, LIST, TM, true>(P, stk, blockDim.x, top);
}

} // namespace oxd

namespace oxl {

// kind: SIM_PROD (production), SIM_DEBUG (seqhis, records, precooked streams), SIM_COUNT
// (visit counting, generating in place like the debug variants). tm: traversal mode bits
// (oxd kernels above); debug launches use the node-index stack without radial culling,
// counting launches the production traversal without the register CSG stacks (which
// change no visit), so they count the visits the production launch makes.
template <bool FP64, bool LIST>
hipError_t launch_simulate_plain(hipStream_t s, const oxd::Params& P, dim3 g, dim3 b, size_t sm, int kind, int tm) {
#define OXR_PLAIN(C, D, T) hipLaunchKernelGGL((oxd::k_simulate<FP64, C, D, LIST, T>), g, b, sm, s, P)
    if (kind == SIM_COUNT) {
        switch (tm & 11) {
            case 0: OXR_PLAIN(true, true, 0); break;
            case 1: OXR_PLAIN(true, true, 1); break;
            case 2: OXR_PLAIN(true, true, 2); break;
            case 3: OXR_PLAIN(true, true, 3); break;
            case 8: OXR_PLAIN(true, true, 8); break;
            case 9: OXR_PLAIN(true, true, 9); break;
            case 10: OXR_PLAIN(true, true, 10); break;
            default: OXR_PLAIN(true, true, 11); break;
        }
    } else if (kind == SIM_DEBUG) {
        if (tm & 2) OXR_PLAIN(false, true, 2);
        else OXR_PLAIN(false, true, 0);
    } else {
        switch (tm & 11) {
            case 0: if ((tm & 4) && !LIST) OXR_PLAIN(false, false, 4 * !LIST); else OXR_PLAIN(false, false, 0); break;
            case 1: if ((tm & 4) && !LIST) OXR_PLAIN(false, false, 1 + 4 * !LIST); else OXR_PLAIN(false, false, 1); break;
            case 2: if ((tm & 4) && !LIST) OXR_PLAIN(false, false, 2 + 4 * !LIST); else OXR_PLAIN(false, false, 2); break;
            case 3: if ((tm & 4) && !LIST) OXR_PLAIN(false, false, 3 + 4 * !LIST); else OXR_PLAIN(false, false, 3); break;
            case 8: if ((tm & 4) && !LIST) OXR_PLAIN(false, false, 8 + 4 * !LIST); else OXR_PLAIN(false, false, 8); break;
            case 9: if ((tm & 4) && !LIST) OXR_PLAIN(false, false, 9 + 4 * !LIST); else OXR_PLAIN(false, false, 9); break;
            case 10: if ((tm & 4) && !LIST) OXR_PLAIN(false, false, 10 + 4 * !LIST); else OXR_PLAIN(false, false, 10); break;
            default: if ((tm & 4) && !LIST) OXR_PLAIN(false, false, 11 + 4 * !LIST); else OXR_PLAIN(false, false, 11); break;
        }
    }
#undef OXR_PLAIN
    return hipGetLastError();
}

// the persistent kernel instance launch_simulate_persist runs for (debug, tm)
template <bool FP64, bool LIST>
const void* persist_kernel(bool debug, int tm) {
#define OXR_K(D, T) reinterpret_cast<const void*>(&oxd::k_simulate_persist<FP64, D, LIST, T>)
    if (debug) return (tm & 2) ? OXR_K(true, 2) : OXR_K(true, 0);
    const bool sh = (tm & 4) && !LIST;
    switch (tm & 11) {
        case 0: return sh ? OXR_K(false, 4 * !LIST) : OXR_K(false, 0);
        case 1: return sh ? OXR_K(false, 1 + 4 * !LIST) : OXR_K(false, 1);
        case 2: return sh ? OXR_K(false, 2 + 4 * !LIST) : OXR_K(false, 2);
        case 3: return sh ? OXR_K(false, 3 + 4 * !LIST) : OXR_K(false, 3);
        case 8: return sh ? OXR_K(false, 8 + 4 * !LIST) : OXR_K(false, 8);
        case 9: return sh ? OXR_K(false, 9 + 4 * !LIST) : OXR_K(false, 9);
        case 10: return sh ? OXR_K(false, 10 + 4 * !LIST) : OXR_K(false, 10);
        default: return sh ? OXR_K(false, 11 + 4 * !LIST) : OXR_K(false, 11);
    }
#undef OXR_K
}

template <bool FP64, bool LIST>
hipError_t launch_simulate_persist(hipStream_t s, const oxd::Params& P, dim3 g, dim3 b, size_t sm, bool debug, int tm) {
#define OXR_PERSIST(D, T) hipLaunchKernelGGL((oxd::k_simulate_persist<FP64, D, LIST, T>), g, b, sm, s, P)
    if (debug) {
        if (tm & 2) OXR_PERSIST(true, 2);
        else OXR_PERSIST(true, 0);
    } else {
        switch (tm & 11) {
            case 0: if ((tm & 4) && !LIST) OXR_PERSIST(false, 4 * !LIST); else OXR_PERSIST(false, 0); break;
            case 1: if ((tm & 4) && !LIST) OXR_PERSIST(false, 1 + 4 * !LIST); else OXR_PERSIST(false, 1); break;
            case 2: if ((tm & 4) && !LIST) OXR_PERSIST(false, 2 + 4 * !LIST); else OXR_PERSIST(false, 2); break;
            case 3: if ((tm & 4) && !LIST) OXR_PERSIST(false, 3 + 4 * !LIST); else OXR_PERSIST(false, 3); break;
            case 8: if ((tm & 4) && !LIST) OXR_PERSIST(false, 8 + 4 * !LIST); else OXR_PERSIST(false, 8); break;
            case 9: if ((tm & 4) && !LIST) OXR_PERSIST(false, 9 + 4 * !LIST); else OXR_PERSIST(false, 9); break;
            case 10: if ((tm & 4) && !LIST) OXR_PERSIST(false, 10 + 4 * !LIST); else OXR_PERSIST(false, 10); break;
            default: if ((tm & 4) && !LIST) OXR_PERSIST(false, 11 + 4 * !LIST); else OXR_PERSIST(false, 11); break;
        }
    }
#undef OXR_PERSIST
    return hipGetLastError();
}

template <int BASE>
hipError_t launch_simulate_simple(hipStream_t s, const oxd::Params& P, dim3 g, dim3 b, size_t sm, bool persist, int tm) {
#define OXR_S(T)                                                                                          \
    do {                                                                                                  \
        if (persist) hipLaunchKernelGGL((oxd::k_simulate_persist<false, false, false, BASE + T>), g, b, sm, s, P); \
        else hipLaunchKernelGGL((oxd::k_simulate<false, false, false, false, BASE + T>), g, b, sm, s, P);  \
    } while (0)
    switch (tm & 15) {
        case 0: OXR_S(0); break;   case 1: OXR_S(1); break;   case 2: OXR_S(2); break;   case 3: OXR_S(3); break;
        case 4: OXR_S(4); break;   case 5: OXR_S(5); break;   case 6: OXR_S(6); break;   case 7: OXR_S(7); break;
        case 8: OXR_S(8); break;   case 9: OXR_S(9); break;   case 10: OXR_S(10); break; case 11: OXR_S(11); break;
        case 12: OXR_S(12); break; case 13: OXR_S(13); break; case 14: OXR_S(14); break; default: OXR_S(15); break;
    }
#undef OXR_S
    return hipGetLastError();
}

template <int BASE>
const void* persist_kernel_simple(int tm) {
#define OXR_K(T) return reinterpret_cast<const void*>(&oxd::k_simulate_persist<false, false, false, BASE + T>)
    switch (tm & 15) {
        case 0: OXR_K(0);   case 1: OXR_K(1);   case 2: OXR_K(2);   case 3: OXR_K(3);
        case 4: OXR_K(4);   case 5: OXR_K(5);   case 6: OXR_K(6);   case 7: OXR_K(7);
        case 8: OXR_K(8);   case 9: OXR_K(9);   case 10: OXR_K(10); case 11: OXR_K(11);
        case 12: OXR_K(12); case 13: OXR_K(13); case 14: OXR_K(14); default: OXR_K(15);
    }
#undef OXR_K
}

} // namespace oxl
