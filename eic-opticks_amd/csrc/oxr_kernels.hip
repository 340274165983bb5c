// oxr_kernels.hip -- gfx950 kernels of the engine and their host-side launchers.
//
//   k_fill_seed        per-photon genstep index (QEvt.cu:181-237 reduce + iexpand)
//   k_generate         production launches: every photon generated by one coherent
//                      pass; writes the photon and its RNG resume point
//   k_simulate         plain form: one lane per photon, CSGOptiX7.cu:405-503 shape
//   k_simulate_persist persistent form: a fixed grid whose lanes refill from a device
//                      photon counter between bounce steps (wave-aggregated atomics)
//                      (both in oxr_sim.h, instantiated in oxr_sim_*.hip)
// Production variants (DBG=false) resume photons that k_generate made; the debug
// variants (seqhis, records, precooked streams, counting) generate in place.
//   k_count/k_group/k_select/k_scatter_lite  ordered hit compaction (SU::count_if/copy_if, SU.cu:49-166)
//   k_trace_rays, k_intersect_prim  geometry queries
//   k_simtrace                      2-D cross-section rays from FRAME gensteps (CSGOptiX7.cu:536-577)
#include "oxr_sim.h"
#include <hipcub/hipcub.hpp>
#include <algorithm>

namespace oxd {

// ------------------------------------------------------------------ seeding
__global__ void k_fill_seed(const long long* __restrict__ offsets, int num_gs, int* __restrict__ seed, long long n) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    seed[i] = genstep_of(offsets, num_gs, i);
}

// ------------------------------------------------------------------ generation
// One lane per photon, every lane generating: the genstep dispatch and the rejection
// loops run coherently here instead of inside the bounce loop.
__global__ void __launch_bounds__(256) k_generate(Params P) {
    long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= P.num_photon) return;
    Lane L;
    if (begin_photon<false>(P, L, idx)) {
        store_photon(P.photon + 4 * idx, L.p);
        P.rstate[idx] = make_ulonglong2(L.r.pos, ((unsigned long long)L.r.p1 << 32) | L.r.p0);
    } else {
        P.rstate[idx] = make_ulonglong2(~0ull, 0ull);
        P.hitflag[idx] = 0;
    }
}

// ------------------------------------------------------------------ hit compaction
constexpr int CHUNK = 4096;   // photons per compaction block (256 lanes x 16)

// one 16-byte load per lane where the flags allow it (each flag byte is 0 or 1)
__global__ void __launch_bounds__(256) k_count(const uint8_t* __restrict__ flag, long long n, int* __restrict__ counts) {
    long long base = (long long)blockIdx.x * CHUNK;
    int c = 0;
    if (base + CHUNK <= n && (reinterpret_cast<uintptr_t>(flag) & 15u) == 0u) {
        const uint4 w = reinterpret_cast<const uint4*>(flag + base)[threadIdx.x];
        c = __popc(w.x) + __popc(w.y) + __popc(w.z) + __popc(w.w);
    } else {
        for (int k = threadIdx.x; k < CHUNK; k += 256) {
            long long i = base + k;
            if (i < n && flag[i]) c++;
        }
    }
    c = (int)wave_sum((unsigned long long)c);
    __shared__ int ws[4];
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

// Sums of the counts of 256 blocks each, for launches of many blocks.
constexpr int GROUP = 256;
__global__ void __launch_bounds__(GROUP) k_group(const int* __restrict__ counts, int nb, int* __restrict__ groups) {
    const int b = blockIdx.x * GROUP + threadIdx.x;
    const unsigned long long c = wave_sum((unsigned long long)(b < nb ? counts[b] : 0));
    __shared__ int ws[GROUP / 64];
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = int(c);
    __syncthreads();
    if (threadIdx.x == 0) groups[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

// The hits in photon order. Each block sums the counts of the blocks before it (with groups,
// of its own group's blocks and the sums of the groups before) instead of waiting for a scan
// kernel, and notes its offset for k_scatter_lite. What the host reads after a launch - the launch counters, the hit count and the
// first hits - is also written straight to pinned host memory (pub), so a launch ends without
// copy commands; the counters are left zero for the next launch.
__global__ void __launch_bounds__(256) k_select(const uint8_t* __restrict__ flag, const float4* __restrict__ photon, long long n,
                                                const int* __restrict__ counts, const int* __restrict__ groups,
                                                long long* __restrict__ offs, float4* __restrict__ hit, long long hit_cap,
                                                unsigned long long* ctr, LaunchResult* pub) {
    __shared__ unsigned long long part[4];
    __shared__ int ws[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    unsigned long long before = 0;
    const unsigned group = groups ? blockIdx.x / GROUP : 0u;
    for (unsigned g = threadIdx.x; g < group; g += 256) before += (unsigned long long)groups[g];
    for (unsigned b = group * GROUP + threadIdx.x; b < blockIdx.x; b += 256) before += (unsigned long long)counts[b];
    before = wave_sum(before);
    if (lane == 0) part[w] = before;
    __syncthreads();
    long long o = (long long)(part[0] + part[1] + part[2] + part[3]);
    const bool last = blockIdx.x == gridDim.x - 1;
    const long long total = last ? o + counts[blockIdx.x] : 0;
    if (threadIdx.x == 0) {
        offs[blockIdx.x] = o;
        if (last) offs[gridDim.x] = total;
    }
    if (last && pub) {
        if (threadIdx.x < 8) {
            pub->counters[threadIdx.x] = ctr[threadIdx.x];
            ctr[threadIdx.x] = 0ull;
        }
        if (threadIdx.x == 0) pub->num_hit = total;
    }
    const long long base = (long long)blockIdx.x * CHUNK;
    for (int k = 0; k < CHUNK && base + k < n; k += 256) {
        long long i = base + k + threadIdx.x;
        bool f = i < n && flag[i];
        uint64_t m = __ballot(f);
        unsigned rank = __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
        if (lane == 0) ws[w] = __popcll(m);
        __syncthreads();
        int ahead = 0;
        for (int q = 0; q < w; q++) ahead += ws[q];
        int tot = ws[0] + ws[1] + ws[2] + ws[3];
        if (f) {
            const long long dst = o + ahead + rank;
            const float4* src = photon + 4 * i;
            const float4 v0 = src[0], v1 = src[1], v2 = src[2], v3 = src[3];
            if (dst < hit_cap) {
                float4* d = hit + 4 * dst;
                d[0] = v0; d[1] = v1; d[2] = v2; d[3] = v3;
            }
            if (pub && dst < LaunchResult::HITS) {
                float4* d = pub->hit + 4 * dst;
                d[0] = v0; d[1] = v1; d[2] = v2; d[3] = v3;
            }
        }
        o += tot;
        __syncthreads();
    }
}

// the same selection of the photonlite items by the offsets k_select left
__global__ void __launch_bounds__(256) k_scatter_lite(const uint8_t* __restrict__ flag, const uint4* __restrict__ lite,
                                                      long long n, const long long* __restrict__ offs,
                                                      uint4* __restrict__ hitlite, long long hit_cap) {
    __shared__ int ws[4];
    long long base = (long long)blockIdx.x * CHUNK;
    long long o = offs[blockIdx.x];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int k = 0; k < CHUNK; k += 256) {
        long long i = base + k + threadIdx.x;
        bool f = i < n && flag[i];
        uint64_t m = __ballot(f);
        unsigned rank = __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
        if (lane == 0) ws[w] = __popcll(m);
        __syncthreads();
        int before = 0;
        for (int q = 0; q < w; q++) before += ws[q];
        int tot = ws[0] + ws[1] + ws[2] + ws[3];
        if (f) {
            long long dst = o + before + rank;
            if (dst < hit_cap) hitlite[dst] = lite[i];
        }
        o += tot;
        __syncthreads();
    }
}

// Serving form's compaction: the same ordered selection, published straight to pinned
// host memory so a finished step needs no copy command. k_scan_host scans the per-block counts in
// one 256-lane workgroup and also writes the offsets and the step's 8 launch counters to the host.
// k_scatter_host stages each 256-photon group's hits in LDS and writes them as one
// contiguous run, so the PCIe writes are whole lines: rows below hcap go to the host
// block, any beyond it to the device buffer at the same row (the host fetches those).
__global__ void __launch_bounds__(256) k_scan_host(const int* __restrict__ counts, int nb, long long* __restrict__ out,
                                                   long long* __restrict__ host_out,
                                                   const unsigned long long* __restrict__ ctr,
                                                   unsigned long long* __restrict__ host_ctr) {
    __shared__ long long part[256];
    long long carry = 0;
    for (int base = 0; base < nb; base += 256) {
        int i = base + threadIdx.x;
        long long v = i < nb ? counts[i] : 0;
        part[threadIdx.x] = v;
        __syncthreads();
        for (int off = 1; off < 256; off <<= 1) {
            long long add = threadIdx.x >= off ? part[threadIdx.x - off] : 0;
            __syncthreads();
            part[threadIdx.x] += add;
            __syncthreads();
        }
        if (i < nb) {
            long long x = carry + part[threadIdx.x] - v;
            out[i] = x;
            host_out[i] = x;
        }
        long long tot = part[255];
        __syncthreads();
        carry += tot;
    }
    if (threadIdx.x == 0) { out[nb] = carry; host_out[nb] = carry; }
    if (threadIdx.x < 8) host_ctr[threadIdx.x] = ctr[threadIdx.x];
}

__global__ void __launch_bounds__(256) k_scatter_host(const uint8_t* __restrict__ flag, const float4* __restrict__ photon,
                                                      long long n, const long long* __restrict__ offs,
                                                      float4* __restrict__ hhit, long long hcap,
                                                      float4* __restrict__ dhit, long long dcap) {
    __shared__ float4 rows[256 * 4];
    __shared__ int ws[4];
    long long base = (long long)blockIdx.x * CHUNK;
    long long o = offs[blockIdx.x];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int k = 0; k < CHUNK; k += 256) {
        long long i = base + k + threadIdx.x;
        bool f = i < n && flag[i];
        uint64_t m = __ballot(f);
        unsigned rank = __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
        if (lane == 0) ws[w] = __popcll(m);
        __syncthreads();
        int before = 0;
        for (int q = 0; q < w; q++) before += ws[q];
        int tot = ws[0] + ws[1] + ws[2] + ws[3];
        if (f) {
            const float4* src = photon + 4 * i;
            int r = before + (int)rank;
#pragma unroll
            for (int q = 0; q < 4; q++) rows[4 * r + q] = src[q];
        }
        __syncthreads();
        for (int j = threadIdx.x; j < 4 * tot; j += 256) {
            long long row = o + (j >> 2);
            if (row < hcap) hhit[4 * o + j] = rows[j];
            else if (row < dcap) dhit[4 * o + j] = rows[j];
        }
        o += tot;
        __syncthreads();
    }
}

// ------------------------------------------------------------------ queries
template <bool FP64, bool LIST, bool FLAT>
__global__ void __launch_bounds__(256) k_trace_rays(Params P, const float4* __restrict__ rays, long long n, float4* __restrict__ prd) {
    extern __shared__ int4 smem4[];
    BNode* top = reinterpret_cast<BNode*>(smem4);
    int* stk = reinterpret_cast<int*>(top + P.ntop) + threadIdx.x;
    stage_top(P, top, P.ntop);
    __syncthreads();
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 a = rays[2 * i], b = rays[2 * i + 1];
    Hit h;
    bool found = trace<FP64, LIST, FLAT>(P.g, mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), a.w, b.w, h, stk, blockDim.x, P.stack_cap,
                                         top, P.ntop);
    float lc = 0.f, lf = 0.f;
    if (found) {
        lc = h.lpos.z / sqrtf(dot(h.lpos, h.lpos));
        lf = (xatan2(h.lpos.y, h.lpos.x) + PIf) / (2.0f * PIf);
    }
    prd[2 * i] = make_float4(h.n.x, h.n.y, h.n.z, h.t);
    prd[2 * i + 1] = make_float4(lc, lf, __uint_as_float(h.ii_id), __uint_as_float(h.gpbd));
}

// simtrace: one ray per slot of the FRAME gensteps (qsim::generate_photon_simtrace_frame,
// qudarap/qsim.h:2459-2510: start at the genstep's local position, direction from two
// uniforms in the grid plane or over the sphere, both through the genstep's 4x4
// transform), traced like CSGOptiX7.cu:536-577 and written as sevent::add_simtrace
// (sysrap/sevent.h:670-696): {normal, t}, {pos + t dir, tmin}, {pos, gpbd}, {dir, iindex_identity},
// refined like the simulate traces when PropagateRefine is on.
// The stream of slot i is the photon stream of index i at uniform 0 (rng init(rng, 0, i)).
template <bool FP64, bool LIST, bool FLAT>
__global__ void __launch_bounds__(256) k_simtrace(Params P, const float4* __restrict__ gs, const long long* __restrict__ offsets,
                                                  int num_gs, long long n, float4* __restrict__ out) {
    extern __shared__ int4 smem4[];
    BNode* top = reinterpret_cast<BNode*>(smem4);
    int* stk = reinterpret_cast<int*>(top + P.ntop) + threadIdx.x;
    stage_top(P, top, P.ntop);
    __syncthreads();
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4* q = gs + 6 * genstep_of(offsets, num_gs, i);
    const int gridaxes = __float_as_int(q[0].y);
    Rng r;
    rng_init(r, P.rng_seed, 0ull, 0ull, 0ull, (unsigned long long)i);
    float u0, u1;
    draw2(r, u0, u1);
    float ph = 2.f * PIf * u0;
    float sinPhi, cosPhi;
    sincos_bounded(ph, sinPhi, cosPhi);
    float cosTheta = 2.f * u1 - 1.f;
    float sinTheta = sqrtf(1.f - cosTheta * cosTheta);
    f3 d;
    switch (gridaxes) {
        case 1: d = mk(0.f, cosPhi, sinPhi); break;                                  // YZ
        case 2: d = mk(cosPhi, 0.f, sinPhi); break;                                  // XZ
        case 3: d = mk(cosPhi, sinPhi, 0.f); break;                                  // XY
        default: d = mk(sinTheta * cosPhi, sinTheta * sinPhi, cosTheta); break;      // XYZ
    }
    const float4 m0 = q[2], m1 = q[3], m2 = q[4], m3 = q[5];   // qat4 rows, translation in m3
    const float px = q[1].x, py = q[1].y, pz = q[1].z;
    f3 o = mk(m0.x * px + m1.x * py + m2.x * pz + m3.x * 1.f,
                  m0.y * px + m1.y * py + m2.y * pz + m3.y * 1.f,
                  m0.z * px + m1.z * py + m2.z * pz + m3.z * 1.f);
    f3 v = mk(m0.x * d.x + m1.x * d.y + m2.x * d.z + m3.x * 0.f,
                  m0.y * d.x + m1.y * d.y + m2.y * d.z + m3.y * 0.f,
                  m0.z * d.x + m1.z * d.y + m2.z * d.z + m3.z * 0.f);
    Hit h;
    float t_approx = NOT_REFINED;
    bool found;
    do {
        found = trace<FP64, LIST, FLAT>(P.g, ray_origin(o, v, t_approx), v, P.tmin, P.tmax, h, stk, blockDim.x, P.stack_cap, top, P.ntop);
        if (!found) h.t = 1.f;
    } while (refine_again(P, h, t_approx));
    if (t_approx != NOT_REFINED) h.t = h.t + t_approx;
    // a miss carries the miss program's q0: the mid-grey background as normal, distance 1
    // (CSGOptiX7.cu:655-682 with SBT::updateMiss, SBT.cc:180-192)
    if (!found) h.n = mk(0.6f, 0.6f, 0.6f);
    const float t = h.t;
    out[4 * i + 0] = make_float4(h.n.x, h.n.y, h.n.z, t);
    out[4 * i + 1] = make_float4(o.x + t * v.x, o.y + t * v.y, o.z + t * v.z, P.tmin);
    out[4 * i + 2] = make_float4(o.x, o.y, o.z, __uint_as_float(h.gpbd));
    out[4 * i + 3] = make_float4(v.x, v.y, v.z, __uint_as_float(h.ii_id));
}

template <bool FP64, bool LIST>
__global__ void __launch_bounds__(256) k_intersect_prim(Geom g, int root, const float4* __restrict__ rays, long long n,
                                                         float4* __restrict__ isect, int* __restrict__ valid) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 a = rays[2 * i], b = rays[2 * i + 1];
    Is is;
    bool v = intersect_prim<FP64, LIST>(is, g.node, root, g.plan, g.itra, a.w, mk(a.x, a.y, a.z), mk(b.x, b.y, b.z));
    isect[i] = make_float4(is.x, is.y, is.z, is.w);
    valid[i] = v ? 1 : 0;
}

} // namespace oxd

// ====================================================================== launchers
namespace oxl {
using namespace oxd;

hipError_t fill_seed(hipStream_t s, const long long* offsets, int num_gs, int* seed, long long n) {
    if (n <= 0) return hipSuccess;
    long long nb = (n + 255) / 256;
    hipLaunchKernelGGL(k_fill_seed, dim3((unsigned)nb), dim3(256), 0, s, offsets, num_gs, seed, n);
    return hipGetLastError();
}

size_t simulate_smem(const Params& P, int block) {
    return size_t(P.ntop) * sizeof(BNode) + size_t(block) * P.stack_cap * (P.tn_stack ? 8 : 4) +
           size_t(P.csg_node4 + P.csg_itra4) * sizeof(float4) + size_t(P.csg_prim) * sizeof(int2);
}

// debug outputs (seqhis, records, precooked streams) select the DBG kernel variants
static bool wants_debug(const Params& P) {
    return P.seq || P.record || P.rec || P.prd || P.pre || P.bounce_out || P.overflow_out || P.lite;
}

bool needs_generate(const Params& P, bool count) { return !count && !wants_debug(P) && !P.gen_inplace; }

hipError_t generate(hipStream_t s, const Params& P) {
    if (P.num_photon <= 0) return hipSuccess;
    long long nb = (P.num_photon + 255) / 256;
    hipLaunchKernelGGL(k_generate, dim3((unsigned)nb), dim3(256), 0, s, P);
    return hipGetLastError();
}

static int trav_mode(const Params& P) { return (P.tn_stack ? 1 : 0) | (P.g.flat ? 2 : 0) | (P.radial ? 8 : 0); }

// kernel variants: FP64 roots, list-node support
#define OXR_B2(a, b, K, ...)                                             \
    do {                                                                 \
        if (a) { if (b) K(true, true, __VA_ARGS__); else K(true, false, __VA_ARGS__); } \
        else   { if (b) K(false, true, __VA_ARGS__); else K(false, false, __VA_ARGS__); } \
    } while (0)

// The distance-carrying traversal stack (P.tn_stack) is compiled into the production and
// counting variants (the counting launch counts the visits the production traversal
// makes); debug launches use the plain stack. Register-resident CSG stacks
// (P.shallow_csg) are compiled into the production variants without list nodes only:
// they give the same intersects as the private-memory stacks of the other variants.
hipError_t simulate_plain(hipStream_t s, const Params& P0, int block, bool fp64, bool count, bool list) {
    if (P0.num_photon <= 0) return hipSuccess;
    Params P = P0;
    if (wants_debug(P)) P.tn_stack = 0;
    const int kind = count ? SIM_COUNT : wants_debug(P) ? SIM_DEBUG : SIM_PROD;
    const bool simple = kind == SIM_PROD && P.simple_leaves && !fp64 && !list;
    if (!simple) P.csg_node4 = P.csg_itra4 = P.csg_prim = 0;   // only the simple-leaf kernels read the LDS copy
    long long nb = (P.num_photon + block - 1) / block;
    size_t sm = simulate_smem(P, block);
    dim3 g((unsigned)nb), b(block);
    const int tm = trav_mode(P) | (kind == SIM_PROD && P.shallow_csg && !list ? 4 : 0);
    if (simple) return P.csg_node4 > 0 ? launch_simulate_simple<48>(s, P, g, b, sm, false, tm)
                                       : launch_simulate_simple<16>(s, P, g, b, sm, false, tm);
    if (fp64) return list ? launch_simulate_plain<true, true>(s, P, g, b, sm, kind, tm)
                          : launch_simulate_plain<true, false>(s, P, g, b, sm, kind, tm);
    return list ? launch_simulate_plain<false, true>(s, P, g, b, sm, kind, tm)
                : launch_simulate_plain<false, false>(s, P, g, b, sm, kind, tm);
}

hipError_t simulate_persist(hipStream_t s, const Params& P0, int block, int grid, bool fp64, bool list) {
    if (P0.num_photon <= 0) return hipSuccess;
    Params P = P0;
    const bool debug = wants_debug(P);
    if (debug) P.tn_stack = 0;
    const bool simple = !debug && P.simple_leaves && !fp64 && !list;
    if (!simple) P.csg_node4 = P.csg_itra4 = P.csg_prim = 0;
    size_t sm = simulate_smem(P, block);
    // no more workgroups than the photons fill: idle ones would stage the tree and add to the
    // counters for nothing (ten photons: 58 us with 768 workgroups, 35 with one)
    dim3 g((unsigned)std::min<long long>(grid, (P.num_photon + block - 1) / block)), b(block);
    const int tm = trav_mode(P) | (!debug && P.shallow_csg && !list ? 4 : 0);
    if (simple) return P.csg_node4 > 0 ? launch_simulate_simple<48>(s, P, g, b, sm, true, tm)
                                       : launch_simulate_simple<16>(s, P, g, b, sm, true, tm);
    if (fp64) return list ? launch_simulate_persist<true, true>(s, P, g, b, sm, debug, tm)
                          : launch_simulate_persist<true, false>(s, P, g, b, sm, debug, tm);
    return list ? launch_simulate_persist<false, true>(s, P, g, b, sm, debug, tm)
                : launch_simulate_persist<false, false>(s, P, g, b, sm, debug, tm);
}

int persist_occupancy(const Params& P0, int block, bool fp64, bool list) {
    Params P = P0;
    const bool debug = wants_debug(P);
    if (debug) P.tn_stack = 0;
    const bool simple = !debug && P.simple_leaves && !fp64 && !list;
    if (!simple) P.csg_node4 = P.csg_itra4 = P.csg_prim = 0;
    size_t sm = simulate_smem(P, block);
    const int tm = trav_mode(P) | (!debug && P.shallow_csg && !list ? 4 : 0);
    const void* f = simple ? (P.csg_node4 > 0 ? persist_kernel_simple<48>(tm) : persist_kernel_simple<16>(tm))
                  : fp64 ? (list ? persist_kernel<true, true>(debug, tm) : persist_kernel<true, false>(debug, tm))
                         : (list ? persist_kernel<false, true>(debug, tm) : persist_kernel<false, false>(debug, tm));
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, block, sm) != hipSuccess) return -1;
    return n;
}

bool production_kernels(const Params& P) { return !wants_debug(P); }

// photon claim order: the generated direction's cell on the octahedral map (|x|+|y|+|z| = 1
// folded onto the square), 256 x 256 cells in Morton order so neighbouring directions get
// neighbouring keys, under the genstep index (one origin per genstep for point sources)
OXD unsigned spread8(unsigned x) {
    x &= 0xffu;
    x = (x | (x << 4)) & 0x0f0fu;
    x = (x | (x << 2)) & 0x3333u;
    x = (x | (x << 1)) & 0x5555u;
    return x;
}

__global__ void __launch_bounds__(256) k_order_key(const float4* __restrict__ photon, const int* __restrict__ seed, long long n,
                                                   unsigned long long* __restrict__ key, unsigned* __restrict__ val) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 m = photon[4 * i + 1];
    const float sc = 1.f / (fabsf(m.x) + fabsf(m.y) + fabsf(m.z) + 1e-30f);
    float u = m.x * sc, v = m.y * sc;
    if (m.z < 0.f) {
        const float uu = (1.f - fabsf(v)) * (u >= 0.f ? 1.f : -1.f), vv = (1.f - fabsf(u)) * (v >= 0.f ? 1.f : -1.f);
        u = uu; v = vv;
    }
    const unsigned qu = min(255u, unsigned(fmaxf(0.f, (u * 0.5f + 0.5f) * 256.f)));
    const unsigned qv = min(255u, unsigned(fmaxf(0.f, (v * 0.5f + 0.5f) * 256.f)));
    key[i] = ((unsigned long long)unsigned(seed[i]) << 16) | (spread8(qu) | (spread8(qv) << 1));
    val[i] = unsigned(i);
}

hipError_t order_photons(hipStream_t s, const Params& P, int key_bits, unsigned long long* key, unsigned* val,
                         void* tmp, size_t* tmp_bytes, const unsigned** perm) {
    const long long n = P.num_photon;
    if (n <= 0 || n > 0x7fffffffll || !P.seed) return hipErrorInvalidValue;
    const int bits = std::min(64, std::max(16, key_bits));
    if (!tmp) {
        return hipcub::DeviceRadixSort::SortPairs(nullptr, *tmp_bytes, key, key + n, val, val + n, int(n), 0, bits, s);
    }
    hipLaunchKernelGGL(k_order_key, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, P.photon, P.seed, n, key, val);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    e = hipcub::DeviceRadixSort::SortPairs(tmp, *tmp_bytes, key, key + n, val, val + n, int(n), 0, bits, s);
    if (e != hipSuccess) return e;
    *perm = val + n;
    return hipSuccess;
}

int compact_blocks(long long n) { return int((n + CHUNK - 1) / CHUNK); }
int compact_counts(long long n) {
    const int nb = compact_blocks(n);
    return nb > COMPACT_GROUPED_FROM ? nb + (nb + GROUP - 1) / GROUP : nb;
}

hipError_t compact(hipStream_t s, const uint8_t* flag, const float4* photon, long long n, int* counts,
                   long long* offs, float4* hit, long long hit_cap, unsigned long long* ctr, LaunchResult* pub) {
    if (n <= 0) return hipSuccess;
    int nb = compact_blocks(n);
    hipLaunchKernelGGL(k_count, dim3(nb), dim3(256), 0, s, flag, n, counts);
    int* groups = nullptr;
    if (nb > COMPACT_GROUPED_FROM) {
        groups = counts + nb;
        hipLaunchKernelGGL(k_group, dim3(unsigned((nb + GROUP - 1) / GROUP)), dim3(GROUP), 0, s, counts, nb, groups);
    }
    hipLaunchKernelGGL(k_select, dim3(nb), dim3(256), 0, s, flag, photon, n, counts, groups, offs, hit, hit_cap, ctr, pub);
    return hipGetLastError();
}

hipError_t compact_host(hipStream_t s, const uint8_t* flag, const float4* photon, long long n, int* counts,
                        long long* offs, long long* host_offs, const unsigned long long* ctr,
                        unsigned long long* host_ctr, float4* hhit, long long hcap, float4* dhit, long long dcap) {
    if (n <= 0) return hipSuccess;
    int nb = compact_blocks(n);
    hipLaunchKernelGGL(k_count, dim3(nb), dim3(256), 0, s, flag, n, counts);
    hipLaunchKernelGGL(k_scan_host, dim3(1), dim3(256), 0, s, counts, nb, offs, host_offs, ctr, host_ctr);
    hipLaunchKernelGGL(k_scatter_host, dim3(nb), dim3(256), 0, s, flag, photon, n, offs, hhit, hcap, dhit, dcap);
    return hipGetLastError();
}

hipError_t scatter_lite(hipStream_t s, const uint8_t* flag, const uint4* lite, long long n, const long long* offs,
                        uint4* hitlite, long long hit_cap) {
    if (n <= 0) return hipSuccess;
    int nb = compact_blocks(n);
    hipLaunchKernelGGL(k_scatter_lite, dim3(nb), dim3(256), 0, s, flag, lite, n, offs, hitlite, hit_cap);
    return hipGetLastError();
}

hipError_t trace_rays(hipStream_t s, const Params& P, const float4* rays, long long n, float4* prd, bool fp64,
                      bool list) {
    if (n <= 0) return hipSuccess;
    long long nb = (n + 255) / 256;
    Params Q = P;
    Q.csg_node4 = Q.csg_itra4 = Q.csg_prim = 0;   // the trace kernels read the node arrays in place
    size_t sm = simulate_smem(Q, 256);
#define OXR_TRACE(F, L, X)                                                                                       \
    do {                                                                                                           \
        if (P.g.flat) hipLaunchKernelGGL((k_trace_rays<F, L, true>), dim3((unsigned)nb), dim3(256), sm, s, P, rays, n, prd); \
        else hipLaunchKernelGGL((k_trace_rays<F, L, false>), dim3((unsigned)nb), dim3(256), sm, s, P, rays, n, prd);         \
    } while (0)
    OXR_B2(fp64, list, OXR_TRACE, 0);
#undef OXR_TRACE
    return hipGetLastError();
}

hipError_t simtrace(hipStream_t s, const Params& P, const float4* gs, const long long* offsets, int num_gs, long long n,
                    float4* out, bool fp64, bool list) {
    if (n <= 0) return hipSuccess;
    long long nb = (n + 255) / 256;
    Params Q = P;
    Q.csg_node4 = Q.csg_itra4 = Q.csg_prim = 0;
    size_t sm = simulate_smem(Q, 256);
#define OXR_SIMTRACE(F, L, X)                                                                                               \
    do {                                                                                                                      \
        if (P.g.flat) hipLaunchKernelGGL((k_simtrace<F, L, true>), dim3((unsigned)nb), dim3(256), sm, s, P, gs, offsets, num_gs, n, out); \
        else hipLaunchKernelGGL((k_simtrace<F, L, false>), dim3((unsigned)nb), dim3(256), sm, s, P, gs, offsets, num_gs, n, out);         \
    } while (0)
    OXR_B2(fp64, list, OXR_SIMTRACE, 0);
#undef OXR_SIMTRACE
    return hipGetLastError();
}

hipError_t intersect_prim(hipStream_t s, const Geom& g, int root, const float4* rays, long long n, float4* isect,
                          int* valid, bool fp64, bool list) {
    if (n <= 0) return hipSuccess;
    long long nb = (n + 255) / 256;
#define OXR_ISECT(F, L, X) hipLaunchKernelGGL((k_intersect_prim<F, L>), dim3((unsigned)nb), dim3(256), 0, s, g, root, rays, n, isect, valid)
    OXR_B2(fp64, list, OXR_ISECT, 0);
#undef OXR_ISECT
    return hipGetLastError();
}

} // namespace oxl
