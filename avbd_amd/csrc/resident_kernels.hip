// resident_kernels.hip -- a whole stretch of iterations of the positional
// solve (every colour phase, Chebyshev step and dual update of
// VBDSolver::solve_Parallel, simulation/VBDSolver.hpp:48-103) in one launch, from
// LDS.
//
// Why: one launch per colour phase leaves a mesh of this size bound by the
// launches.  Each phase of the 32^3 cube (9,000 vertices) spends 3.5-5 us in
// dispatch, in the first dependent loads from caches that the kernel boundary
// has just invalidated, and in the drain, against about 2 us of arithmetic.
//
// One workgroup owns a patch of the mesh (resident.hpp): its tets, particles
// and contacts are loaded into LDS once per launch; the neighbouring
// particles (halo) are kept there as copies.  After solving its vertices of a
// colour a patch publishes those that other patches hold as halo, and before
// the next colour takes the neighbours' new positions; nothing else crosses
// workgroups, since the Chebyshev step of a halo copy is the same arithmetic
// on the same values as its owner's.
//
// What bounds it now is the chain of one phase: LDS reads of a lane's two or
// three incidences (2,400 cycles for wavefront 0 in FP64 at 8 lanes: nine
// positions and five constants each, by all wavefronts of the CU), their sum over
// the lanes and the 3x3 solve (600), sending (1,000), then waiting for the
// neighbours' words (2,100); 4 times per iteration.  Wavefronts wait two thirds of
// their cycles; the LDS pipe is active in 20 % of the CU's and a quarter of that
// is bank conflicts.  Loading the patch and the handshake take 45,000 cycles per
// launch, a residual check 17,000.
// One launch per phase before -> now: FP64 32^3 to a residual target 36.6 ->
// 14.4 us per iteration, checks every 10 included (18.8 with one launch per
// check); 64 FP64 cubes 48.5 -> 27.3 ms; FP32 32^3 step of 10 iterations 365 ->
// 215 us, 15^3 of 20 430 -> 242 us, 512 cubes of 4 to 16 cells 49.4 -> 39.7 ms per 10
// steps with the read-back.
//
// Exchange: every 32-bit piece of a position travels in an 8-byte word next
// to a 32-bit tag (the number of the exchange), written and read with relaxed
// agent-scope atomics.  A word is its own flag, so no fence, no cache
// write-back and no second round trip is needed: a reader polls the words
// themselves until every tag is the expected one.  A word cannot be
// overwritten before it has been read: its owner solves the vertex again only
// after it has received, in the same iteration, the results that its readers
// computed from it.
//
// Residual checks (ResidentCheck): a launch covers several check intervals.
// After each one every patch publishes the sum of its |r_v|^2 the same way,
// takes those of all patches of its cluster and adds them in one order, so all
// of them reach the same decision without a further exchange.  Two sets of
// words, used in turn: a patch that sends its sum for check k has read those of
// check k - 1, so the words of k - 1 are free once every sum of k has arrived.
//
// Waits end: the patches of a scene depend on each other, so they must all be
// running.  Each announces itself after loading its patch and waits until
// the cluster is complete (or has polled `gather_polls` times; the decision is
// one compare-and-swap word, the same for all).  A complete cluster's workgroups
// stay resident, so every later wait is for a running workgroup.  An incomplete
// cluster gives up before anything is written, and its first patch alone runs
// the scene from device memory.  Later waits are bounded as well (they set
// status bit 1 and go on).  Waits are counted in polls (0.12 us each from an
// otherwise idle memory) and not by the clock, which runs on while the process is
// switched out.
//
// The arithmetic of an item is that of the per-phase kernels (tet_device.hpp:
// L lanes per vertex, the same incidence order and lane sums), so results
// do not depend on the partition and equal the per-phase kernels' bit for bit
// at the same L.
#include "resident.hpp"
#include "tet_device.hpp"
#include "tet_device_f64.hpp"

namespace avbd {

namespace {

using word_t = unsigned long long;

template <class R>
struct Kind;
template <>
struct Kind<float> {
    using V3 = float3;
    using V4 = float4;
    using Sym = Sym3;
    static constexpr uint32_t kWords = 3;   // 32-bit pieces of a position
    __device__ static V3 v3(float x, float y, float z) { return make_float3(x, y, z); }
    __device__ static V4 v4(float x, float y, float z, float w) { return make_float4(x, y, z, w); }
    __device__ static uint32_t word(V4 p, uint32_t j) {
        return __float_as_uint(j == 0 ? p.x : (j == 1 ? p.y : p.z));
    }
};
template <>
struct Kind<double> {
    using V3 = D3;
    using V4 = double4;
    using Sym = SymD;
    static constexpr uint32_t kWords = 6;
    __device__ static V3 v3(double x, double y, double z) { return D3{x, y, z}; }
    __device__ static V4 v4(double x, double y, double z, double w) { return make_double4(x, y, z, w); }
    __device__ static uint32_t word(V4 p, uint32_t j) {
        const word_t b = (word_t)__double_as_longlong(j < 2 ? p.x : (j < 4 ? p.y : p.z));
        return j & 1u ? (uint32_t)(b >> 32) : (uint32_t)b;
    }
};

template <bool DAMP>
__device__ __forceinline__ void shape_incidence(float3 p0, float3 p1, float3 p2, float3 p3, float4 r1, float4 r2,
                                                float4 r3, uint32_t local, const TetDamp* damp, uint32_t t,
                                                float inv_dt, float3& g, Sym3& h) {
    nh_incidence_pos<DAMP>(p0, p1, p2, p3, r1, r2, r3, local, damp, t, inv_dt, g, h);
}
template <bool DAMP>
__device__ __forceinline__ void shape_incidence(D3 p0, D3 p1, D3 p2, D3 p3, float4 r1, float4 r2, float4 r3,
                                                uint32_t local, const TetDamp* damp, uint32_t t, double inv_dt, D3& g,
                                                SymD& h) {
    nh_incidence<DAMP>(p0, p1, p2, p3, r1, r2, r3, local, damp, t, inv_dt, g, h);
}
// Place of a lane's terms in its group's sum (FP64 adds them in lane order).
template <class R, int L>
__device__ __forceinline__ uint32_t first_incidence(uint32_t lane) {
    if constexpr (sizeof(R) == 4) return sum_place<L>(lane);
    else return lane;
}
__device__ __forceinline__ void dual(GroundRec& c, float3 p) { ground_dual_update(c, make_float4(p.x, p.y, p.z, 0.f)); }
__device__ __forceinline__ void dual(GroundRec& c, D3 p) { ground_dual_update(c, p); }

template <class R>
struct Args {
    ResidentDev r;
    typename Kind<R>::V4 *x, *y, *last, *lastlast;
    GroundRec* ground;
    const int32_t* ground_of;
    const TetRec* tets;
    const TetDamp* damp;
    const TetEdges* edges;
    const ResCtl* rc;
    const float* omega_tab;
    const uint32_t* frozen;
    ResidentCheck chk;   // every: iterations of the launch when it has no checks
    R inv_dt, inv_dt2;
};

template <int L, bool HESS, class V, class S>
__device__ __forceinline__ void sum_group(V& g, S& h) {
    g.x = group_sum<L>(g.x);
    g.y = group_sum<L>(g.y);
    g.z = group_sum<L>(g.z);
    if constexpr (HESS) {
        h.a00 = group_sum<L>(h.a00);
        h.a11 = group_sum<L>(h.a11);
        h.a22 = group_sum<L>(h.a22);
        h.a01 = group_sum<L>(h.a01);
        h.a02 = group_sum<L>(h.a02);
        h.a12 = group_sum<L>(h.a12);
    }
}

__device__ __forceinline__ float residual2(float4 xv, float4 yv, float3 g, float inv_dt2) {
    const float md = xv.w * inv_dt2;
    const float rx = md * (xv.x - yv.x) + g.x, ry = md * (xv.y - yv.y) + g.y, rz = md * (xv.z - yv.z) + g.z;
    return rx * rx + ry * ry + rz * rz;
}
__device__ __forceinline__ double residual2(double4 xv, double4 yv, D3 g, double inv_dt2) {
    const double md = xv.w * inv_dt2;
    const double rx = md * (xv.x - yv.x) + g.x, ry = md * (xv.y - yv.y) + g.y, rz = md * (xv.z - yv.z) + g.z;
    return rx * rx + ry * ry + rz * rz;
}

template <class R>
__device__ __forceinline__ R chebyshev(R w, R x, R xll) {
    return w * (x - xll) + xll;
}

// The converged test of a scene with residual sum r2 (that of the launch which
// records the checks: residual_collect_kernel).
__device__ __forceinline__ bool converged(const ResidentCheck& k, uint32_t scene, double r2) {
    const double m = k.mg2[scene];
    return k.per_scene ? r2 <= k.tol2 * m : !(m > 0) || r2 / m <= k.tol2;
}

// Sum over the workgroup in a fixed order, the same value in every thread.
template <int B>
__device__ __forceinline__ double block_sum(double v, double* red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    __syncthreads();   // red is free
    if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0;
#pragma unroll
    for (int w = 0; w < B / 64; w++) t += red[w];
    return t;
}

// Edge constants of a tet as corner a sees them.
__device__ __forceinline__ uint32_t weight_index(uint32_t a, uint32_t j) {
    // kEdgeWeight[a][j] in nibble a
    constexpr uint32_t kTable[3] = {0x2100u, 0x5341u, 0x4532u};
    return (kTable[j] >> (4u * a)) & 7u;
}

__device__ __forceinline__ ResidentGround to_lds(const GroundRec& r) {
    return ResidentGround{r.k_n,      r.k_t,  r.k_b,  r.lambda_n, r.lambda_t, r.lambda_b,
                          r.C_n_prev, r.mu_s, r.mu_k, r.cp_x,     r.cp_z,     r.flags};
}
__device__ __forceinline__ GroundRec to_rec(const ResidentGround& l) {
    GroundRec r{};
    r.k_n = l.k_n;
    r.k_t = l.k_t;
    r.k_b = l.k_b;
    r.lambda_n = l.lambda_n;
    r.lambda_t = l.lambda_t;
    r.lambda_b = l.lambda_b;
    r.C_n_prev = l.C_n_prev;
    r.mu_s = l.mu_s;
    r.mu_k = l.mu_k;
    r.cp_x = l.cp_x;
    r.cp_z = l.cp_z;
    r.flags = l.flags;
    return r;
}

// A scene whose patches could not all run at once: its first patch runs the
// stretch alone on the state in device memory, patch by patch (a workgroup's
// own global writes are visible to it after a barrier).
template <class R, int L, bool DAMP, int B>
__device__ __forceinline__ void run_alone(const Args<R>& a, uint32_t first, uint32_t count, uint32_t scene,
                                          uint32_t checks, double* red) {
    using K = Kind<R>;
    using V3 = typename K::V3;
    using V4 = typename K::V4;
    const uint32_t lane = threadIdx.x % L, group = threadIdx.x / L, groups = B / L;
    const uint32_t nc = a.r.n_colors;
    const float* omega = a.omega_tab + (a.rc ? a.rc->iter : 0u);
    auto pos = [&](uint32_t v) {
        const V4 p = a.x[v];
        return K::v3(p.x, p.y, p.z);
    };
    constexpr bool EDGES = resident_edges(sizeof(R), DAMP);
    auto item = [&](const ResidentPatch& p, uint32_t k, V3 xa, V3& g, typename K::Sym& h) {
        const uint32_t it = a.r.item[p.item_off + k].x, begin = it & 0xffffu, cnt = it >> 16;
        g = K::v3(0, 0, 0);
        h = {0, 0, 0, 0, 0, 0};
        for (uint32_t j = first_incidence<R, L>(lane); j < cnt; j += L) {
            const uint32_t code = a.r.inc[p.inc_off + begin + j].y >> 16, c = code & 3u;
            const uint32_t t = a.r.tet[p.tet_off + (code >> 2)];
            uint4 idx;
            float4 r1, r2, r3;
            load_tet(a.tets, t, idx, r1, r2, r3);
            if constexpr (!EDGES) {
                shape_incidence<DAMP>(pos(idx.x), pos(idx.y), pos(idx.z), pos(idx.w), r1, r2, r3, c, a.damp, t,
                                      a.inv_dt, g, h);
            } else {
                const TetEdges& e = a.edges[t];
                const uint32_t n[4] = {idx.x, idx.y, idx.z, idx.w};
                // the other corners in kEdgeCorner order
                const uint32_t i1 = c == 0 ? n[1] : n[0], i2 = c == 0 || c == 3 ? n[2] : (c == 1 ? n[3] : n[1]),
                               i3 = c == 0 || c == 2 ? n[3] : (c == 1 ? n[2] : n[1]);
                edge_incidence(pos(i1) - xa, pos(i2) - xa, pos(i3) - xa, e.w[weight_index(c, 0)], e.w[weight_index(c, 1)],
                               e.w[weight_index(c, 2)], e.h, e.b, g, h);
            }
        }
    };
    for (uint32_t n = 0; n < checks; n++) {
    for (uint32_t i = 0; i < a.chk.every; i++) {
        for (uint32_t c = 0; c < nc; c++) {
            for (uint32_t q = first; q < first + count; q++) {
                const ResidentPatch p = a.r.patches[q];
                const uint32_t* col = a.r.col + p.col_off;
                for (uint32_t k = col[c] + group; k < col[c + 1]; k += groups) {
                    const uint32_t v = a.r.gid[p.gid_off + k];
                    const V4 xv = a.x[v];
                    V3 g;
                    typename K::Sym h;
                    item(p, k, K::v3(xv.x, xv.y, xv.z), g, h);
                    sum_group<L, true>(g, h);
                    if (lane != 0) continue;
                    const int32_t gi = a.ground_of[v];
                    if (gi >= 0) ground_accumulate(a.ground[gi], K::v3(xv.x, xv.y, xv.z), g, h);
                    a.x[v] = block_step(xv, a.y[v], g, h, a.inv_dt2);
                }
            }
            __syncthreads();
        }
        const R w = *omega++;
        for (uint32_t q = first; q < first + count; q++) {
            const ResidentPatch p = a.r.patches[q];
            for (uint32_t k = threadIdx.x; k < p.own; k += B) {
                const uint32_t v = a.r.gid[p.gid_off + k];
                const V4 xc = a.x[v], xl = a.last[v], xll = a.lastlast[v];
                const V4 xp = K::v4(chebyshev(w, xc.x, xll.x), chebyshev(w, xc.y, xll.y), chebyshev(w, xc.z, xll.z),
                                    xc.w);
                a.x[v] = xp;
                a.lastlast[v] = xl;
                a.last[v] = xp;
                const int32_t gi = a.ground_of[v];
                if (gi >= 0) {
                    GroundRec rec = a.ground[gi];
                    dual(rec, K::v3(xp.x, xp.y, xp.z));
                    a.ground[gi] = rec;
                }
            }
        }
        __syncthreads();
    }
    if (!a.chk.hist) return;
    for (uint32_t q = first; q < first + count; q++) {
        const ResidentPatch p = a.r.patches[q];
        double r2 = 0;
        for (uint32_t k = group; k < p.items; k += groups) {
            const uint32_t v = a.r.gid[p.gid_off + k];
            const V4 xv = a.x[v];
            V3 g;
            typename K::Sym h;
            item(p, k, K::v3(xv.x, xv.y, xv.z), g, h);
            sum_group<L, false>(g, h);
            if (lane != 0) continue;
            const int32_t gi = a.ground_of[v];
            if (gi >= 0) ground_accumulate(a.ground[gi], K::v3(xv.x, xv.y, xv.z), g, h);
            r2 += residual2(xv, a.y[v], g, a.inv_dt2);
        }
        r2 = block_sum<B>(r2, red);
        // under tag 0, which no exchange waits for
        if (threadIdx.x < 2)
            __hip_atomic_store(a.r.sums + 2 * q + threadIdx.x, (word_t)Kind<double>::word(make_double4(r2, 0, 0, 0), threadIdx.x),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    double sum = 0;
    for (uint32_t q = threadIdx.x; q < count; q += B) {
        const word_t* w = a.r.sums + 2 * (first + q);
        const word_t lo = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                     hi = __hip_atomic_load(w + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sum += __longlong_as_double((long long)(hi << 32 | lo));
    }
    sum = block_sum<B>(sum, red);
    if (threadIdx.x == 0) {
        a.chk.hist[scene * a.chk.per_launch + n] = sum;
        a.chk.ran[scene] = n + 1;
    }
    if (converged(a.chk, scene, sum)) return;
    }
}

// A lane's incidence, read from LDS in two steps: what does not change
// (indices, tet constants), and then the positions.
template <class R>
struct LdsView {
    const R *edge, *x;
    const float4* quad;
    const TetDamp* damp;
    const uint2* tix;
    const uint8_t* inc;
    uint32_t tets;
    R inv_dt;
    __device__ typename Kind<R>::V3 pos(uint32_t k) const { return Kind<R>::v3(x[3 * k], x[3 * k + 1], x[3 * k + 2]); }
};
template <class R, bool DAMP, bool EDGES = resident_edges(sizeof(R), DAMP)>
struct Staged {
    uint32_t code;
    uint2 ix;
    float4 r1, r2, r3;
    __device__ void read(const LdsView<R>& v, uint32_t e) {
        code = reinterpret_cast<const uint16_t*>(v.inc)[e];
        const uint32_t t = code >> 2;
        ix = v.tix[t];
        r1 = v.quad[3 * t];
        r2 = v.quad[3 * t + 1];
        r3 = v.quad[3 * t + 2];
    }
    struct Pos {
        typename Kind<R>::V3 p0, p1, p2, p3;
    };
    __device__ Pos gather(const LdsView<R>& v) const {
        return Pos{v.pos(ix.x & 0xffffu), v.pos(ix.x >> 16), v.pos(ix.y & 0xffffu), v.pos(ix.y >> 16)};
    }
    __device__ void add(const LdsView<R>& v, const Pos& p, typename Kind<R>::V3, typename Kind<R>::V3& g,
                        typename Kind<R>::Sym& h) const {
        shape_incidence<DAMP>(p.p0, p.p1, p.p2, p.p3, r1, r2, r3, code & 3u, v.damp, code >> 2, v.inv_dt, g, h);
    }
};
template <class R, bool DAMP>
struct Staged<R, DAMP, true> {
    uint2 e;   // the three other particles, (tet << 2) | corner
    R w1, w2, w3, h, b;
    __device__ void read(const LdsView<R>& v, uint32_t k) {
        e = reinterpret_cast<const uint2*>(v.inc)[k];
        const uint32_t t = e.y >> 18, a = (e.y >> 16) & 3u;
        w1 = v.edge[__umul24(weight_index(a, 0), v.tets) + t];
        w2 = v.edge[__umul24(weight_index(a, 1), v.tets) + t];
        w3 = v.edge[__umul24(weight_index(a, 2), v.tets) + t];
        h = v.edge[6 * v.tets + t];
        b = v.edge[7 * v.tets + t];
    }
    struct Pos {
        typename Kind<R>::V3 p1, p2, p3;
    };
    __device__ Pos gather(const LdsView<R>& v) const {
        return Pos{v.pos(e.x & 0xffffu), v.pos(e.x >> 16), v.pos(e.y & 0xffffu)};
    }
    __device__ void add(const LdsView<R>&, const Pos& p, typename Kind<R>::V3 xa, typename Kind<R>::V3& g,
                        typename Kind<R>::Sym& hh) const {
        edge_incidence(p.p1 - xa, p.p2 - xa, p.p3 - xa, w1, w2, w3, h, b, g, hh);
    }
};

// Workgroup barrier over LDS only: __syncthreads also waits for the position
// words on their way to memory, which no thread of this workgroup reads.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

constexpr uint32_t kWaitPolls = 1u << 24;   // about 2 s: the bound of an exchange wait

template <class R, int L, bool DAMP, int B>
__global__ __launch_bounds__(B) void resident_kernel(Args<R> a) {
    using K = Kind<R>;
    using V3 = typename K::V3;
    using V4 = typename K::V4;
    constexpr uint32_t W = K::kWords;
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ uint32_t decision, dead;
    __shared__ double red[B / 64];
    if (a.rc && a.rc->done) return;
    const ResidentPatch p = a.r.patches[blockIdx.x];
    if (a.frozen && a.frozen[p.scene]) return;
    const uint32_t tid = threadIdx.x, nc = a.r.n_colors;
    // check intervals of this launch (the step's budget is chk.total of them)
    const uint32_t checks = a.chk.hist ? min(a.chk.per_launch, a.chk.total - min(a.chk.total, a.rc->checks)) : 1u;
    const bool has_ground = a.r.has_ground;
    const ResidentLds o =
        resident_lds(p.own, p.items, p.local, p.tets, p.inc, p.targets, nc, sizeof(R), DAMP, has_ground);
    R* edge = reinterpret_cast<R*>(lds + o.edge);
    float4* quad = reinterpret_cast<float4*>(lds + o.quad);
    TetDamp* damp = reinterpret_cast<TetDamp*>(lds + o.damp);
    uint2* tix = reinterpret_cast<uint2*>(lds + o.tix);
    R* x = reinterpret_cast<R*>(lds + o.x);
    R* last = reinterpret_cast<R*>(lds + o.last);
    R* lastlast = reinterpret_cast<R*>(lds + o.lastlast);
    R* ym = reinterpret_cast<R*>(lds + o.ym);
    ResidentGround* ground = reinterpret_cast<ResidentGround*>(lds + o.ground);
    R* force = reinterpret_cast<R*>(lds + o.force);
    int32_t* gof = reinterpret_cast<int32_t*>(lds + o.gof);
    uint2* item = reinterpret_cast<uint2*>(lds + o.item);
    uint32_t* target = reinterpret_cast<uint32_t*>(lds + o.target);
    uint32_t* col = reinterpret_cast<uint32_t*>(lds + o.col);
    const LdsView<R> view{edge, x, quad, damp, tix, lds + o.inc, p.tets, a.inv_dt};

    // The ground force on an own particle at its current position.  It changes
    // only with the Chebyshev / dual step (the particle itself moves in its own
    // phase alone), so it is formed there and not in the colour phases.
    auto ground_terms = [&](uint32_t k, const GroundRec& rec, V3 q) {
        const V3 f = ground_force(rec, q);
        force[3 * k] = f.x;
        force[3 * k + 1] = f.y;
        force[3 * k + 2] = f.z;
    };

    // ---- load the patch
    for (uint32_t t = tid; t < p.tets; t += B) {
        const uint32_t g = a.r.tet[p.tet_off + t];
        if constexpr (!resident_edges(sizeof(R), DAMP)) {
            uint4 idx;
            float4 r1, r2, r3;
            load_tet(a.tets, g, idx, r1, r2, r3);
            quad[3 * t] = r1;
            quad[3 * t + 1] = r2;
            quad[3 * t + 2] = r3;
            tix[t] = a.r.tix[p.tet_off + t];
            if constexpr (DAMP) damp[t] = a.damp[g];
        } else {
            const TetEdges e = a.edges[g];
#pragma unroll
            for (int j = 0; j < 6; j++) edge[j * p.tets + t] = e.w[j];
            edge[6 * p.tets + t] = e.h;
            edge[7 * p.tets + t] = e.b;
        }
    }
    for (uint32_t k = tid; k < p.local; k += B) {
        const uint32_t v = a.r.gid[p.gid_off + k];
        const V4 xv = a.x[v], xl = a.last[v], xll = a.lastlast[v];
        x[3 * k] = xv.x;
        x[3 * k + 1] = xv.y;
        x[3 * k + 2] = xv.z;
        last[3 * k] = xl.x;
        last[3 * k + 1] = xl.y;
        last[3 * k + 2] = xl.z;
        lastlast[3 * k] = xll.x;
        lastlast[3 * k + 1] = xll.y;
        lastlast[3 * k + 2] = xll.z;
        if (k < p.own) {
            const V4 yv = a.y[v];
            ym[4 * k] = yv.x;
            ym[4 * k + 1] = yv.y;
            ym[4 * k + 2] = yv.z;
            ym[4 * k + 3] = xv.w;
            if (has_ground) {
                const int32_t gi = a.ground_of[v];
                gof[k] = gi;
                if (gi >= 0) {
                    const GroundRec rec = a.ground[gi];
                    ground[k] = to_lds(rec);
                    ground_terms(k, rec, K::v3(xv.x, xv.y, xv.z));
                }
            }
        }
    }
    for (uint32_t k = tid; k < p.items; k += B) item[k] = a.r.item[p.item_off + k];
    for (uint32_t k = tid; k < p.targets; k += B) target[k] = a.r.target[p.target_off + k];
    for (uint32_t k = tid; k < 2u * (nc + 1u); k += B) col[k] = a.r.col[p.col_off + k];
    for (uint32_t k = tid; k < p.inc; k += B) {
        const uint2 e = a.r.inc[p.inc_off + k];
        if constexpr (!resident_edges(sizeof(R), DAMP))
            reinterpret_cast<uint16_t*>(lds + o.inc)[k] = (uint16_t)(e.y >> 16);
        else reinterpret_cast<uint2*>(lds + o.inc)[k] = e;
    }
    const uint32_t base = p.count > 1 ? a.r.epoch[blockIdx.x] : 0u;
    if (tid == 0) dead = 0;
    __syncthreads();

    // ---- is the whole cluster running?
    if (p.count > 1) {
        if (tid == 0) {
            uint32_t* arrived = a.r.sync + 2 * p.first;
            uint32_t* word = arrived + 1;   // 2 * launch: go, 2 * launch + 1: give up
            const uint32_t launch = a.r.launches[blockIdx.x] + 1u;   // the same for every patch of the cluster
            a.r.launches[blockIdx.x] = launch;
            const uint32_t want = 2u * launch;
            const bool full =
                __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.count - 1u;
            if (full)   // everyone has arrived: ready for the next launch
                __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint32_t patience = a.r.alternate && (launch & 1u) ? 0u : a.r.gather_polls;
            uint32_t polls = 0;
            uint32_t now = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            while ((int32_t)(now - want) < 0) {
                if (full || polls++ >= patience) {
                    uint32_t seen = now;
                    const uint32_t next = full ? want : want + 1u;
                    now = __hip_atomic_compare_exchange_strong(word, &seen, next, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT)
                              ? next
                              : seen;
                } else {
                    __builtin_amdgcn_s_sleep(1);
                    now = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            decision = now & 1u;
        }
        __syncthreads();
        if (decision) {
            if (blockIdx.x == p.first) run_alone<R, L, DAMP, B>(a, p.first, p.count, p.scene, checks, red);
            return;   // the exchange did not run: the epochs stay
        }
    }

    const uint32_t lane = tid % L, group = tid / L, place = first_incidence<R, L>(lane);
    constexpr uint32_t groups = B / L;
    // the payload of an exchange word, once it carries `tag`
    auto wait_word = [&](const word_t* src, uint32_t tag) {
        for (uint32_t polls = 0;; polls++) {
            const word_t u = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((uint32_t)(u >> 32) == tag) return (uint32_t)u;
            if (*(volatile uint32_t*)&dead || polls > kWaitPolls) {
                *(volatile uint32_t*)&dead = 1;
                atomicOr(a.r.status, 2u);
                return 0u;
            }
        }
    };
    // takes the halo of colour c at exchange `tag`: the slots of a colour are
    // contiguous, and so are their places in x, so a thread moves one 32-bit piece
    // (threads from the top: the low ones have the items)
    auto refresh = [&](uint32_t c, uint32_t tag) {
        const uint32_t h0 = col[nc + 1 + c], h1 = col[nc + 2 + c];
        const word_t* src = a.r.xch + (size_t)(p.slot + (h0 - p.own)) * W;
        uint32_t* dst = reinterpret_cast<uint32_t*>(x) + h0 * W;
        for (uint32_t k = B - 1 - tid; k < (h1 - h0) * W; k += B) dst[k] = wait_word(src + k, tag);
    };
    // the scene's sum of the patches' v after exchange `tag`
    auto scene_sum = [&](double v, uint32_t tag, uint32_t turn) {
        v = block_sum<B>(v, red);
        if (p.count == 1) return v;
        word_t* set = a.r.sums + 2 * (size_t)(turn * a.r.n_patches + p.first);
        if (tid < 2)
            __hip_atomic_store(set + 2 * (blockIdx.x - p.first) + tid,
                               (word_t)tag << 32 | Kind<double>::word(make_double4(v, 0, 0, 0), tid), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        double sum = 0;
        for (uint32_t q = tid; q < p.count; q += B) {
            const word_t lo = wait_word(set + 2 * q, tag), hi = wait_word(set + 2 * q + 1, tag);
            sum += __longlong_as_double((long long)(hi << 32 | lo));
        }
        return block_sum<B>(sum, red);
    };

    // A lane's first incidence of a colour phase is read ahead: indices and
    // constants do not change, so the chain item -> incidence -> tet runs while the
    // phase before ends.  (Two or three at once took 80 more registers and gave
    // nothing: 117 instead of 114 ms for 6350 FP64 iterations at 32^3.)
    uint2 it = make_uint2(0, 0);
    Staged<R, DAMP> st;
    auto read_item = [&](uint32_t k) {
        it = item[k];
        if (place < it.x >> 16) st.read(view, (it.x & 0xffffu) + place);
    };
    // The item's own state, which its phases before do not change either (only
    // the Chebyshev / dual step does).
    V4 xv = K::v4(0, 0, 0, 0), yv = xv;
    V3 gf = K::v3(0, 0, 0);
    struct {
        float k_n, k_t, k_b;
    } gk{};
    bool touches = false;
    auto read_own = [&](uint32_t k) {
        xv = K::v4(x[3 * k], x[3 * k + 1], x[3 * k + 2], ym[4 * k + 3]);
        yv = K::v4(ym[4 * k], ym[4 * k + 1], ym[4 * k + 2], 0);
        touches = has_ground && gof[k] >= 0;
        if (has_ground) {
            const ResidentGround& gr = ground[k];   // (unset without a contact, and not used then)
            gk = {gr.k_n, gr.k_t, gr.k_b};
            gf = K::v3(force[3 * k], force[3 * k + 1], force[3 * k + 2]);
        }
    };
    auto read_ahead_own = [&](uint32_t c) {
        const uint32_t k = col[c] + group;
        if (k < col[c + 1]) read_own(k);
    };
    auto read_ahead = [&](uint32_t c, bool own) {
        const uint32_t k = col[c] + group;
        if (k >= col[c + 1]) return;
        read_item(k);
        if (own) read_own(k);
    };
    auto gather = [&](V3 xa, V3& g, typename K::Sym& h) {
        const uint32_t begin = it.x & 0xffffu, cnt = it.x >> 16;
        g = K::v3(0, 0, 0);
        h = {0, 0, 0, 0, 0, 0};
        for (uint32_t j = place; j < cnt;) {
            st.add(view, st.gather(view), xa, g, h);
            j += L;
            if (j < cnt) st.read(view, begin + j);
        }
    };

    // sends the new position of the current item to its readers: lane j the piece
    // j % W to reader j / W, j / W + per, ... (target holds their word offsets)
    constexpr uint32_t per = L >= W ? L / W : 1u;
    const uint32_t reader = L >= W ? lane / W : 0u, piece = L >= W ? lane % W : lane;
    auto send = [&](V4 nx, uint32_t tag) {
        const uint32_t n0 = it.y & 0xffffu, n1 = n0 + (it.y >> 16);
        if (reader >= per) return;
#pragma unroll
        for (uint32_t j = 0; j < W; j += L) {   // more than one piece per lane only when L < W
            if (piece + j >= W) break;
            const word_t u = (word_t)tag << 32 | K::word(nx, piece + j);
            for (uint32_t n = n0 + reader; n < n1; n += per)
                __hip_atomic_store(a.r.xch + (target[n] + piece + j), u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };

    // ---- the iterations
    const float* omega = a.omega_tab + (a.rc ? a.rc->iter : 0u);
    uint32_t tag = base;
    for (uint32_t n = 0; n < checks; n++) {
        read_ahead(0, true);
        for (uint32_t i = 0; i < a.chk.every; i++) {
            tag++;
            const R w = *omega++;
            for (uint32_t c = 0; c < nc; c++) {
                const uint32_t end = col[c + 1], begin = col[c] + group;
                for (uint32_t k = begin; k < end; k += groups) {
                    if (k != begin) {
                        read_item(k);
                        read_own(k);
                    }
                    V3 g;
                    typename K::Sym h;
                    gather(K::v3(xv.x, xv.y, xv.z), g, h);
                    sum_group<L, true>(g, h);
                    // every lane of the group solves the block: the same instructions
                    // as one lane would issue, and each can then send a piece of the result
                    if (touches) ground_add(gk, gf, g, h);
                    const V4 nx = block_step(xv, yv, g, h, a.inv_dt2);
                    send(nx, tag);
                    if (lane == 0) {
                        x[3 * k] = nx.x;
                        x[3 * k + 1] = nx.y;
                        x[3 * k + 2] = nx.z;
                    }
                }
                read_ahead(c + 1 < nc ? c + 1 : 0u, c + 1 < nc);
                // a vertex of colour c has no neighbour of colour c, so the halo of
                // this colour can change while other wavefronts still solve it
                refresh(c, tag);
                lds_barrier();
            }
            for (uint32_t k = tid; k < p.local; k += B) {
                R q[3];
    #pragma unroll
                for (int j = 0; j < 3; j++) {
                    const R xll = lastlast[3 * k + j];
                    q[j] = chebyshev(w, x[3 * k + j], xll);
                    lastlast[3 * k + j] = last[3 * k + j];
                    last[3 * k + j] = q[j];
                    x[3 * k + j] = q[j];
                }
                if (has_ground && k < p.own && gof[k] >= 0) {
                    GroundRec rec = to_rec(ground[k]);
                    dual(rec, K::v3(q[0], q[1], q[2]));
                    ground[k] = to_lds(rec);
                    ground_terms(k, rec, K::v3(q[0], q[1], q[2]));
                }
            }
            lds_barrier();
            read_ahead_own(0);
        }
        if (!a.chk.hist) break;
        double r2 = 0;
        for (uint32_t k = group; k < p.items; k += groups) {
            read_item(k);
            read_own(k);
            V3 g;
            typename K::Sym h;
            gather(K::v3(xv.x, xv.y, xv.z), g, h);
            sum_group<L, false>(g, h);
            if (lane == 0) {
                if (touches) ground_add(gk, gf, g, h);
                r2 += residual2(xv, yv, g, a.inv_dt2);
            }
        }
        r2 = scene_sum(r2, tag, n & 1u);
        if (tid == 0 && blockIdx.x == p.first) {
            a.chk.hist[p.scene * a.chk.per_launch + n] = r2;
            a.chk.ran[p.scene] = n + 1;
        }
        if (converged(a.chk, p.scene, r2)) break;   // the same in every patch of the scene
    }

    // ---- the state back
    for (uint32_t k = tid; k < p.own; k += B) {
        const uint32_t v = a.r.gid[p.gid_off + k];
        const R m = ym[4 * k + 3];
        a.x[v] = K::v4(x[3 * k], x[3 * k + 1], x[3 * k + 2], m);
        a.last[v] = K::v4(last[3 * k], last[3 * k + 1], last[3 * k + 2], m);
        a.lastlast[v] = K::v4(lastlast[3 * k], lastlast[3 * k + 1], lastlast[3 * k + 2], m);
        if (has_ground && gof[k] >= 0) {
            GroundRec& rec = a.ground[gof[k]];
            const ResidentGround l = ground[k];
            rec.k_n = l.k_n;
            rec.k_t = l.k_t;
            rec.k_b = l.k_b;
            rec.lambda_n = l.lambda_n;
            rec.lambda_t = l.lambda_t;
            rec.lambda_b = l.lambda_b;
            rec.flags = l.flags;
        }
    }
    if (tid == 0 && p.count > 1) a.r.epoch[blockIdx.x] = tag;
}

// Launches, or with per_cu set asks how many workgroups fit on a CU.
template <class R, int L, bool DAMP, int B>
void dispatch_block(hipStream_t s, const Args<R>& a, uint32_t* per_cu) {
    // more than 64 KB of LDS has to be asked for
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&resident_kernel<R, L, DAMP, B>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)a.r.lds_bytes);
    if (per_cu) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &n, reinterpret_cast<const void*>(&resident_kernel<R, L, DAMP, B>), B, a.r.lds_bytes) != hipSuccess)
            (void)hipGetLastError();
        *per_cu = (uint32_t)(n > 1 ? n : 1);
        return;
    }
    hipLaunchKernelGGL((resident_kernel<R, L, DAMP, B>), dim3(a.r.n_patches), dim3(B), a.r.lds_bytes, s, a);
}

template <class R, int L, bool DAMP>
void dispatch(hipStream_t s, const Args<R>& a, uint32_t* per_cu) {
    if constexpr (sizeof(R) == 4)
        if (a.r.block == 1024) return dispatch_block<R, L, DAMP, 1024>(s, a, per_cu);
    dispatch_block<R, L, DAMP, 512>(s, a, per_cu);
}

template <class R>
void launch(hipStream_t s, const Args<R>& a, bool damping, uint32_t* per_cu = nullptr) {
#define AVBD_RES_CASE(LL)                                     \
    case LL:                                                   \
        if (damping) dispatch<R, LL, true>(s, a, per_cu);      \
        else dispatch<R, LL, false>(s, a, per_cu);             \
        break;
    switch (a.r.lanes) {
        AVBD_RES_CASE(4)
        AVBD_RES_CASE(8)
        AVBD_RES_CASE(16)
        AVBD_RES_CASE(32)
        default: break;
    }
#undef AVBD_RES_CASE
}

}  // namespace

uint32_t resident_per_cu(const ResidentDev& r, bool fp64, bool damping) {
    uint32_t n = 1;
    if (fp64) {
        Args<double> a{};
        a.r = r;
        launch<double>(nullptr, a, damping, &n);
    } else {
        Args<float> a{};
        a.r = r;
        launch<float>(nullptr, a, damping, &n);
    }
    return n;
}

void launch_resident(hipStream_t s, const ResidentDev& r, const DevState& d, bool damping, float dt, const ResCtl* rc,
                     const float* omega_tab, const ResidentCheck& chk) {
    if (chk.every == 0) return;
    Args<float> a{r,      d.x,       d.y,      d.x_last, d.x_lastlast, d.ground,
                  d.ground_of, d.tets, d.damp, r.edges, rc, omega_tab,
                  d.frozen, chk, 1.0f / dt, 1.0f / (dt * dt)};
    launch<float>(s, a, damping);
}

void launch_resident_f64(hipStream_t s, const ResidentDev& r, const F64State& f, bool damping, double dt,
                         const ResCtl* rc, const float* omega_tab, const ResidentCheck& chk) {
    if (chk.every == 0) return;
    const double inv_dt = 1.0 / dt;
    Args<double> a{r,      f.x,       f.y,      f.x_last, f.x_lastlast, f.ground,
                   f.ground_of, f.tets, f.damp, r.edges, rc, omega_tab,
                   f.frozen, chk, inv_dt, inv_dt * inv_dt};
    launch<double>(s, a, damping);
}

// Records the checks of a resident launch.  Per check: the sums over all
// scenes (a scene that had stopped counts with the residual it stopped at), in
// the order of residual_decide_kernel, one wavefront per check; then the step's
// counters, and the scenes that stopped are frozen.  One workgroup; it runs once
// per launch of about a hundred iterations.
__global__ __launch_bounds__(1024) void residual_collect_kernel(ResCtl* rc, ResidentCheck k, double* acc_scene,
                                                                uint32_t n_scenes, SceneFreeze fz) {
    __shared__ uint32_t most, reached;
    if (rc->done) return;
    if (threadIdx.x == 0) {
        most = 0;
        reached = 0xFFFFFFFFu;
    }
    __syncthreads();
    const uint32_t iter = rc->iter, checks = rc->checks;
    for (uint32_t s = threadIdx.x; s < n_scenes; s += 1024) {
        uint32_t ran = k.ran[s];
        const bool stopped = fz.frozen && fz.frozen[s];
        if (stopped) ran = k.ran[s] = 0;
        if (ran) acc_scene[s] = k.hist[s * k.per_launch + ran - 1];
        atomicMax(&most, ran);
        if (!fz.frozen || stopped) continue;
        const uint32_t n = ran ? ran : 1u;   // a scene without particles has no patch
        if (converged(k, s, ran ? acc_scene[s] : 0.0)) {
            fz.frozen[s] = 1;
            fz.iters[s] = iter + n * k.every;
        }
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t n = threadIdx.x >> 6; n < most; n += 16) {
        double r[4] = {0, 0, 0, 0}, m[4] = {0, 0, 0, 0}, w = 0;
        for (uint32_t s0 = 0; s0 < n_scenes; s0 += 256)
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                const uint32_t s = s0 + 64 * j + lane;
                if (s >= n_scenes) break;
                const double v = n < k.ran[s] ? k.hist[s * k.per_launch + n] : acc_scene[s], mg = k.mg2[s];
                r[j] += v;
                m[j] += mg;
                if (mg > 0) w = fmax(w, v / mg);
            }
        double rs = (r[0] + r[2]) + (r[1] + r[3]), ms = (m[0] + m[2]) + (m[1] + m[3]);
        for (int off = 32; off > 0; off >>= 1) {
            rs += __shfl_down(rs, off);
            ms += __shfl_down(ms, off);
            w = fmax(w, __shfl_xor(w, off));
        }
        if (lane == 0) {
            if (checks + n < kMaxResidualChecks) {
                rc->rel[checks + n] = ms > 0 ? sqrt(rs / ms) : 0.0;
                rc->worst[checks + n] = sqrt(w);
            }
            if (w <= k.tol2) atomicMin(&reached, n);
        }
    }
    __syncthreads();
    for (uint32_t s = threadIdx.x; s < n_scenes; s += 1024) k.ran[s] = 0;
    if (threadIdx.x == 0) {
        rc->checks = checks + most;
        rc->iter = iter + most * k.every;
        if (reached < most || (most == 0 && checks < k.total)) {   // (no check run: every scene is frozen)
            rc->done = 1;
            rc->last_iters = rc->iter;
        }
    }
}

void launch_residual_collect(hipStream_t s, ResCtl* rc, const ResidentCheck& chk, double* acc_scene, uint32_t n_scenes,
                             const SceneFreeze& fz) {
    hipLaunchKernelGGL(residual_collect_kernel, dim3(1), dim3(1024), 0, s, rc, chk, acc_scene, n_scenes, fz);
}

}  // namespace avbd
