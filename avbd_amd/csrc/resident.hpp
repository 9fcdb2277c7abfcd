// resident.hpp -- the resident solve: data shared by the host partitioner
// (resident_host.cpp) and the kernel (resident_kernels.hip).
//
// Every scene is cut into patches of neighbouring particles; one workgroup
// owns a patch, keeps its tets, its particles and a copy of the neighbouring
// particles (the halo) in LDS, and runs a whole stretch of iterations (every
// colour phase, Chebyshev step and dual update) in one launch.  The patches of
// one scene (a cluster) exchange the positions of boundary vertices after
// each colour through tagged words in device memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "internal.hpp"

namespace avbd {

struct alignas(16) ResidentPatch {
    uint32_t own, items, local, tets;   // particles owned (the first `items` are work items), own + halo, tets
    uint32_t inc, targets;              // tet incidences of the items; halo slots they are sent to
    uint32_t gid_off, tet_off, inc_off, item_off, col_off, target_off;   // into the arrays below
    uint32_t slot;                      // exchange slot of the first halo particle
    uint32_t scene;
    uint32_t first, count;              // the cluster's patches [first, first + count)
};

// Contact state of an own particle as the iterations need it (GroundRec
// without k_start, which only the start of a step reads).
struct alignas(16) ResidentGround {
    float k_n, k_t, k_b, lambda_n, lambda_t, lambda_b, C_n_prev, mu_s, mu_k, cp_x, cp_z;
    uint32_t flags;
};

// An undamped FP64 state works on the tets' edge constants (TetEdges); FP32 and
// damped scenes on the rest shape.
__host__ __device__ constexpr bool resident_edges(uint32_t real, bool damp) { return real == 8 && !damp; }

// LDS layout of a patch, in bytes (the same function sizes the launch and
// carves the array in the kernel).  Edge constants: eight arrays (arrays and not
// records, whose 32-word stride would put every lane on the same few banks) and
// 8 bytes per incidence; else rest shape, corners, with damping E_prev, and
// 2 bytes per incidence.
struct ResidentLds {
    uint32_t edge, quad, damp, tix, x, last, lastlast, ym, ground, force, gof, item, target, col, inc, total;
};
__host__ __device__ inline ResidentLds resident_lds(uint32_t own, uint32_t items, uint32_t local, uint32_t tets,
                                                    uint32_t inc, uint32_t targets, uint32_t colors, uint32_t real,
                                                    bool damp, bool ground) {
    ResidentLds l;
    const bool edges = resident_edges(real, damp);
    uint32_t at = 0;
    auto take = [&](uint32_t bytes) {
        const uint32_t o = at;
        at += (bytes + 15u) & ~15u;
        return o;
    };
    l.edge = take(edges ? 8u * real * tets : 0u);
    l.quad = take(edges ? 0u : 48u * tets);
    l.damp = take(damp ? 32u * tets : 0u);
    l.tix = take(edges ? 0u : 8u * tets);
    l.inc = take((edges ? 8u : 2u) * inc);
    l.x = take(3u * real * local);
    l.last = take(3u * real * local);
    l.lastlast = take(3u * real * local);
    l.ym = take(4u * real * own);
    l.ground = take(ground ? (uint32_t)sizeof(ResidentGround) * own : 0u);
    l.force = take(ground ? 3u * real * own : 0u);
    l.gof = take(ground ? 4u * own : 0u);
    l.item = take(8u * items);
    l.target = take(4u * targets);
    l.col = take(8u * (colors + 1u));
    l.total = at;
    return l;
}

struct ResidentPlan {
    std::vector<ResidentPatch> patches;
    std::vector<uint32_t> gid;     // per local particle its global index: own items by colour, other own, then the
                                   // halo by colour (fixed particles last)
    std::vector<uint32_t> tet;     // global tet of every patch tet
    std::vector<uint16_t> tix;     // its four local particles
    std::vector<uint16_t> inc;     // per incidence, by item in pool order: the three other local particles
                                   // (kEdgeCorner order) and (patch tet << 2) | corner
    std::vector<uint32_t> item;    // per item: first incidence | count << 16, first target | count << 16
    std::vector<uint32_t> target;  // first exchange word of each halo slot that an item's position is sent to
    std::vector<uint32_t> col;     // per patch: colours + 1 item offsets, colours + 1 halo offsets (local indices)
    uint32_t slots = 0, lds_bytes = 0, max_cluster = 0;
};

struct ResidentLimits {
    uint32_t real_bytes;      // 4 or 8
    bool damp, ground;
    uint32_t lds_bytes;       // LDS a workgroup may use
    uint32_t max_cluster;     // patches of one scene (all must be resident at once)
    uint32_t target;          // tet incidences per patch aimed at
};

// Partition every scene (recursive coordinate bisection of `pos`, 3 doubles
// per particle); false when some scene does not fit the limits.
bool build_resident(const HostModel& m, const ColorPlan& plan, const double* pos, const ResidentLimits& lim,
                    ResidentPlan& out);

// Threads of a patch's workgroup: 1024 where one phase has more items than 512
// threads hold groups of `lanes` (512 scenes: 45.2 -> 40.8 ms; where all fit, idle
// wavefronts cost 2.45 -> 2.71 ms at 32^3); FP64 stays at 512, where its registers fit.
uint32_t resident_block(const ResidentPlan& plan, uint32_t colors, const ResidentLimits& lim, uint32_t lanes);

// What a launch runs: check intervals of `every` iterations until the scene has
// converged, per_launch of them at most and `total` in a step (hist set), or
// just `every` iterations (hist null).
struct ResidentCheck {
    uint32_t every = 0, per_launch = 0, total = 0;
    uint32_t per_scene = 0;       // the scenes of a batch stop on their own
    double tol2 = 0;
    const double* mg2 = nullptr;  // per scene: ||M g||^2 over its free particles
    double* hist = nullptr;       // per scene per_launch residual sums
    uint32_t* ran = nullptr;      // per scene: checks of this launch (0 again once recorded)
};

// Device side of the plan plus the state the kernel works on.
struct ResidentDev {
    const ResidentPatch* patches = nullptr;
    const uint32_t* gid = nullptr;
    const uint32_t* tet = nullptr;
    const uint2* tix = nullptr;
    const uint2* inc = nullptr;
    const uint2* item = nullptr;
    const uint32_t* target = nullptr;
    const uint32_t* col = nullptr;
    const TetEdges* edges = nullptr;     // per tet (undamped FP64 state)
    unsigned long long* xch = nullptr;   // per halo slot 3 (FP32) or 6 (FP64) tagged words
    unsigned long long* sums = nullptr;  // two sets of two tagged words per patch: its residual sum
    uint32_t* epoch = nullptr;           // per patch: exchanges per colour so far (the tag base)
    uint32_t* launches = nullptr;        // per patch: launches so far
    uint32_t* sync = nullptr;            // per patch (the cluster's first one): arrivals, decision word
    uint32_t* status = nullptr;          // = DevState::status
    uint32_t n_patches = 0, n_colors = 0, lds_bytes = 0, max_cluster = 0, lanes = 8, block = 512;
    uint32_t cus = 0, per_cu = 0;        // of the device; workgroups of this launch that fit on one of them
    uint32_t gather_polls = 0;           // polls after which a patch no longer waits for its cluster to be resident
    bool alternate = false;              // for tests: odd launches do not wait for it
    bool has_ground = false;
};

// The iterations of `chk` from omega_tab[0] (in residual mode omega_tab[rc->iter]).
void launch_resident(hipStream_t s, const ResidentDev& r, const DevState& d, bool damping, float dt, const ResCtl* rc,
                     const float* omega_tab, const ResidentCheck& chk);
void launch_resident_f64(hipStream_t s, const ResidentDev& r, const F64State& f, bool damping, double dt,
                         const ResCtl* rc, const float* omega_tab, const ResidentCheck& chk);
// Workgroups of the context's launch that fit on one CU at once.
uint32_t resident_per_cu(const ResidentDev& r, bool fp64, bool damping);
// After a launch with checks: the step's residual record, counters and frozen scenes.
void launch_residual_collect(hipStream_t s, ResCtl* rc, const ResidentCheck& chk, double* acc_scene, uint32_t n_scenes,
                             const SceneFreeze& fz);

}  // namespace avbd
