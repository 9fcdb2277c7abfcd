// lbvh_kernels.hip -- device LBVH broad phase over triangle primitives.
//
// Bit-exact with the reference's CPU builder on identical inputs:
//   * bounds, centroids and Morton codes are computed in FP64 from the FP32
//     state, without contraction (this file is compiled with -ffp-contract=off):
//     CollisionPrimitivePool::speculativeGlobalBounds (collision/CollisionPrimitivePool.hpp:160-174),
//     LBVHBuilder::computeAABB_MortonCode (collision/LBVHBuilder.cpp:98-127),
//     morton3D_64 / expandBits21 (collision/LBVHBuilder.hpp:65-86);
//   * the sort orders by (code, original index) -- what a stable LSD radix sort
//     of the codes produces (common/Algorithm.hpp:22-56);
//   * the hierarchy is Karras (2012) with the reference's delta, including the
//     index tie-break of commonPrefixLen (collision/LBVHBuilder.hpp:33-41,
//     collision/LBVHBuilder.cpp:181-286);
//   * node boxes are the min/max over the leaves a node covers -- what the
//     reference's bottom-up refit computes (collision/LBVHBuilder.cpp:410-453);
//     min/max are exact, so any evaluation order gives the same bits;
//   * traversal reports every leaf pair (a < b) whose closed boxes overlap,
//     the set produced by LBVHTraversal::traverseSelfIterative
//     (collision/LBVHTraversal.hpp:30-88); eight lanes walk the tree per leaf,
//     reading a packed record of both children per visit.
//
// With a few thousand to a few ten thousand primitives every kernel here is a
// chain of dependent loads on a nearly empty device, so each is arranged to
// shorten that chain.  12,288 triangles of a cube, beside the solve, before -> now:
// scan 8.8 -> 6.1, rank 10.7 -> 5.6, hierarchy 29 -> 12.5, traversal 104 -> 24.5 us;
// the whole build, which the step waits for, 205 -> 93 us.
#include "lbvh.hpp"

#include <type_traits>

namespace avbd {

namespace {

constexpr uint32_t INV = 0xFFFFFFFFu;

__device__ __forceinline__ uint64_t expand_bits21(uint64_t v) {
    v &= 0x1FFFFFull;
    v = (v | (v << 32)) & 0x1F00000000FFFFull;
    v = (v | (v << 16)) & 0x1F0000FF0000FFull;
    v = (v | (v << 8)) & 0x100F00F00F00F00Full;
    v = (v | (v << 4)) & 0x10C30C30C30C30C3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}

__device__ __forceinline__ uint64_t morton_axis(double p) {
    double s = p * 2097152.0;
    s = s < 0.0 ? 0.0 : (s > 2097151.0 ? 2097151.0 : s);   // std::clamp(s, 0, 2097151)
    return expand_bits21(static_cast<uint64_t>(s));
}

__device__ __forceinline__ int clz64(uint64_t x) { return x == 0 ? 64 : __builtin_clzll(x); }

__device__ __forceinline__ int common_prefix_len(uint64_t ci, uint32_t i, uint64_t cj, uint32_t j) {
    if (ci == cj) return 64 + clz64(static_cast<uint64_t>(i) ^ static_cast<uint64_t>(j));
    return clz64(ci ^ cj);
}

__global__ void tri_aabb_kernel(const uint32_t* __restrict__ tris, uint32_t n, const float4* __restrict__ x,
                                const float4* __restrict__ v, double dt, double* __restrict__ aabb) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    double b[6] = {__DBL_MAX__, __DBL_MAX__, __DBL_MAX__, -__DBL_MAX__, -__DBL_MAX__, -__DBL_MAX__};
    for (int c = 0; c < 3; c++) {
        const uint32_t p = tris[3 * t + c];
        const float4 xp = x[p], vp = v[p];
        const double a[3] = {xp.x, xp.y, xp.z};
        const double w[3] = {vp.x, vp.y, vp.z};
        for (int k = 0; k < 3; k++) {
            const double e = a[k] + dt * w[k];
            b[k] = fmin(b[k], a[k]);
            b[3 + k] = fmax(b[3 + k], a[k]);
            b[k] = fmin(b[k], e);
            b[3 + k] = fmax(b[3 + k], e);
        }
    }
    for (int k = 0; k < 6; k++) aabb[6 * t + k] = b[k];
}

constexpr uint32_t BUCKET_SHIFT = 50;   // codes have 63 bits: the top 13 pick the bucket
constexpr uint32_t N_BUCKETS = 1u << 13;
constexpr uint32_t BUCKETS_PER_THREAD = N_BUCKETS / 1024;

// Box of all lanes' boxes in lane 0 of the wavefront.
__device__ __forceinline__ void wave_union(double b[6]) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < 3; k++) {
            b[k] = fmin(b[k], __shfl_xor(b[k], off));
            b[3 + k] = fmax(b[3 + k], __shfl_xor(b[3 + k], off));
        }
}

// One block: scene box = union of the primitive boxes (in registers, then one
// exchange between the wavefronts); also resets the pair counter
// and the bucket counts of this build.
__global__ __launch_bounds__(1024) void scene_box_kernel(const double* __restrict__ aabb, uint32_t n,
                                                         double* __restrict__ sbox, uint32_t* __restrict__ counters,
                                                         uint32_t* __restrict__ bucket_count) {
    __shared__ double red[6][16];
    for (uint32_t k = threadIdx.x; k < N_BUCKETS; k += blockDim.x) bucket_count[k] = 0;
    double b[6] = {__DBL_MAX__, __DBL_MAX__, __DBL_MAX__, -__DBL_MAX__, -__DBL_MAX__, -__DBL_MAX__};
#pragma unroll 4
    for (uint32_t t = threadIdx.x; t < n; t += 1024)
#pragma unroll
        for (int k = 0; k < 3; k++) {
            b[k] = fmin(b[k], aabb[6 * (size_t)t + k]);
            b[3 + k] = fmax(b[3 + k], aabb[6 * (size_t)t + 3 + k]);
        }
    wave_union(b);
    if ((threadIdx.x & 63u) == 0)
#pragma unroll
        for (int k = 0; k < 6; k++) red[k][threadIdx.x >> 6] = b[k];
    __syncthreads();
    if (threadIdx.x < 6) {
        const uint32_t k = threadIdx.x;
        double v = red[k][0];
        for (int w = 1; w < 16; w++) v = k < 3 ? fmin(v, red[k][w]) : fmax(v, red[k][w]);
        sbox[k] = v;
    }
    if (threadIdx.x == 0) {
        counters[0] = 0;   // pair count
        counters[1] = 0;
    }
}

__global__ void morton_kernel(const double* __restrict__ aabb, uint32_t n, const double* __restrict__ sbox,
                              uint64_t* __restrict__ keys, uint32_t* __restrict__ bucket_count) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    uint64_t code = 0;
    for (int k = 0; k < 3; k++) {
        const double ext = fmax(sbox[3 + k] - sbox[k], 1e-6);
        const double c = (aabb[6 * t + k] + aabb[6 * t + 3 + k]) * 0.5;
        code |= morton_axis((c - sbox[k]) / ext) << k;
    }
    keys[t] = code;
    atomicAdd(&bucket_count[code >> BUCKET_SHIFT], 1u);
}

// Sort by (code, original index) -- the order a stable LSD radix sort of the
// codes produces -- in short fully parallel passes: morton_kernel counts codes
// per bucket of their top 13 bits; one block scans the 8,192 counts; every
// primitive takes a slot in its bucket; every primitive counts the keys of
// its bucket that precede it and lands at bucket offset + count.
__global__ __launch_bounds__(1024) void bucket_scan_kernel(uint32_t* __restrict__ count, uint32_t* __restrict__ offset,
                                                           uint32_t n) {
    static_assert(BUCKETS_PER_THREAD == 8, "two uint4 per thread");
    __shared__ uint32_t part[16];
    const uint32_t t = threadIdx.x;   // eight consecutive buckets per thread
    const uint4 a = reinterpret_cast<const uint4*>(count)[2 * t], b = reinterpret_cast<const uint4*>(count)[2 * t + 1];
    const uint32_t local = a.x + a.y + a.z + a.w + b.x + b.y + b.z + b.w;
    uint32_t incl = local;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(incl, off);
        if ((int)(t & 63u) >= off) incl += v;
    }
    if ((t & 63u) == 63u) part[t >> 6] = incl;
    __syncthreads();
    uint32_t run = incl - local;
    for (uint32_t w = 0; w < (t >> 6); w++) run += part[w];
    uint4 o, q;
    o.x = run;
    o.y = o.x + a.x;
    o.z = o.y + a.y;
    o.w = o.z + a.z;
    q.x = o.w + a.w;
    q.y = q.x + b.x;
    q.z = q.y + b.y;
    q.w = q.z + b.z;
    reinterpret_cast<uint4*>(offset)[2 * t] = o;
    reinterpret_cast<uint4*>(offset)[2 * t + 1] = q;
    // reused as the fill cursor by bucket_place_kernel
    reinterpret_cast<uint4*>(count)[2 * t] = reinterpret_cast<uint4*>(count)[2 * t + 1] = make_uint4(0, 0, 0, 0);
    if (t == 0) offset[N_BUCKETS] = n;
}

__global__ void bucket_place_kernel(const uint64_t* __restrict__ keys, uint32_t n, const uint32_t* __restrict__ offset,
                                    uint32_t* __restrict__ cursor, uint32_t* __restrict__ slots,
                                    uint64_t* __restrict__ slot_keys) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t key = keys[i];
    const uint32_t b = (uint32_t)(key >> BUCKET_SHIFT);
    const uint32_t s = offset[b] + atomicAdd(&cursor[b], 1u);
    slots[s] = i;
    slot_keys[s] = key;   // beside the index, so that ranking does not chase it
}

__global__ void bucket_rank_kernel(const uint64_t* __restrict__ keys, uint32_t n, const uint32_t* __restrict__ offset,
                                   const uint32_t* __restrict__ slots, const uint64_t* __restrict__ slot_keys,
                                   uint64_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t ki = keys[i];
    const uint32_t b = (uint32_t)(ki >> BUCKET_SHIFT);
    const uint32_t lo = offset[b], hi = offset[b + 1];
    uint32_t rank = lo;
#pragma unroll 4
    for (uint32_t s = lo; s < hi; s++) {
        const uint64_t kj = slot_keys[s];
        const uint32_t j = slots[s];
        rank += ((kj < ki) | ((kj == ki) & (j < i))) ? 1u : 0u;
    }
    keys_out[rank] = ki;
    vals_out[rank] = i;
}

// Aligned range-union table over the sorted leaves: entry (k, j) of level k is
// the union of leaves [j 2^k, (j+1) 2^k).  An internal node covers a
// contiguous leaf range, so its box is the union of O(2 log n) entries.
__device__ __forceinline__ uint32_t level_offset(uint32_t n, uint32_t k) {
    uint32_t off = 0;
    for (uint32_t q = 0; q < k; q++) off += (n + (1u << q) - 1) >> q;
    return off;
}

__global__ __launch_bounds__(256) void leaf_table_kernel(const double* __restrict__ aabb,
                                                         const uint32_t* __restrict__ sorted, uint32_t n,
                                                         double* __restrict__ node_box, double* __restrict__ table,
                                                         uint32_t levels_local) {
    __shared__ double sb[6][256];
    const uint32_t l = blockIdx.x * 256 + threadIdx.x;
    double b[6];
    if (l < n) {
        const uint32_t prim = sorted[l];
        for (int k = 0; k < 6; k++) b[k] = aabb[6 * prim + k];
        for (int k = 0; k < 6; k++) {
            node_box[6 * l + k] = b[k];
            table[6 * l + k] = b[k];
        }
    } else {
        for (int k = 0; k < 3; k++) {
            b[k] = __DBL_MAX__;
            b[3 + k] = -__DBL_MAX__;
        }
    }
    for (int k = 0; k < 6; k++) sb[k][threadIdx.x] = b[k];
    __syncthreads();
    for (uint32_t lev = 1; lev <= levels_local; lev++) {
        const uint32_t w = 1u << lev;
        if ((threadIdx.x & (w - 1)) == 0) {
            const uint32_t o = threadIdx.x + (w >> 1);
            for (int k = 0; k < 3; k++) {
                sb[k][threadIdx.x] = fmin(sb[k][threadIdx.x], sb[k][o]);
                sb[3 + k][threadIdx.x] = fmax(sb[3 + k][threadIdx.x], sb[3 + k][o]);
            }
            const uint32_t j = l >> lev;
            if (j < ((n + w - 1) >> lev)) {
                const uint32_t base = level_offset(n, lev) + j;
                for (int k = 0; k < 6; k++) table[6 * base + k] = sb[k][threadIdx.x];
            }
        }
        __syncthreads();
    }
}

// Levels above one block: a single block folds pairs level by level.
__global__ __launch_bounds__(1024) void upper_table_kernel(uint32_t n, double* table, uint32_t first_level,
                                                           uint32_t last_level) {
    for (uint32_t lev = first_level; lev <= last_level; lev++) {
        const uint32_t cnt = (n + (1u << lev) - 1) >> lev;
        const uint32_t prev_cnt = (n + (1u << (lev - 1)) - 1) >> (lev - 1);
        const uint32_t po = level_offset(n, lev - 1), o = level_offset(n, lev);
        for (uint32_t j = threadIdx.x; j < cnt; j += blockDim.x) {
            const double* a = table + 6 * (po + 2 * j);
            double b[6];
            for (int k = 0; k < 6; k++) b[k] = a[k];
            if (2 * j + 1 < prev_cnt) {
                const double* c = a + 6;
                for (int k = 0; k < 3; k++) {
                    b[k] = fmin(b[k], c[k]);
                    b[3 + k] = fmax(b[3 + k], c[3 + k]);
                }
            }
            for (int k = 0; k < 6; k++) table[6 * (o + j) + k] = b[k];
        }
        __syncthreads();
    }
}

// Union of the leaves [lo, hi] by 16 lanes.  The range is at most one left and
// one right table entry per level (left where ceil(lo / 2^k) is odd, right where
// floor((hi + 1) / 2^k) is odd, while the first is below the second), and a
// lane takes one level: `off`: the offset of level `lane`.
__device__ __forceinline__ void range_union16(const double* __restrict__ table, uint32_t n, uint32_t lo, uint32_t hi,
                                              uint32_t lane, uint32_t off, double* box) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
        box[k] = __DBL_MAX__;
        box[3 + k] = -__DBL_MAX__;
    }
    auto add = [&](uint32_t entry) {
        const double* e = table + 6 * (size_t)entry;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            box[c] = fmin(box[c], e[c]);
            box[3 + c] = fmax(box[3 + c], e[3 + c]);
        }
    };
    for (uint32_t k = lane; k < 32 && ((hi + 1 - lo) >> k) != 0; k += 16) {
        const uint32_t l = (uint32_t)(((uint64_t)lo + (1ull << k) - 1) >> k), r = (hi + 1) >> k;
        if (l >= r) break;   // also on every level above
        const uint32_t base = k < 16 ? off : level_offset(n, k);
        if (l & 1u) add(base + l);
        if (r & 1u) add(base + r - 1);
    }
    // butterfly over the 16 lanes of a DPP row
    auto other = [](double v, auto ctrl) {
        const uint64_t u = (uint64_t)__double_as_longlong(v);
        constexpr int C = decltype(ctrl)::value;
        const int a = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, C, 0xf, 0xf, true);
        const int b = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), C, 0xf, 0xf, true);
        return __longlong_as_double((long long)((uint64_t)(uint32_t)b << 32 | (uint32_t)a));
    };
    auto fold = [&](auto ctrl) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            box[c] = fmin(box[c], other(box[c], ctrl));
            box[3 + c] = fmax(box[3 + c], other(box[3 + c], ctrl));
        }
    };
    fold(std::integral_constant<int, 0xB1>{});    // quad_perm [1, 0, 3, 2]
    fold(std::integral_constant<int, 0x4E>{});    // quad_perm [2, 3, 0, 1]
    fold(std::integral_constant<int, 0x141>{});   // row_half_mirror
    fold(std::integral_constant<int, 0x140>{});   // row_mirror
}

// 16 lanes per internal node.  The two searches along the sorted codes test 16
// positions at a time (four rounds of loads for 65,536 primitives instead of
// one per halving) and the boxes' table entries are read side by side.
constexpr uint32_t KARRAS_LANES = 16;
__global__ __launch_bounds__(256) void karras_kernel(const uint64_t* __restrict__ code,
                                                     const uint32_t* __restrict__ sorted, uint32_t n,
                                                     uint32_t* __restrict__ left, uint32_t* __restrict__ right,
                                                     uint32_t* __restrict__ parent, uint32_t* __restrict__ range_hi,
                                                     const double* __restrict__ table, double* __restrict__ node_box,
                                                     TravNode* __restrict__ trav) {
    const int N = (int)n;
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) / KARRAS_LANES);
    const uint32_t lane = threadIdx.x % KARRAS_LANES, row = (threadIdx.x & 63u) / KARRAS_LANES * KARRAS_LANES;
    if (lane == 0) {
        if (i == 0) parent[N > 1 ? N : 0] = INV;   // the root has no parent
        if (i < N) range_hi[i] = (uint32_t)i;      // a leaf covers itself
    }
    if (i >= N - 1) return;   // a node's lanes leave together
    const uint64_t ci = code[i];
    const uint32_t si = sorted[i];
    auto delta = [&](int b) -> int {   // of leaf i and leaf b
        if (b < 0 || b >= N) return -1;
        return common_prefix_len(ci, si, code[b], sorted[b]);
    };
    const int before = delta(i - 1), after = delta(i + 1);
    const int d = after - before >= 0 ? 1 : -1;
    const int dmin = d > 0 ? before : after;
    // the last offset o < limit with delta(i + o d) > bound (true up to it)
    auto last = [&](int limit, int bound) -> int {
        int64_t l = 0, step = 1;
        while (16 * step < limit) step *= 16;
        for (; step >= 1; step /= 16) {
            const int64_t o = l + (int64_t)(lane + 1) * step;
            const bool ok = o < limit && delta(i + (int)o * d) > bound;
            l += step * __popcll((__ballot(ok) >> row) & 0xFFFFull);
        }
        return (int)l;
    };
    const int l = last(N, dmin);
    const int j = i + l * d;
    const int dnode = delta(j);
    const int s = last(l, dnode);
    const int gamma = i + s * d + (d < 0 ? d : 0);
    const uint32_t g = (uint32_t)i + n;
    const uint32_t lc = (min(i, j) == gamma) ? (uint32_t)gamma : n + (uint32_t)gamma;
    const uint32_t rc = (max(i, j) == gamma + 1) ? (uint32_t)gamma + 1 : n + (uint32_t)gamma + 1;
    // children cover [lo, gamma] and [gamma + 1, hi]; the node's box is the
    // union of theirs (min/max are exact: the same bits as one range union)
    TravNode t;
    t.child[0] = lc;
    t.child[1] = rc;
    t.lo[0] = (uint32_t)min(i, j);
    t.hi[0] = (uint32_t)gamma;
    t.lo[1] = (uint32_t)gamma + 1;
    t.hi[1] = (uint32_t)max(i, j);
    t.pad[0] = t.pad[1] = 0;
    const uint32_t off = level_offset(n, lane);
    range_union16(table, n, t.lo[0], t.hi[0], lane, off, t.box[0]);
    range_union16(table, n, t.lo[1], t.hi[1], lane, off, t.box[1]);
    if (lane == 0) {
        left[g] = lc;
        right[g] = rc;
        parent[lc] = g;
        parent[rc] = g;
        range_hi[g] = (uint32_t)max(i, j);
        trav[i] = t;
    }
    if (lane == 1)
        for (int k = 0; k < 3; k++) {
            node_box[6 * (size_t)g + k] = fmin(t.box[0][k], t.box[1][k]);
            node_box[6 * (size_t)g + 3 + k] = fmax(t.box[0][3 + k], t.box[1][3 + k]);
        }
}

// Closed-box overlap; every operand is already in registers, so the six
// tests are evaluated together (no short-circuit chain of dependent reads).
__device__ __forceinline__ bool overlap(const double* a, const double* b) {
    return (a[0] <= b[3]) & (a[3] >= b[0]) & (a[1] <= b[4]) & (a[4] >= b[1]) & (a[2] <= b[5]) & (a[5] >= b[2]);
}

constexpr uint32_t TRAVERSE_LANES = 8;     // per leaf
constexpr uint32_t TRAVERSE_BLOCK = 128;
constexpr uint32_t TRAVERSE_LEAVES = TRAVERSE_BLOCK / TRAVERSE_LANES;
constexpr uint32_t TRAVERSE_WIDE = 64;     // stack height up to which all lanes take a node
constexpr uint32_t TRAVERSE_STACK = TRAVERSE_WIDE + TRAVERSE_LANES + 96;
constexpr uint32_t TRAVERSE_OUT = 1024;    // pairs buffered per block

// Eight lanes per leaf i share a stack in LDS, from the root: in a round each
// takes a node, reads its 128-byte TravNode (both children's boxes and ranges)
// in one go and tests both children; the inner ones that overlap go back to the
// stack, leaves are recorded as pairs (i, j), j > i; children whose last leaf is
// <= i are skipped.  A leaf of a closed surface visits about a hundred nodes,
// which one after the other were a hundred dependent loads (104 us for 12,288
// triangles); in rounds they are about 25.  Above TRAVERSE_WIDE entries only one
// node is taken at a time, so that the stack then grows by at most the depth of
// the tree (63 code bits and 32 of the index: 95).  Pairs are buffered in LDS and
// written with one global atomic reservation per block (a pair counter hit by
// every pair serialises at L2).
__global__ __launch_bounds__(TRAVERSE_BLOCK) void traverse_kernel(uint32_t n, const TravNode* __restrict__ trav,
                                                                  const double* __restrict__ node_box,
                                                                  uint32_t* __restrict__ pairs, uint32_t cap,
                                                                  uint32_t* __restrict__ counters) {
    __shared__ uint32_t stack_mem[TRAVERSE_LEAVES][TRAVERSE_STACK];
    __shared__ uint2 out[TRAVERSE_OUT];
    __shared__ uint32_t out_n, block_base;
    const uint32_t lane = threadIdx.x % TRAVERSE_LANES, leaf = threadIdx.x / TRAVERSE_LANES;
    const uint32_t shift = (threadIdx.x & 63u) / TRAVERSE_LANES * TRAVERSE_LANES;
    const uint32_t i = blockIdx.x * TRAVERSE_LEAVES + leaf;
    uint32_t* stack = stack_mem[leaf];
    if (threadIdx.x == 0) out_n = 0;
    if (lane == 0) stack[0] = n;   // the root (n > 1: internal)
    __syncthreads();
    auto write = [&](uint32_t slot, uint32_t a, uint32_t b) {
        if (slot < cap) {
            pairs[2 * (size_t)slot] = a;
            pairs[2 * (size_t)slot + 1] = b;
        }
    };
    auto emit = [&](uint32_t j) {
        const uint32_t k = atomicAdd(&out_n, 1u);
        if (k < TRAVERSE_OUT) out[k] = make_uint2(i, j);
        else write(atomicAdd(&counters[0], 1u), i, j);   // rare overflow of the buffer: reserve directly
    };
    if (i + 1 < n) {   // the last leaf has no partner j > i
        double bi[6];
#pragma unroll
        for (int k = 0; k < 6; k++) bi[k] = node_box[6 * (size_t)i + k];
        uint32_t sp = 1;   // the same in the leaf's lanes
        while (sp) {
            const uint32_t take = sp > TRAVERSE_WIDE ? 1u : min(sp, TRAVERSE_LANES);
            sp -= take;
            bool h0 = false, h1 = false;
            uint32_t c0 = 0, c1 = 0;
            if (lane < take) {
                const TravNode r = trav[stack[sp + lane] - n];
                c0 = r.child[0];
                c1 = r.child[1];
                h0 = (r.hi[0] > i) & overlap(bi, r.box[0]);
                h1 = (r.hi[1] > i) & overlap(bi, r.box[1]);
                if (h0 && c0 < n) {
                    emit(c0);
                    h0 = false;
                }
                if (h1 && c1 < n) {
                    emit(c1);
                    h1 = false;
                }
            }
            // every lane has read its node before the stack is written (one wavefront)
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const uint32_t m0 = (uint32_t)(__ballot(h0) >> shift) & 0xFFu, m1 = (uint32_t)(__ballot(h1) >> shift) & 0xFFu;
            const uint32_t below = (1u << lane) - 1u, n0 = (uint32_t)__popc(m0);
            if (h0) stack[sp + (uint32_t)__popc(m0 & below)] = c0;
            if (h1) stack[sp + n0 + (uint32_t)__popc(m1 & below)] = c1;
            sp += n0 + (uint32_t)__popc(m1);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
    __syncthreads();
    const uint32_t total = min(out_n, TRAVERSE_OUT);
    if (threadIdx.x == 0) block_base = total ? atomicAdd(&counters[0], total) : 0u;
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < total; k += TRAVERSE_BLOCK) write(block_base + k, out[k].x, out[k].y);
}

inline uint32_t nblk(uint32_t n, uint32_t b) { return (n + b - 1) / b; }

}  // namespace

uint32_t lbvh_table_entries(uint32_t n) {
    uint32_t total = 0;
    for (uint32_t k = 0; (1u << k) < 2 * n; k++) total += (n + (1u << k) - 1) >> k;
    return total;
}

void launch_lbvh_bounds(hipStream_t s, const LbvhDev& b, const float4* x, const float4* v, double dt) {
    if (b.n == 0) return;
    hipLaunchKernelGGL(tri_aabb_kernel, dim3(nblk(b.n, 256)), dim3(256), 0, s, b.tris, b.n, x, v, dt, b.aabb);
}

void launch_lbvh_tree(hipStream_t s, const LbvhDev& b) {
    const uint32_t n = b.n;
    if (n == 0) return;
    uint32_t top = 0;   // highest table level: 2^top >= n
    while ((1u << top) < n) top++;
    hipLaunchKernelGGL(scene_box_kernel, dim3(1), dim3(1024), 0, s, b.aabb, n, b.sbox, b.counters, b.bucket_count);
    hipLaunchKernelGGL(morton_kernel, dim3(nblk(n, 256)), dim3(256), 0, s, b.aabb, n, b.sbox, b.keys,
                       b.bucket_count);
    hipLaunchKernelGGL(bucket_scan_kernel, dim3(1), dim3(1024), 0, s, b.bucket_count, b.bucket_offset, n);
    hipLaunchKernelGGL(bucket_place_kernel, dim3(nblk(n, 256)), dim3(256), 0, s, b.keys, n, b.bucket_offset,
                       b.bucket_count, b.slots, b.slot_keys);
    hipLaunchKernelGGL(bucket_rank_kernel, dim3(nblk(n, 256)), dim3(256), 0, s, b.keys, n, b.bucket_offset, b.slots,
                       b.slot_keys, b.keys_sorted, b.sorted);
    hipLaunchKernelGGL(leaf_table_kernel, dim3(nblk(n, 256)), dim3(256), 0, s, b.aabb, b.sorted, n, b.node_box,
                       b.table, top < 8 ? top : 8u);
    if (top > 8) hipLaunchKernelGGL(upper_table_kernel, dim3(1), dim3(1024), 0, s, n, b.table, 9u, top);
    hipLaunchKernelGGL(karras_kernel, dim3(nblk(n, 256 / KARRAS_LANES)), dim3(256), 0, s, b.keys_sorted, b.sorted, n, b.left,
                       b.right, b.parent, b.range_hi, b.table, b.node_box, b.trav);
    hipLaunchKernelGGL(traverse_kernel, dim3(nblk(n, TRAVERSE_LEAVES)), dim3(TRAVERSE_BLOCK), 0, s, n, b.trav,
                       b.node_box, b.pairs, b.pair_cap, b.counters);
}

void launch_lbvh_build(hipStream_t s, const LbvhDev& b, const float4* x, const float4* v, double dt) {
    launch_lbvh_bounds(s, b, x, v, dt);
    launch_lbvh_tree(s, b);
}

}  // namespace avbd
