// tet_device.hpp -- FP32 device functions of one positional vertex-block
// solve (Neo-Hookean incidence, ground AL terms, 3x3 LDL^T, Chebyshev step,
// dual update), shared by the per-phase kernels (vbd_kernels.hip) and the
// resident solve (resident_kernels.hip).  Both files are compiled with
// -ffp-contract=on, so a function rounds the same way in either.
//
// The order of every sum and each rounding here is part of the framework's
// results: friction branches on the last bit (ground_dual_update), and over a
// batch of 942,000 vertices a form that differs by one rounding moves single
// vertices by up to a third of the velocities' rms (an energy from edge vectors and
// a solve by reciprocals took 32 instead of 40 ms there per 10 steps, and were taken
// back for that).
#pragma once

#include "internal.hpp"

namespace avbd {
namespace {

struct Sym3 {
    float a00, a11, a22, a01, a02, a12;
};

__device__ __forceinline__ float3 f3(float4 v) { return make_float3(v.x, v.y, v.z); }
__device__ __forceinline__ float3 operator-(float3 a, float3 b) { return make_float3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ float3 operator+(float3 a, float3 b) { return make_float3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ float3 operator*(float s, float3 a) { return make_float3(s * a.x, s * a.y, s * a.z); }
__device__ __forceinline__ float dot3(float3 a, float3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ float3 cross3(float3 a, float3 b) {
    return make_float3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}

// Load a 64-byte tet record with four 16-byte loads.
__device__ __forceinline__ void load_tet(const TetRec* __restrict__ tets, uint32_t t, uint4& idx, float4& r1,
                                         float4& r2, float4& r3) {
    const uint4* p = reinterpret_cast<const uint4*>(tets + t);
    idx = p[0];
    const float4* f = reinterpret_cast<const float4*>(p);
    r1 = f[1];
    r2 = f[2];
    r3 = f[3];
}

// One tet incidence of the stable Neo-Hookean energy
// (NeoHookeanEnergySolver::accumulate, energy/elastic/NeoHookeanEnergySolver.hpp:121-227).
// q = Q.row(local) for local < 3, -(Q.row0 + Q.row1 + Q.row2) for local 3 (the
// reference's sign = -1 folded into q; every term is linear in q or quadratic).
// The record (idx, r1..r3) is already loaded; t indexes the damping record.
// nh_incidence_pos takes the four vertex positions already gathered.
template <bool DAMP>
__device__ __forceinline__ void nh_incidence_pos(float3 p0, float3 p1, float3 p2, float3 p3, float4 r1, float4 r2,
                                                 float4 r3, uint32_t local, const TetDamp* __restrict__ damp,
                                                 uint32_t t, float inv_dt, float3& g, Sym3& h) {
    // r1 = q00 q01 q02 q10 ; r2 = q11 q12 q20 q21 ; r3 = q22 VL VM alpha
    const float3 d0 = p0 - p3, d1 = p1 - p3, d2 = p2 - p3;
    const float q00 = r1.x, q01 = r1.y, q02 = r1.z, q10 = r1.w, q11 = r2.x, q12 = r2.y, q20 = r2.z, q21 = r2.w,
                q22 = r3.x;
    const float VL = r3.y, VM = r3.z, alpha = r3.w;
    // F = D Q: column c of F = d0 Q[0][c] + d1 Q[1][c] + d2 Q[2][c]
    const float3 f0 = q00 * d0 + q10 * d1 + q20 * d2;
    const float3 f1 = q01 * d0 + q11 * d1 + q21 * d2;
    const float3 f2 = q02 * d0 + q12 * d1 + q22 * d2;
    const float3 c0 = cross3(f1, f2), c1 = cross3(f2, f0), c2 = cross3(f0, f1);
    const float J = dot3(f0, c0);
    float3 q;
    if (local == 0) q = make_float3(q00, q01, q02);
    else if (local == 1) q = make_float3(q10, q11, q12);
    else if (local == 2) q = make_float3(q20, q21, q22);
    else q = make_float3(-(q00 + q10 + q20), -(q01 + q11 + q21), -(q02 + q12 + q22));
    const float3 Fq = q.x * f0 + q.y * f1 + q.z * f2;
    const float3 Fc = q.x * c0 + q.y * c1 + q.z * c2;
    const float hyd = VL * (J - alpha);
    const float q2 = dot3(q, q);
    g = g + (hyd * Fc + VM * Fq);
    const float dev = VM * q2;
    h.a00 += VL * Fc.x * Fc.x + dev;
    h.a11 += VL * Fc.y * Fc.y + dev;
    h.a22 += VL * Fc.z * Fc.z + dev;
    h.a01 += VL * Fc.x * Fc.y;
    h.a02 += VL * Fc.x * Fc.z;
    h.a12 += VL * Fc.y * Fc.z;
    if constexpr (DAMP) {
        const TetDamp dr = damp[t];
        const float dm = dr.damp;
        // Edot = (0.5 F^T F - 0.5 I - E_prev) / dt, symmetric
        const float e00 = (0.5f * dot3(f0, f0) - 0.5f - dr.e00) * inv_dt;
        const float e11 = (0.5f * dot3(f1, f1) - 0.5f - dr.e11) * inv_dt;
        const float e22 = (0.5f * dot3(f2, f2) - 0.5f - dr.e22) * inv_dt;
        const float e01 = (0.5f * dot3(f0, f1) - dr.e01) * inv_dt;
        const float e02 = (0.5f * dot3(f0, f2) - dr.e02) * inv_dt;
        const float e12 = (0.5f * dot3(f1, f2) - dr.e12) * inv_dt;
        const float3 Eq = make_float3(e00 * q.x + e01 * q.y + e02 * q.z, e01 * q.x + e11 * q.y + e12 * q.z,
                                      e02 * q.x + e12 * q.y + e22 * q.z);
        const float3 FEq = Eq.x * f0 + Eq.y * f1 + Eq.z * f2;
        g = g + dm * FEq;
        const float diag = dm * dot3(q, Eq);
        const float a = 0.5f * dm * inv_dt;
        // F F^T rows: (F F^T)_ij = sum_c F_ic F_jc
        const float ff00 = f0.x * f0.x + f1.x * f1.x + f2.x * f2.x;
        const float ff11 = f0.y * f0.y + f1.y * f1.y + f2.y * f2.y;
        const float ff22 = f0.z * f0.z + f1.z * f1.z + f2.z * f2.z;
        const float ff01 = f0.x * f0.y + f1.x * f1.y + f2.x * f2.y;
        const float ff02 = f0.x * f0.z + f1.x * f1.z + f2.x * f2.z;
        const float ff12 = f0.y * f0.z + f1.y * f1.z + f2.y * f2.z;
        h.a00 += diag + a * (q2 * ff00 + Fq.x * Fq.x);
        h.a11 += diag + a * (q2 * ff11 + Fq.y * Fq.y);
        h.a22 += diag + a * (q2 * ff22 + Fq.z * Fq.z);
        h.a01 += a * (q2 * ff01 + Fq.x * Fq.y);
        h.a02 += a * (q2 * ff02 + Fq.x * Fq.z);
        h.a12 += a * (q2 * ff12 + Fq.y * Fq.z);
    }
}

// A lane's incidence of the work-item order: the record, then the gathered
// positions, then the terms (three steps, so that several can be in flight).
template <bool DAMP>
struct TetInc {
    uint4 idx;
    float4 r1, r2, r3;
    struct Pos {
        float3 p0, p1, p2, p3;
    };
    __device__ void load(const TetRec* __restrict__ irec, uint32_t k) { load_tet(irec, k, idx, r1, r2, r3); }
    __device__ Pos gather(const float4* x) const {
        return Pos{f3(x[idx.x]), f3(x[idx.y]), f3(x[idx.z]), f3(x[idx.w & 0x3fffffffu])};
    }
    __device__ void add(const Pos& p, const TetDamp* __restrict__ damp, uint32_t t, float inv_dt, float3& g,
                        Sym3& h) const {
        nh_incidence_pos<DAMP>(p.p0, p.p1, p.p2, p.p3, r1, r2, r3, idx.w >> 30, damp, t, inv_dt, g, h);
    }
};

// Ground AL contact contribution (CollisionConstraintEnergySolver::accumulate<3>,
// energy/collision/CollisionConstraintEnergySolver.hpp:180-285 with the ground
// constraint of energy/collision/GroundCollisionEnergySolver.hpp:27-60).
__device__ __forceinline__ float3 ground_force(const GroundRec& c, float3 p) {
    const float Cn = -p.y, Ct = p.x - c.cp_x, Cb = p.z - c.cp_z;
    const float Ccorr = Cn - kAlpha * c.C_n_prev;
    const float lnp = fmaxf(0.0f, c.k_n * Ccorr + c.lambda_n);
    float lt = c.k_t * Ct + c.lambda_t;
    float lb = c.k_b * Cb + c.lambda_b;
    const float mag = sqrtf(lt * lt + lb * lb);
    const float mu = (c.flags & GF_USE_STATIC) ? c.mu_s : c.mu_k;
    const float lmax = mu * lnp;
    if (mag > lmax) {
        const float nrm = mag + 1e-8f;
        lt = lt / nrm * lmax;
        lb = lb / nrm * lmax;
    }
    return make_float3(lt, -lnp, lb);
}
template <class Rec>
__device__ __forceinline__ void ground_add(const Rec& c, float3 f, float3& g, Sym3& h) {
    g.x += f.x;
    g.y += f.y;
    g.z += f.z;
    h.a00 += c.k_t;
    h.a11 += c.k_n;
    h.a22 += c.k_b;
}
__device__ __forceinline__ void ground_accumulate(const GroundRec& c, float3 p, float3& g, Sym3& h) {
    ground_add(c, ground_force(c, p), g, h);
}

// Solve (m/dt^2 I + H) dx = b for symmetric positive definite H by LDL^T.
__device__ __forceinline__ float3 ldlt3(const Sym3& A, float3 b) {
    const float d0 = A.a00;
    const float l10 = A.a01 / d0, l20 = A.a02 / d0;
    const float d1 = A.a11 - l10 * A.a01;
    const float l21 = (A.a12 - l20 * A.a01) / d1;
    const float d2 = A.a22 - l20 * A.a02 - l21 * l21 * d1;
    const float z0 = b.x;
    const float z1 = b.y - l10 * z0;
    const float z2 = b.z - l20 * z0 - l21 * z1;
    const float x2 = z2 / d2;
    const float x1 = z1 / d1 - l21 * x2;
    const float x0 = z0 / d0 - l10 * x1 - l20 * x2;
    return make_float3(x0, x1, x2);
}

// Sum over the L lanes of a group; every lane gets it.  Ascending butterfly in
// DPP moves (quad permutes, then mirrors of 8 and 16 lanes, which meet a lane
// of the other half since each half is already uniform): a register operand
// modifier instead of an LDS-pipe permute of about 130 cycles per step.
// Lane l holds the terms of place sum_place<L>(l), l with its bits reversed, so
// that the places are added as a butterfly from L / 2 down to 1 does: that order is
// part of an FP32 step's result (a contact that leaves static friction by one last
// bit moves a vertex by millimetres).
template <int L>
__device__ __forceinline__ uint32_t sum_place(uint32_t lane) {
    return __brev(lane) >> (32 - __builtin_ctz(L));
}
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_move(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __uint_as_float(dpp_move<CTRL>(__float_as_uint(v)));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140;
template <int L>
__device__ __forceinline__ float group_sum(float v) {
    static_assert(L == 4 || L == 8 || L == 16 || L == 32, "lanes per vertex");
    v = dpp_add<kDppXor1>(v);
    v = dpp_add<kDppXor2>(v);
    if constexpr (L >= 8) v = dpp_add<kDppHalfMirror>(v);
    if constexpr (L >= 16) v = dpp_add<kDppMirror>(v);
    if constexpr (L >= 32) v += __shfl_xor(v, 16);
    return v;
}

// Inertia term and 3x3 solve of a vertex block with energy gradient g and
// Hessian h; returns the new position (mass kept in w).
__device__ __forceinline__ float4 block_step(float4 xv, float4 yv, float3 g, Sym3 h, float inv_dt2) {
    const float3 p = f3(xv);
    const float md = xv.w * inv_dt2;   // m / dt^2
    h.a00 += md;
    h.a11 += md;
    h.a22 += md;
    const float3 b = make_float3(-md * (p.x - yv.x) - g.x, -md * (p.y - yv.y) - g.y, -md * (p.z - yv.z) - g.z);
    const float3 dx = ldlt3(h, b);
    return make_float4(p.x + dx.x, p.y + dx.y, p.z + dx.z, xv.w);
}

// _particleChebyshevAcceleration (VBDSolver.hpp:513-536) of one position.
__device__ __forceinline__ float4 cheb_apply(float4 xp, float4 xll, float omega) {
    xp.x = omega * (xp.x - xll.x) + xll.x;
    xp.y = omega * (xp.y - xll.y) + xll.y;
    xp.z = omega * (xp.z - xll.z) + xll.z;
    return xp;
}

// CollisionConstraintEnergySolver::updateAfterIteration (CollisionConstraintEnergySolver.hpp:60-134)
// of one ground record at the extrapolated position xp.
__device__ __forceinline__ void ground_dual_update(GroundRec& c, float4 xp) {
    const float Cn = -xp.y, Ct = xp.x - c.cp_x, Cb = xp.z - c.cp_z;
    const float Ccorr = Cn - kAlpha * c.C_n_prev;
    const float lnp = c.k_n * Ccorr + c.lambda_n;
    const float ltp = c.k_t * Ct + c.lambda_t;
    const float lbp = c.k_b * Cb + c.lambda_b;
    if (lnp > 0.f) c.k_n += kBeta * fabsf(Ccorr);
    c.lambda_n = fmaxf(0.f, lnp);
    const float mag = sqrtf(ltp * ltp + lbp * lbp);
    float lmax = ((c.flags & GF_USE_STATIC) ? c.mu_s : c.mu_k) * c.lambda_n;
    if (mag < lmax) {
        c.k_t += kBeta * fabsf(Ct);
        c.k_b += kBeta * fabsf(Cb);
        c.lambda_t = ltp;
        c.lambda_b = lbp;
        c.flags |= GF_UNCLAMPED;
    } else {
        if (c.flags & GF_USE_STATIC) {
            c.flags &= ~GF_USE_STATIC;
            lmax = c.mu_k * lnp;
        }
        c.lambda_t = ltp / (mag + 1e-8f) * lmax;
        c.lambda_b = lbp / (mag + 1e-8f) * lmax;
        c.flags &= ~GF_UNCLAMPED;
    }
}

}  // namespace
}  // namespace avbd
