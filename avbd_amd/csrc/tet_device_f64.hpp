// tet_device_f64.hpp -- FP64 device functions of one positional vertex-block
// solve, shared by the per-phase kernels (vbd_fp64.hip) and the resident
// solve (resident_kernels.hip); see tet_device.hpp.
#pragma once

#include <type_traits>

#include "internal.hpp"

namespace avbd {
namespace {

struct D3 {
    double x, y, z;
};
__device__ __forceinline__ D3 dd3(double4 v) { return D3{v.x, v.y, v.z}; }
__device__ __forceinline__ D3 operator-(D3 a, D3 b) { return D3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ D3 operator+(D3 a, D3 b) { return D3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ D3 operator*(double s, D3 a) { return D3{s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ double dot3(D3 a, D3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ D3 cross3(D3 a, D3 b) {
    return D3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

struct SymD {
    double a00, a11, a22, a01, a02, a12;
};

// Deformation gradient columns f_c = sum_r d_r Q[r][c] of a record
// (r1 = q00 q01 q02 q10, r2 = q11 q12 q20 q21, r3 = q22 VL VM alpha).
__device__ __forceinline__ void deform(D3 p0, D3 p1, D3 p2, D3 p3, float4 r1, float4 r2, float4 r3, D3& f0, D3& f1,
                                       D3& f2) {
    const D3 d0 = p0 - p3, d1 = p1 - p3, d2 = p2 - p3;
    f0 = (double)r1.x * d0 + (double)r1.w * d1 + (double)r2.z * d2;
    f1 = (double)r1.y * d0 + (double)r2.x * d1 + (double)r2.w * d2;
    f2 = (double)r1.z * d0 + (double)r2.y * d1 + (double)r3.x * d2;
}

// One tet incidence of the stable Neo-Hookean energy in FP64
// (NeoHookeanEnergySolver::accumulate, energy/elastic/NeoHookeanEnergySolver.hpp:121-227):
// Gauss-Newton hydrostatic term, exact deviatoric term, strain-rate damping.
template <bool DAMP>
__device__ __forceinline__ void nh_incidence(D3 p0, D3 p1, D3 p2, D3 p3, float4 r1, float4 r2, float4 r3,
                                             uint32_t local, const TetDamp* __restrict__ damp, uint32_t t,
                                             double inv_dt, D3& g, SymD& h) {
    D3 f0, f1, f2;
    deform(p0, p1, p2, p3, r1, r2, r3, f0, f1, f2);
    const double q00 = r1.x, q01 = r1.y, q02 = r1.z, q10 = r1.w, q11 = r2.x, q12 = r2.y, q20 = r2.z, q21 = r2.w,
                 q22 = r3.x;
    const double VL = r3.y, VM = r3.z, alpha = r3.w;
    const D3 c0 = cross3(f1, f2), c1 = cross3(f2, f0), c2 = cross3(f0, f1);
    const double J = dot3(f0, c0);
    D3 q;
    if (local == 0) q = D3{q00, q01, q02};
    else if (local == 1) q = D3{q10, q11, q12};
    else if (local == 2) q = D3{q20, q21, q22};
    else q = D3{-(q00 + q10 + q20), -(q01 + q11 + q21), -(q02 + q12 + q22)};
    const D3 Fq = q.x * f0 + q.y * f1 + q.z * f2;
    const D3 Fc = q.x * c0 + q.y * c1 + q.z * c2;
    const double hyd = VL * (J - alpha);
    const double q2 = dot3(q, q);
    g = g + (hyd * Fc + VM * Fq);
    const double dev = VM * q2;
    h.a00 += VL * Fc.x * Fc.x + dev;
    h.a11 += VL * Fc.y * Fc.y + dev;
    h.a22 += VL * Fc.z * Fc.z + dev;
    h.a01 += VL * Fc.x * Fc.y;
    h.a02 += VL * Fc.x * Fc.z;
    h.a12 += VL * Fc.y * Fc.z;
    if constexpr (DAMP) {
        const TetDamp dr = damp[t];
        const double dm = dr.damp;
        const double e00 = (0.5 * dot3(f0, f0) - 0.5 - dr.e00) * inv_dt;
        const double e11 = (0.5 * dot3(f1, f1) - 0.5 - dr.e11) * inv_dt;
        const double e22 = (0.5 * dot3(f2, f2) - 0.5 - dr.e22) * inv_dt;
        const double e01 = (0.5 * dot3(f0, f1) - dr.e01) * inv_dt;
        const double e02 = (0.5 * dot3(f0, f2) - dr.e02) * inv_dt;
        const double e12 = (0.5 * dot3(f1, f2) - dr.e12) * inv_dt;
        const D3 Eq = D3{e00 * q.x + e01 * q.y + e02 * q.z, e01 * q.x + e11 * q.y + e12 * q.z,
                         e02 * q.x + e12 * q.y + e22 * q.z};
        const D3 FEq = Eq.x * f0 + Eq.y * f1 + Eq.z * f2;
        g = g + dm * FEq;
        const double diag = dm * dot3(q, Eq);
        const double a = 0.5 * dm * inv_dt;
        const double ff00 = f0.x * f0.x + f1.x * f1.x + f2.x * f2.x;
        const double ff11 = f0.y * f0.y + f1.y * f1.y + f2.y * f2.y;
        const double ff22 = f0.z * f0.z + f1.z * f1.z + f2.z * f2.z;
        const double ff01 = f0.x * f0.y + f1.x * f1.y + f2.x * f2.y;
        const double ff02 = f0.x * f0.z + f1.x * f1.z + f2.x * f2.z;
        const double ff12 = f0.y * f0.z + f1.y * f1.z + f2.y * f2.z;
        h.a00 += diag + a * (q2 * ff00 + Fq.x * Fq.x);
        h.a11 += diag + a * (q2 * ff11 + Fq.y * Fq.y);
        h.a22 += diag + a * (q2 * ff22 + Fq.z * Fq.z);
        h.a01 += a * (q2 * ff01 + Fq.x * Fq.y);
        h.a02 += a * (q2 * ff02 + Fq.x * Fq.z);
        h.a12 += a * (q2 * ff12 + Fq.y * Fq.z);
    }
}

// One incidence of an undamped tet from its edges (EdgeRec64).
__device__ __forceinline__ void edge_incidence(D3 e1, D3 e2, D3 e3, double w1, double w2, double w3, double hn, double b,
                                               D3& g, SymD& h) {
    const D3 u = e2 - e1, v = e3 - e1;
    const D3 n = D3{__builtin_fma(u.y, v.z, -(u.z * v.y)), __builtin_fma(u.z, v.x, -(u.x * v.z)),
                    __builtin_fma(u.x, v.y, -(u.y * v.x))};
    const double k = -__builtin_fma(hn, __builtin_fma(n.x, e1.x, __builtin_fma(n.y, e1.y, n.z * e1.z)), b);
    g.x += __builtin_fma(k, n.x, __builtin_fma(w1, e1.x, __builtin_fma(w2, e2.x, w3 * e3.x)));
    g.y += __builtin_fma(k, n.y, __builtin_fma(w1, e1.y, __builtin_fma(w2, e2.y, w3 * e3.y)));
    g.z += __builtin_fma(k, n.z, __builtin_fma(w1, e1.z, __builtin_fma(w2, e2.z, w3 * e3.z)));
    const double dev = (w1 + w2) + w3;
    const D3 t = hn * n;
    h.a00 += __builtin_fma(t.x, n.x, -dev);
    h.a11 += __builtin_fma(t.y, n.y, -dev);
    h.a22 += __builtin_fma(t.z, n.z, -dev);
    h.a01 = __builtin_fma(t.x, n.y, h.a01);
    h.a02 = __builtin_fma(t.x, n.z, h.a02);
    h.a12 = __builtin_fma(t.y, n.z, h.a12);
}

// A lane's incidence (see TetInc of tet_device.hpp): with damping the rest shape,
// without the edge constants.
struct TetInc64 {
    using Rec = TetRec;
    uint4 idx;
    float4 r1, r2, r3;
    struct Pos {
        D3 p0, p1, p2, p3;
    };
    __device__ void load(const TetRec* __restrict__ irec, uint32_t k) {
        const uint4* p = reinterpret_cast<const uint4*>(irec + k);
        idx = p[0];
        const float4* f = reinterpret_cast<const float4*>(p);
        r1 = f[1];
        r2 = f[2];
        r3 = f[3];
    }
    __device__ Pos gather(const double4* x) const {
        return Pos{dd3(x[idx.x]), dd3(x[idx.y]), dd3(x[idx.z]), dd3(x[idx.w & 0x3fffffffu])};
    }
    __device__ void add(const Pos& p, D3, const TetDamp* __restrict__ damp, uint32_t t, double inv_dt, D3& g,
                        SymD& h) const {
        nh_incidence<true>(p.p0, p.p1, p.p2, p.p3, r1, r2, r3, idx.w >> 30, damp, t, inv_dt, g, h);
    }
};
struct EdgeInc64 {
    using Rec = EdgeRec64;
    double2 c0, c1;   // w1 w2, w3 h
    uint4 d;          // b, the first two of the other vertices
    uint32_t i3;
    struct Pos {
        D3 p1, p2, p3;
    };
    __device__ void load(const EdgeRec64* __restrict__ irec, uint32_t k) {
        const double2* p = reinterpret_cast<const double2*>(irec + k);
        c0 = p[0];
        c1 = p[1];
        d = reinterpret_cast<const uint4*>(p)[2];
        i3 = irec[k].i[2];
    }
    __device__ Pos gather(const double4* x) const { return Pos{dd3(x[d.z]), dd3(x[d.w]), dd3(x[i3])}; }
    __device__ void add(const Pos& p, D3 xa, const TetDamp*, uint32_t, double, D3& g, SymD& h) const {
        const double b = __longlong_as_double((long long)((unsigned long long)d.y << 32 | d.x));
        edge_incidence(p.p1 - xa, p.p2 - xa, p.p3 - xa, c0.x, c0.y, c1.x, c1.y, b, g, h);
    }
};
template <bool DAMP>
using Inc64 = std::conditional_t<DAMP, TetInc64, EdgeInc64>;

// Ground AL contact (CollisionConstraintEnergySolver::accumulate<3> with the
// ground constraint, energy/collision/GroundCollisionEnergySolver.hpp:27-60).
__device__ __forceinline__ D3 ground_force(const GroundRec& c, D3 p) {
    const double Cn = -p.y, Ct = p.x - (double)c.cp_x, Cb = p.z - (double)c.cp_z;
    const double Ccorr = Cn - (double)kAlpha * c.C_n_prev;
    const double lnp = fmax(0.0, (double)c.k_n * Ccorr + c.lambda_n);
    double lt = (double)c.k_t * Ct + c.lambda_t;
    double lb = (double)c.k_b * Cb + c.lambda_b;
    const double mag = sqrt(lt * lt + lb * lb);
    const double mu = (c.flags & GF_USE_STATIC) ? c.mu_s : c.mu_k;
    const double lmax = mu * lnp;
    if (mag > lmax) {
        const double nrm = mag + 1e-8;
        lt = lt / nrm * lmax;
        lb = lb / nrm * lmax;
    }
    return D3{lt, -lnp, lb};
}
template <class Rec>
__device__ __forceinline__ void ground_add(const Rec& c, D3 f, D3& g, SymD& h) {
    g.x += f.x;
    g.y += f.y;
    g.z += f.z;
    h.a00 += c.k_t;
    h.a11 += c.k_n;
    h.a22 += c.k_b;
}
__device__ __forceinline__ void ground_accumulate(const GroundRec& c, D3 p, D3& g, SymD& h) {
    ground_add(c, ground_force(c, p), g, h);
}

// Dual + stiffness-ramp update of one ground record at the extrapolated
// position (CollisionConstraintEnergySolver::updateAfterIteration,
// energy/collision/CollisionConstraintEnergySolver.hpp:60-134).
__device__ __forceinline__ void ground_dual_update(GroundRec& c, D3 xp) {
    const double Cn = -xp.y, Ct = xp.x - (double)c.cp_x, Cb = xp.z - (double)c.cp_z;
    const double Ccorr = Cn - (double)kAlpha * c.C_n_prev;
    const double lnp = (double)c.k_n * Ccorr + c.lambda_n;
    const double ltp = (double)c.k_t * Ct + c.lambda_t;
    const double lbp = (double)c.k_b * Cb + c.lambda_b;
    if (lnp > 0.0) c.k_n = (float)(c.k_n + (double)kBeta * fabs(Ccorr));
    const double ln = fmax(0.0, lnp);
    c.lambda_n = (float)ln;
    const double mag = sqrt(ltp * ltp + lbp * lbp);
    double lmax = ((c.flags & GF_USE_STATIC) ? c.mu_s : c.mu_k) * ln;
    if (mag < lmax) {
        c.k_t = (float)(c.k_t + (double)kBeta * fabs(Ct));
        c.k_b = (float)(c.k_b + (double)kBeta * fabs(Cb));
        c.lambda_t = (float)ltp;
        c.lambda_b = (float)lbp;
        c.flags |= GF_UNCLAMPED;
    } else {
        if (c.flags & GF_USE_STATIC) {
            c.flags &= ~GF_USE_STATIC;
            lmax = c.mu_k * lnp;
        }
        c.lambda_t = (float)(ltp / (mag + 1e-8) * lmax);
        c.lambda_b = (float)(lbp / (mag + 1e-8) * lmax);
        c.flags &= ~GF_UNCLAMPED;
    }
}

__device__ __forceinline__ D3 ldlt3(const SymD& A, D3 b) {
    // one reciprocal per pivot: eight quotients took five more division sequences
    const double d0 = A.a00;
    const double r0 = 1.0 / d0;
    const double l10 = A.a01 * r0, l20 = A.a02 * r0;
    const double d1 = A.a11 - l10 * A.a01;
    const double r1 = 1.0 / d1;
    const double l21 = (A.a12 - l20 * A.a01) * r1;
    const double d2 = A.a22 - l20 * A.a02 - l21 * l21 * d1;
    const double r2 = 1.0 / d2;
    const double z0 = b.x;
    const double z1 = b.y - l10 * z0;
    const double z2 = b.z - l20 * z0 - l21 * z1;
    const double x2 = z2 * r2;
    const double x1 = z1 * r1 - l21 * x2;
    const double x0 = z0 * r0 - l10 * x1 - l20 * x2;
    return D3{x0, x1, x2};
}

// Sum over the L lanes of a group (see group_sum of tet_device.hpp).
template <int CTRL>
__device__ __forceinline__ double dpp_add64(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
    return v + __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
template <int L>
__device__ __forceinline__ double group_sum(double v) {
    static_assert(L == 4 || L == 8 || L == 16 || L == 32, "lanes per vertex");
    v = dpp_add64<0xB1>(v);
    v = dpp_add64<0x4E>(v);
    if constexpr (L >= 8) v = dpp_add64<0x141>(v);
    if constexpr (L >= 16) v = dpp_add64<0x140>(v);
    if constexpr (L >= 32) v += __shfl_xor(v, 16);
    return v;
}

// Inertia term and 3x3 solve of a vertex block; the new position (mass in w).
__device__ __forceinline__ double4 block_step(double4 xv, double4 yv, D3 g, SymD h, double inv_dt2) {
    const D3 p = dd3(xv);
    const double md = xv.w * inv_dt2;
    h.a00 += md;
    h.a11 += md;
    h.a22 += md;
    const D3 b = D3{-md * (p.x - yv.x) - g.x, -md * (p.y - yv.y) - g.y, -md * (p.z - yv.z) - g.z};
    const D3 dx = ldlt3(h, b);
    return make_double4(p.x + dx.x, p.y + dx.y, p.z + dx.z, xv.w);
}

}  // namespace
}  // namespace avbd
