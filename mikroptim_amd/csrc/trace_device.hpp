// Per-ray device math of the trace and of its reverse (adjoint) sweep, templated on the number
// type R (double or df64 for the forward trace; double for the reverse sweep).
//
// Formulas and branch rules follow the reference's shared math core:
//   surface steps        include/mikroptim/trace/surface_ops.hpp:122-203 (FP64: the same
//                        intersection and refraction in optical direction cosines)
//   surface propagation  include/mikroptim/trace/trace.hpp:175-229 (stop/plane/sphere only)
//   reference spheres    include/mikroptim/trace/reference_sphere.hpp:56-143
//   reverse steps        include/mikroptim/trace/adjoint_backward.hpp:115-241, 373-464
// The FP64 surface steps spell their fmas out (no contraction left to the compiler, so every kernel
// that inlines them computes the same bits); the rest is compiled with FMA contraction (hipcc
// default). Results differ from the FP64 CPU oracle by rounding only, which the parity tests
// bound per ray.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "df64.hpp"
#include "mikroptim_types.h"

namespace mkod {

// Number-type helpers of the forward trace: R = double (every mode) or df64 (the RESIDUALS /
// MERIT traces with MKO_PRECISION_DF64). For double they are the identity.
template <class R>
__device__ __forceinline__ R num(double x) {
    return x;
}
template <>
__device__ __forceinline__ df64 num<df64>(double x) {
    return df64_from(x);
}
__device__ __forceinline__ double to_double(double x) { return x; }
__device__ __forceinline__ double to_double(df64 x) { return df64_to(x); }

template <class R>
struct V3 {
    R x, y, z;
};
template <class R>
__device__ __forceinline__ V3<R> operator+(V3<R> a, V3<R> b) {
    return {a.x + b.x, a.y + b.y, a.z + b.z};
}
template <class R>
__device__ __forceinline__ V3<R> operator-(V3<R> a, V3<R> b) {
    return {a.x - b.x, a.y - b.y, a.z - b.z};
}
template <class R>
__device__ __forceinline__ V3<R> operator*(R s, V3<R> a) {
    return {s * a.x, s * a.y, s * a.z};
}
template <class R>
__device__ __forceinline__ V3<R>& operator+=(V3<R>& a, V3<R> b) {
    a.x += b.x;
    a.y += b.y;
    a.z += b.z;
    return a;
}
template <class R>
__device__ __forceinline__ R dot(V3<R> a, V3<R> b) {
    return a.x * b.x + a.y * b.y + a.z * b.z;
}
template <class R>
__device__ __forceinline__ V3<R> cross(V3<R> a, V3<R> b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

__device__ __forceinline__ double dsqrt(double x) { return __builtin_sqrt(x); }
__device__ __forceinline__ float dsqrt(float x) { return __builtin_sqrtf(x); }
__device__ __forceinline__ df64 dsqrt(df64 x) { return sqrt(x); }
template <class R>
__device__ __forceinline__ R rnorm(V3<R> a) {
    return num<R>(1.0) / dsqrt(dot(a, a));
}
__device__ __forceinline__ float rnorm(V3<float> a) { return 1.0f / dsqrt(dot(a, a)); }

constexpr uint8_t kBranchRegular = 0, kBranchSoftMissed = 1, kBranchSoftTIR = 2;

__device__ __forceinline__ bool in_piston(uint8_t s) {
    return s == MKO_STATUS_OK || s == MKO_STATUS_SOFT_MISSED || s == MKO_STATUS_SOFT_TIR;
}
__device__ __forceinline__ bool is_soft(uint8_t s) {
    return s == MKO_STATUS_SOFT_MISSED || s == MKO_STATUS_SOFT_TIR;
}

// Division, reciprocal and square root of the FP64 traces and of the reverse sweep: hardware
// reciprocal / reciprocal square root refined by Newton steps (a few ulp) instead of the correctly
// rounded IEEE sequences with their scaling and fix-up steps. These paths need ~1e-15 relative
// accuracy (Jacobian columns are compared to 1e-10, OPD to 1e-12 mm per ray); the df64 trace keeps its
// own operations.
// Measured on MI355X (2^20 arguments over 2^+-30): v_rcp_f64 and v_rsq_f64 are accurate to
// ~5e-8; one Newton step gives 2.1e-15, two give <= 0.5 ulp. The quotient a * r with one residual
// correction and the square root after one Goldschmidt step plus one correction are within
// 0.5 ulp (1.1e-16) as well.
__device__ __forceinline__ double rcp_nr1(double b) {
    const double r = __builtin_amdgcn_rcp(b);
    return __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
}
__device__ __forceinline__ double rev_rcp(double b) {
    const double r = rcp_nr1(b);
    return __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
}
__device__ __forceinline__ double rev_div(double a, double b) {
    const double r = rcp_nr1(b);
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}
__device__ __forceinline__ double rev_sqrt(double x) {
    if (!(x > 0.0)) return __builtin_sqrt(x);
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    const double d = __builtin_fma(-g, g, x);
    return __builtin_fma(d, h, g);
}

// rev_sqrt that also returns 1 / (2 sqrt(x)): the Goldschmidt iteration's refined half reciprocal
// (~1e-15 relative), for callers that divide by twice the root.
__device__ __forceinline__ double rev_sqrt_half_rcp(double x, double& half_rcp) {
    if (!(x > 0.0)) {
        const double g = __builtin_sqrt(x);
        half_rcp = 0.5 / g;
        return g;
    }
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    const double d = __builtin_fma(-g, g, x);
    half_rcp = h;
    return __builtin_fma(d, h, g);
}

template <class R>
struct RayAdj {
    V3<R> p, d;
};

// Forward-trace division / square root: the Newton-refined forms above in double, df64's own.
__device__ __forceinline__ double fdiv(double a, double b) { return rev_div(a, b); }
__device__ __forceinline__ df64 fdiv(df64 a, df64 b) { return a / b; }
__device__ __forceinline__ double fsqrt(double x) { return rev_sqrt(x); }
__device__ __forceinline__ df64 fsqrt(df64 x) { return dsqrt(x); }

// Accumulator of soft ray failure (SoftFailure, surface_ops.hpp:94).
struct Soft {
    double penalty;
    uint8_t first;
    __device__ __forceinline__ void add(double amount, uint8_t kind) {
        penalty += amount;
        if (first == MKO_STATUS_OK) first = kind;
    }
};

template <class R>
struct RayT {
    V3<R> p, d;
    R opl;
};
using Ray = RayT<double>;

// One surface step in df64 (propagate_surface_local with transfer, sphere intersection and
// refraction; FP64 traces take momentum_step). c = effective curvature (0 for stop and plane), t =
// vertex distance from the previous surface, nb = medium before, mu = nb / n_after. Returns a
// TraceStatus (Ok also for soft continuations, whose kind goes to `soft` and whose branch bits go
// to `branch`).
template <bool kSoft, class R>
__device__ __forceinline__ uint8_t surface_step(RayT<R>& r, R c, R t, R nb, R mu, Soft& soft,
                                                uint8_t& branch) {
    const R zero = num<R>(0.0), one = num<R>(1.0);
    if (!(r.d.z > zero)) return MKO_STATUS_BACKWARD;
    // transfer_to_tangent_plane
    r.p.z -= t;
    const R s0 = fdiv(-r.p.z, r.d.z);
    r.p.x += s0 * r.d.x;
    r.p.y += s0 * r.d.y;
    r.p.z = zero;
    // intersect_sphere
    const R H = c * (r.p.x * r.p.x + r.p.y * r.p.y);
    const R B = r.d.z - c * (r.p.x * r.d.x + r.p.y * r.d.y);
    const R D = B * B - c * H;
    R s;
    bool missed = false;
    if (D < zero) {
        if (!kSoft || (!(c > zero) && !(c < zero))) return MKO_STATUS_MISSED;
        soft.add(-to_double(D), MKO_STATUS_SOFT_MISSED);
        s = B / c;
        missed = true;
    } else {
        const R denom = B + fsqrt(D);
        if (!(denom > zero)) return MKO_STATUS_MISSED;
        s = fdiv(H, denom);
    }
    r.p = r.p + s * r.d;
    r.opl += nb * (s0 + s);
    // refract_sphere
    V3<R> N{-c * r.p.x, -c * r.p.y, one - c * r.p.z};
    if (kSoft && missed) N = rnorm(N) * N;
    const R cosI = dot(r.d, N);
    const R k = one - mu * mu * (one - cosI * cosI);
    if (k < zero) {
        if (!kSoft) return MKO_STATUS_TIR;
        soft.add(-to_double(k), MKO_STATUS_SOFT_TIR);
        const V3<R> tau = r.d - cosI * N;
        r.d = rnorm(tau) * tau;
        branch = uint8_t((missed ? kBranchSoftMissed : 0) | kBranchSoftTIR);
        return MKO_STATUS_OK;
    }
    r.d = mu * r.d + (fsqrt(k) - mu * cosI) * N;
    branch = missed ? kBranchSoftMissed : kBranchRegular;
    return MKO_STATUS_OK;
}

// reference_sphere_step (kind last_surface) / image_sphere_step (image kinds).
template <bool kSoft, class R>
__device__ __forceinline__ uint8_t reference_step(RayT<R>& r, V3<R> M, R kappa, int kind,
                                                  R n_image, Soft& soft, uint8_t& branch) {
    const R zero = num<R>(0.0), one = num<R>(1.0);
    const V3<R> q = r.p - M;
    const R b = -dot(q, r.d);
    branch = kBranchRegular;
    if (kind == MKO_REF_LAST_SURFACE) {
        const R g = dot(r.p, r.p - num<R>(2.0) * M);
        const R disc = b * b - g;
        if (disc < zero) {
            const R radius_sq = dot(M, M);
            if (!kSoft || !(radius_sq > zero)) return MKO_STATUS_MISSED;
            soft.add(-to_double(disc) / to_double(radius_sq), MKO_STATUS_SOFT_MISSED);
            r.p = r.p + b * r.d;
            r.opl += n_image * b;
            branch = kBranchSoftMissed;
            return MKO_STATUS_SOFT_MISSED;
        }
        const R root = fsqrt(disc);
        const bool real_image = M.z >= zero;
        const R denom = real_image ? b + root : b - root;
        if (!(real_image ? denom > zero : denom < zero)) return MKO_STATUS_MISSED;
        const R s = fdiv(g, denom);
        r.p = r.p + s * r.d;
        r.opl += n_image * s;
        return MKO_STATUS_OK;
    }
    const V3<R> cq = cross(q, r.d);
    const R t = -dot(cq, cq);
    const R disc = one + kappa * kappa * t;
    R step;
    uint8_t st = MKO_STATUS_OK;
    if (disc >= zero) {
        step = b - fdiv(kappa * t, fsqrt(disc) + one);
    } else if (kSoft && disc < zero) {
        step = b - kappa * t;
        st = MKO_STATUS_SOFT_MISSED;
    } else {
        return MKO_STATUS_MISSED;
    }
    if (!(step >= zero) && !(step < zero)) return MKO_STATUS_MISSED;
    if (st == MKO_STATUS_SOFT_MISSED) {
        soft.add(-to_double(disc), MKO_STATUS_SOFT_MISSED);
        branch = kBranchSoftMissed;
    }
    r.p = r.p + b * r.d;
    r.opl += n_image * step;
    return st;
}

// ---- reverse sweep ------------------------------------------------------------------------------

// Reverse of one stop/plane/sphere step (refracting_step_backward). (p, d): state before the
// surface; adj: adjoint of the state after it on entry, of the state before it on return.
// Adds the adjoints of the vertex distance t, the curvature c and the indices to tb/cb/nbb/nab.
template <class R>
__device__ __forceinline__ void refracting_step_backward(V3<R> p, V3<R> d, R t, R c, R n_before,
                                                         R n_after, uint8_t branch, R seed_opl,
                                                         R seed_pen, RayAdj<R>& adj, R& tb,
                                                         R& cb_out, R& nbb, R& nab) {
    const R z = p.z - t;
    const R rdz = rev_rcp(d.z);
    const R s0 = -z * rdz;
    const R x = p.x + s0 * d.x;
    const R y = p.y + s0 * d.y;
    const R rr = x * x + y * y;
    const R H = c * rr;
    const R xd = x * d.x + y * d.y;
    const R B = d.z - c * xd;
    const R D = B * B - c * H;
    const bool missed = (branch & kBranchSoftMissed) != 0;
    const bool tir = (branch & kBranchSoftTIR) != 0;
    R root_d = R(0);
    R s;
    if (missed) {
        s = B / c;
    } else {
        root_d = rev_sqrt(D);
        s = rev_div(H, B + root_d);
    }
    const V3<R> q{x + s * d.x, y + s * d.y, s * d.z};
    const V3<R> n_raw{-c * q.x, -c * q.y, R(1) - c * q.z};
    R inv_norm = R(1);
    V3<R> N = n_raw;
    if (missed) {
        inv_norm = rnorm(n_raw);
        N = inv_norm * n_raw;
    }
    const R mu = rev_div(n_before, n_after);
    const R cos_i = dot(d, N);
    const R sin2 = R(1) - cos_i * cos_i;
    const R k = R(1) - mu * mu * sin2;

    const V3<R> qb_out = adj.p;
    const V3<R> d1b = adj.d;
    RayAdj<R> in{{R(0), R(0), R(0)}, {R(0), R(0), R(0)}};
    V3<R> nb{R(0), R(0), R(0)};
    R cosb = R(0), kb = R(0), mub = R(0);
    if (tir) {
        const V3<R> tau = d - cos_i * N;
        const R inv_tau = rnorm(tau);
        const V3<R> d1 = inv_tau * tau;
        const V3<R> taub = inv_tau * (d1b - dot(d1, d1b) * d1);
        in.d += taub;
        cosb += -dot(taub, N);
        nb += (-cos_i) * taub;
        kb += -seed_pen;
    } else {
        const R root_k = rev_sqrt(k);
        const R a = root_k - mu * cos_i;
        in.d += mu * d1b;
        nb += a * d1b;
        const R ab = dot(d1b, N);
        mub += dot(d1b, d);
        kb += rev_div(ab, R(2) * root_k);
        mub += -ab * cos_i;
        cosb += -ab * mu;
    }
    mub += -kb * R(2) * mu * sin2;
    cosb += kb * R(2) * mu * mu * cos_i;
    in.d += cosb * N;
    nb += cosb * d;
    nbb += mub / n_after;
    nab += -mub * mu / n_after;
    V3<R> nrb = nb;
    if (missed) nrb = inv_norm * (nb - dot(N, nb) * N);
    const V3<R> qb = qb_out + (-c) * nrb;
    R cb = -dot(q, nrb);
    R xb = qb.x;
    R yb = qb.y;
    R sb = dot(qb, d);
    in.d += s * qb;
    sb += seed_opl * n_before;
    R s0b = seed_opl * n_before;
    nbb += seed_opl * (s0 + s);
    R hb = R(0), bb = R(0);
    if (missed) {
        bb += sb / c;
        cb += -sb * s / c;
        const R db = -seed_pen;
        bb += db * R(2) * B;
        cb += -db * H;
        hb += -db * c;
    } else {
        const R inv = rev_rcp(R(2) * root_d);
        hb += sb * inv;
        bb += -sb * s * R(2) * inv;
        cb += sb * s * s * inv;
    }
    cb += hb * rr;
    xb += hb * R(2) * c * x;
    yb += hb * R(2) * c * y;
    in.d.z += bb;
    cb += -bb * xd;
    xb += -bb * c * d.x;
    yb += -bb * c * d.y;
    in.d.x += -bb * c * x;
    in.d.y += -bb * c * y;
    // transfer
    in.p.x += xb;
    in.p.y += yb;
    s0b += xb * d.x + yb * d.y;
    in.d.x += xb * s0;
    in.d.y += yb * s0;
    const R qq = s0b * rdz;
    tb += qq;
    in.p.z += -qq;
    in.d.z += -qq * s0;
    cb_out += cb;
    adj = in;
}

// Reverse of the reference-sphere step; returns the adjoint of M_z (the working distance) and
// adds the adjoint of the image-space index to nib.
template <class R>
__device__ __forceinline__ R reference_step_backward(V3<R> p, V3<R> d, V3<R> M, R kappa, int kind,
                                                     R n_image, uint8_t branch, R seed_opl,
                                                     R seed_pen, RayAdj<R>& adj, R& nib) {
    const V3<R> q = p - M;
    const R b = -dot(q, d);
    const bool missed = (branch & kBranchSoftMissed) != 0;
    V3<R> center_adj{R(0), R(0), R(0)};
    if (kind == MKO_REF_LAST_SURFACE) {
        const R g = dot(p, p - R(2) * M);
        const R disc = b * b - g;
        const R sigma = M.z >= R(0) ? R(1) : R(-1);
        R s, root = R(0);
        if (missed) {
            s = b;
        } else {
            root = dsqrt(disc);
            s = g / (b + sigma * root);
        }
        const R sb = seed_opl * n_image;
        nib += seed_opl * s;
        R bb, gb;
        if (missed) {
            bb = sb;
            gb = R(0);
            const R radius_sq = dot(M, M);
            const R discb = -seed_pen / radius_sq;
            bb += discb * R(2) * b;
            gb += -discb;
            center_adj += (seed_pen * R(2) * disc / (radius_sq * radius_sq)) * M;
        } else {
            gb = sb * sigma / (R(2) * root);
            bb = -sb * sigma * s / root;
        }
        RayAdj<R> in{{R(0), R(0), R(0)}, {R(0), R(0), R(0)}};
        in.p += (-bb) * d;
        in.d += (-bb) * q;
        center_adj += bb * d;
        in.p += (R(2) * gb) * (p - M);
        center_adj += (R(-2) * gb) * p;
        adj = in;
        return center_adj.z;
    }
    const V3<R> c = cross(q, d);
    const R t = -dot(c, c);
    R step, dstep_dt, tb = R(0);
    if (missed) {
        step = b - kappa * t;
        dstep_dt = -kappa;
        tb += seed_pen * (-(kappa * kappa));
    } else {
        const R u = dsqrt(R(1) + kappa * kappa * t);
        step = b - kappa * t / (u + R(1));
        dstep_dt = -kappa / (R(2) * u);
    }
    const R sb = seed_opl * n_image;
    nib += seed_opl * step;
    const R bb = sb;
    tb += sb * dstep_dt;
    const V3<R> qb = (-bb) * d + (R(-2) * tb) * cross(d, c);
    const V3<R> db = (-bb) * q + (R(-2) * tb) * cross(c, q);
    adj.p = qb;
    adj.d = db;
    center_adj += (R(-1)) * qb;
    return center_adj.z;
}

// ---- the trace and the reverse sweep in optical direction cosines ---------------------------------
//
// State on a surface: the point p in its frame and the momentum P = n d (n d the optical direction
// cosines). Constants of the step from surface s - 1 to s, staged once per (variant, wavelength);
// 64 bytes, read as 16-byte words by wave-uniform addresses.
struct alignas(16) Step {
    double c;   // effective curvature of surface s (0 for stop and plane)
    double t;   // vertex distance from surface s - 1 to s
    double ni2; // -1 / n^2, n the medium before the surface
    double n2;  // n^2
    double cn2; // c n^2
    double dn2; // n_after^2 - n^2
    double n;   // n_after
    double cna; // c n_after^2
};

// sqrt(x) and 1 / (2 sqrt(x)) from the estimate y of 1 / sqrt(x): rev_sqrt_half_rcp's iteration.
__device__ __forceinline__ double sqrt_from(double x, double y, double& half_rcp) {
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    half_rcp = h;
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
// sqrt(x) for x > 0 without a branch; 0 for x = 0. A negative or NaN x gives an unspecified value:
// the steps test x.
__device__ __forceinline__ double sqrt_pos(double x) {
    double h;
    return sqrt_from(x, __builtin_amdgcn_rsq(__builtin_fmax(x, 0x1p-900)), h);
}
// The root of a squared P . N that the reverse sweep forms from the way back, and 1 / (2 root). The
// trace accepted the ray with a square >= 0; rounding, some 2^-52 n^2, may leave this one below zero
// where the ray grazes the surface, so it is held at `least`, 2^-54 of the first medium's n^2
// (sweep_least): the gradients stay those of a grazing ray instead of overflowing. (2^-52 of each
// gap's n^2 would be one product more per surface, 2 % of the fused kernel's time.)
__device__ __forceinline__ double sweep_least(double n0) { return 0x1p-54 * (n0 * n0); }
__device__ __forceinline__ double sweep_root(double x, double least, double& half_rcp) {
    const double v = __builtin_fmax(x, least);
    return sqrt_from(v, __builtin_amdgcn_rsq(v), half_rcp);
}

// The line through Q (in the frame of surface s) along +-P: its point nearest the vertex, where
// Q0 . P = 0, then the sphere from there: with H = c |Q0|^2 - 2 Q0_z the incidence term
// (P . N)^2 = D = P_z^2 - c n^2 H, the distance (in units of P) to the sphere is H / (P_z +
// sqrt(D)), without cancellation for P_z > 0, and P . N = sqrt(D) there (N the unit normal towards
// +z). No division by d_z, no product of direction and normal: one division and one root.
struct StepFoot {
    double l0, x, y, z, H, E, D;
};
__device__ __forceinline__ StepFoot step_foot(V3<double> Q, V3<double> P, double c, double ni2,
                                              double cn2) {
#pragma clang fp contract(off)
    StepFoot f;
    f.l0 = __builtin_fma(Q.z, P.z, __builtin_fma(Q.y, P.y, Q.x * P.x)) * ni2;
    f.x = __builtin_fma(f.l0, P.x, Q.x);
    f.y = __builtin_fma(f.l0, P.y, Q.y);
    f.z = __builtin_fma(f.l0, P.z, Q.z);
    const double q2 = __builtin_fma(f.z, f.z, __builtin_fma(f.y, f.y, f.x * f.x));
    f.H = __builtin_fma(c, q2, -(f.z + f.z));
    f.E = P.z * P.z;
    f.D = __builtin_fma(-cn2, f.H, f.E);
    return f;
}

// P + g N, N the unit normal at p. N_z first, then g N_z into P_z: the rounding of a sum P_z + g before
// the rest of the term is that of a number of n's size, and P strays further from Snell's law and from
// length n (path lengths 1.05 times further off, of rays near a failure 1.27 times, at the same number
// of operations).
__device__ __forceinline__ V3<double> add_normal(V3<double> P, double g, V3<double> p, double c) {
#pragma clang fp contract(off)
    const double cg = c * g, Nz = __builtin_fma(-c, p.z, 1.0);
    return V3<double>{__builtin_fma(-cg, p.x, P.x), __builtin_fma(-cg, p.y, P.y),
                      __builtin_fma(g, Nz, P.z)};
}

// One surface step in hard failure mode: (p, P, opl) from surface s - 1 to s. Every operation runs
// for every ray and one test ends a failed one (precedence: backward, missed, TIR; its state is
// then of no use). Missed: no intersection (D < 0), or the ray meets the tangent plane beyond the
// sphere's visible cap (d_z - c (x d_x + y d_y) <= 0 there, the reference's intersect_sphere),
// which is P_z^2 + c n^2 Q0_z <= 0. Products and sums are spelled out, so that every kernel that
// inlines the step computes the same bits. a: P . N at the surface.
__device__ __forceinline__ uint8_t momentum_step(V3<double>& p, V3<double>& P, double& opl,
                                                 const Step& k, double& a) {
#pragma clang fp contract(off)
    const StepFoot f = step_foot(V3<double>{p.x, p.y, p.z - k.t}, P, k.c, k.ni2, k.cn2);
    const bool backward = !(P.z > 0.0);
    a = sqrt_pos(f.D);
    const double lam = rev_div(f.H, P.z + a);
    p = V3<double>{__builtin_fma(lam, P.x, f.x), __builtin_fma(lam, P.y, f.y),
                   __builtin_fma(lam, P.z, f.z)};
    opl = __builtin_fma(k.n2, f.l0 + lam, opl);
    const double k2 = f.D + k.dn2;
    P = add_normal(P, sqrt_pos(k2) - a, p, k.c);
    const bool missed = !(f.D >= 0.0) || !(__builtin_fma(k.cn2, f.z, f.E) > 0.0);
    if (backward || missed || k2 < 0.0) [[unlikely]]
        return backward ? uint8_t(MKO_STATUS_BACKWARD)
               : missed ? uint8_t(MKO_STATUS_MISSED)
                        : uint8_t(MKO_STATUS_TIR);
    return MKO_STATUS_OK;
}

// Soft continuations of a step (rare): p on the surface or, after a miss, nearest the sphere's
// centre; a = P . N and k2 = a^2 + dn2 of a hit. Direction space: unit normal after a miss, TIR
// continues along the surface tangent.
__device__ __forceinline__ void soft_refract(V3<double> p, V3<double>& P, const Step& k, double nb,
                                             double a, double k2, bool missed, Soft& soft,
                                             uint8_t& branch) {
#pragma clang fp contract(off)
    V3<double> N{-k.c * p.x, -k.c * p.y, __builtin_fma(-k.c, p.z, 1.0)};
    const V3<double> d{P.x / nb, P.y / nb, P.z / nb};
    const double mu = nb / k.n;
    double cosI = a / nb, kk = k2 / (k.n * k.n);
    if (missed) {
        const double w = 1.0 / __builtin_sqrt(N.x * N.x + N.y * N.y + N.z * N.z);
        N = V3<double>{w * N.x, w * N.y, w * N.z};
        cosI = d.x * N.x + d.y * N.y + d.z * N.z;
        kk = 1.0 - mu * mu * (1.0 - cosI * cosI);
    }
    branch = missed ? kBranchSoftMissed : kBranchRegular;
    V3<double> e;
    if (kk < 0.0) {
        soft.add(-kk, MKO_STATUS_SOFT_TIR);
        branch = uint8_t(branch | kBranchSoftTIR);
        e = V3<double>{d.x - cosI * N.x, d.y - cosI * N.y, d.z - cosI * N.z};
        const double w = 1.0 / __builtin_sqrt(e.x * e.x + e.y * e.y + e.z * e.z);
        e = V3<double>{w * e.x, w * e.y, w * e.z};
    } else {
        const double g = __builtin_sqrt(kk) - mu * cosI;
        e = V3<double>{mu * d.x + g * N.x, mu * d.y + g * N.y, mu * d.z + g * N.z};
    }
    P = V3<double>{k.n * e.x, k.n * e.y, k.n * e.z};
}

// The step in soft failure mode (nb: the medium before): a miss on a curved surface continues from
// the line's point nearest the sphere's centre (the vertex of the intersection's quadratic), TIR
// along the surface, each adding its penalty; a regular ray takes momentum_step's operations.
__device__ __forceinline__ uint8_t momentum_step_soft(V3<double>& p, V3<double>& P, double& opl,
                                                      const Step& k, double nb, double& a,
                                                      Soft& soft, uint8_t& branch) {
#pragma clang fp contract(off)
    if (!(P.z > 0.0)) return MKO_STATUS_BACKWARD;
    const StepFoot f = step_foot(V3<double>{p.x, p.y, p.z - k.t}, P, k.c, k.ni2, k.cn2);
    double lam;
    const bool missed = f.D < 0.0;
    a = 0.0;
    if (missed) {
        if (!(k.c > 0.0) && !(k.c < 0.0)) return MKO_STATUS_MISSED;
        soft.add(f.D * k.ni2, MKO_STATUS_SOFT_MISSED);
        lam = P.z / k.cn2;
    } else {
        a = sqrt_pos(f.D);
        if (!(f.D >= 0.0) || !(__builtin_fma(k.cn2, f.z, f.E) > 0.0)) return MKO_STATUS_MISSED;
        lam = rev_div(f.H, P.z + a);
    }
    p = V3<double>{__builtin_fma(lam, P.x, f.x), __builtin_fma(lam, P.y, f.y),
                   __builtin_fma(lam, P.z, f.z)};
    opl = __builtin_fma(k.n2, f.l0 + lam, opl);
    const double k2 = f.D + k.dn2;
    if (missed || k2 < 0.0) [[unlikely]] {
        soft_refract(p, P, k, nb, a, k2, missed, soft, branch);
        return MKO_STATUS_OK;
    }
    P = add_normal(P, sqrt_pos(k2) - a, p, k.c);
    branch = kBranchRegular;
    return MKO_STATUS_OK;
}

// Reverse sweep of one regular ray (no soft continuation) from its state on the last surface.
//
// By Fermat's principle the optical path to the reference sphere changes, for a change of a
// parameter, by the change of the path's own pieces at fixed points of incidence, plus P . dE for
// the displacement dE of the ray's end on the reference sphere, which is not zero where the ray
// leaves the sphere's normal. That second part is a linear functional of the ray; pulled back
// through the system it is carried by one neighbouring ray (dq, dP), because the map of rays is
// symplectic. So with K the change of the local path as a function of the ray,
//     d(OPL)/d(theta) = K + dK along (dq, dP):
//   thickness t_s:  K = P_z in the gap
//   curvature c_j:  K = (P . N - P' . N) |q|^2 / 2 (the surface moves along N by |q|^2 / 2)
//   index n_s:      K = the length of the ray in the medium
// The sweep traces the ray backwards (no record of its states) and the neighbouring ray with it.
// A general adjoint state (six components through every operation of the step) took 162 vector
// instructions per surface, this form about 90. Equivalent to backward_ray's sums
// (adjoint_backward.hpp:119-241), checked against them and against 64-bit tangents.
struct SweepState {
    V3<double> q, P, dq, dP, N;
    double a, ha; // P . N and 1 / (2 P . N)
};

// The neighbouring ray of a linear functional A . dq + B . dP of the ray (p, P) on a surface with
// normal N: dq = B modulo P on the tangent plane, dP = -A modulo N and normal to P.
__device__ __forceinline__ SweepState sweep_start(V3<double> p, V3<double> P, V3<double> A,
                                                  V3<double> B, double c) {
    SweepState w;
    w.q = p;
    w.P = P;
    w.N = V3<double>{-c * p.x, -c * p.y, 1.0 - c * p.z};
    w.a = dot(P, w.N);
    const double ra = rev_rcp(w.a);
    w.ha = 0.5 * ra;
    const double mu = dot(w.N, B) * ra, nu = dot(P, A) * ra;
    w.dq = V3<double>{B.x - mu * P.x, B.y - mu * P.y, B.z - mu * P.z};
    w.dP = V3<double>{nu * w.N.x - A.x, nu * w.N.y - A.y, nu * w.N.z - A.z};
    return w;
}

// Backwards through the refraction at surface j (k: its step): P and dP become those before the
// surface; returns the curvature gradient. On entry a = P' . N.
__device__ __forceinline__ double sweep_refract(SweepState& w, const Step& k, double least) {
    double h;
    const double a = sweep_root(__builtin_fma(w.a, w.a, -k.dn2), least, h);
    const double g = w.a - a;
    const double u = dot(w.dP, w.N) - k.c * dot(w.P, w.dq); // change of P' . N
    const double dg = u * g * (h + h);                      // minus the change of g
    const double cg = k.c * g;
    w.P = V3<double>{w.P.x - g * w.N.x, w.P.y - g * w.N.y, w.P.z - g * w.N.z};
    w.dP = V3<double>{w.dP.x + (dg * w.N.x + cg * w.dq.x), w.dP.y + (dg * w.N.y + cg * w.dq.y),
                      w.dP.z + (dg * w.N.z + cg * w.dq.z)};
    const double r = 0.5 * dot(w.q, w.q);
    return dg * r - g * (r + dot(w.q, w.dq));
}

// Backwards through the gap between surface s = j - 1 (curvature c, cna = c n^2) and j (k: its
// step): the state and the neighbouring ray on surface s. kIndex: length is the gradient with
// respect to the gap's index.
template <bool kIndex>
__device__ __forceinline__ void sweep_transfer(SweepState& w, const Step& k, double c, double cna,
                                               double n, double least, double& length) {
    const StepFoot f = step_foot(V3<double>{w.q.x, w.q.y, w.q.z + k.t}, w.P, c, k.ni2, cna);
    w.a = sweep_root(f.D, least, w.ha);
    const double lam = rev_div(f.H, w.P.z + w.a);
    w.q = V3<double>{f.x + lam * w.P.x, f.y + lam * w.P.y, f.z + lam * w.P.z};
    const double back = f.l0 + lam; // q = Q + back P
    w.N = V3<double>{-c * w.q.x, -c * w.q.y, 1.0 - c * w.q.z};
    const double before = kIndex ? dot(w.P, w.dq) : 0.0;
    w.dq = V3<double>{w.dq.x + back * w.dP.x, w.dq.y + back * w.dP.y, w.dq.z + back * w.dP.z};
    const double mu = dot(w.N, w.dq) * (w.ha + w.ha);
    w.dq = V3<double>{w.dq.x - mu * w.P.x, w.dq.y - mu * w.P.y, w.dq.z - mu * w.P.z};
    if constexpr (kIndex) // n |back| + (P . dq_j - P . dq_s) / n, 1 / n = -n ni2
        length = -n * (back + k.ni2 * (before - dot(w.P, w.dq)));
}

// The functional of a regular ray at the reference sphere (reference_step): V = n step(p, d), A =
// dV/dp + P, B = dV/dP, and with it the sweep's start; mz: the gradient with respect to M_z, step:
// the path's length to the sphere.
__device__ __forceinline__ SweepState sweep_reference(V3<double> p, V3<double> d, V3<double> M,
                                                      double kappa, int kind, double n,
                                                      double c_last, double& mz, double& step) {
    const V3<double> q = p - M;
    const double b = -dot(q, d);
    const V3<double> P{n * d.x, n * d.y, n * d.z};
    V3<double> A, B;
    if (kind == MKO_REF_LAST_SURFACE) {
        const double g = dot(p, p - 2.0 * M);
        double h;
        const double root = rev_sqrt_half_rcp(b * b - g, h);
        const double sigma = M.z >= 0.0 ? 1.0 : -1.0;
        step = rev_div(g, b + sigma * root);
        const double gb = n * sigma * h;       // dV/dg
        const double bb = -2.0 * gb * step;    // dV/db
        const double wq = 2.0 * gb;
        A = V3<double>{P.x - bb * d.x + wq * q.x, P.y - bb * d.y + wq * q.y,
                       P.z - bb * d.z + wq * q.z};
        const double rb = -rev_div(bb, n);
        B = V3<double>{rb * q.x, rb * q.y, rb * q.z};
        mz = bb * d.z - wq * p.z;
    } else {
        const V3<double> cr = cross(q, d);
        const double t = -dot(cr, cr);
        double h;
        const double u = rev_sqrt_half_rcp(1.0 + kappa * kappa * t, h);
        step = b - kappa * rev_div(t, u + 1.0);
        const double tb = -n * kappa * h; // dV/dt
        const V3<double> dc = cross(d, cr), cq = cross(cr, q);
        const V3<double> pb{-n * d.x - 2.0 * tb * dc.x, -n * d.y - 2.0 * tb * dc.y,
                            -n * d.z - 2.0 * tb * dc.z};
        A = pb + P;
        const double rn = rev_rcp(n);
        B = V3<double>{-q.x - 2.0 * tb * cq.x * rn, -q.y - 2.0 * tb * cq.y * rn,
                       -q.z - 2.0 * tb * cq.z * rn};
        mz = -pb.z;
    }
    return sweep_start(p, P, A, B, c_last);
}

} // namespace mkod
