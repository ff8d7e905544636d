// gfx950 kernels of the batched forward-and-Jacobian path and their device-level C entry points.
//
// Work decomposition, where a kernel's own comment says nothing else: one workgroup per (variant,
// tuple), tuple = (field f, wavelength l), t = f * L + l, of 256 lanes or of the waves that the
// largest tuple's rays fill; the tuple's rays sit on lanes, ray k on lane k mod lanes (iteration k /
// lanes). Small tuples share workgroups (trace_pack_kernel, prefilter_kernel). The surface table of
// the (variant, wavelength) is staged once per workgroup in LDS (Step: curvature, vertex distance and
// the products of the media that a step takes; the df64 trace: curvature, vertex distance, index, mu =
// n/n'), so the per-ray surface loop reads wave-uniform LDS broadcasts. Every reduction over rays
// (piston, merit partials, piston projection of the Jacobian) has a fixed order: lane-local sum in
// iteration order, xor-butterfly inside the wave, waves summed in index order; results depend only
// on the tuple, never on the batch composition or the launch.
//
// Reference counterparts: residuals_kernel src/cuda/residuals.cu:58, merit_kernel +
// merit_finalize_kernel src/cuda/merit.cu:63/207, fd_difference_kernel src/cuda/fd_jacobian.cu:65,
// adjoint_jacobian_kernel src/cuda/adjoint_jacobian.cu:119, gram_kernel
// src/cuda/normal_equations.cu:48.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <cstdio>
#include <mutex>
#include <stdexcept>
#include <string>
#include <type_traits>

#include "error.hpp"
#include "gauss_legendre_table.h"
#include "internal.hpp"
#include "launch_plan.hpp"
#include "mikroptim_hip.h"
#include "constraints.hpp"
#include "trace_device.hpp"

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kMaxFields = 32;
constexpr int kMaxWavelengths = 32;
constexpr int kMaxRaysPerLane = 8; // tuples of at most 2048 rays
constexpr double kPi = 3.14159265358979323846264338327950288;

using mkod::Ray;
using mkod::Soft;
using mkod::V3;

// Everything a trace kernel needs, passed by value (< 1.5 KB of kernel arguments).
struct TraceParams {
    const double* curvature;
    const double* thickness;
    const double* index;
    const double* pupil_radius;
    const double* field_angle;
    const double* field_target;
    const double* reference_curvature;
    int V, S, L, F, T;
    int source, ref_kind;
    int rings, spokes, soft, precision;
    double fail_weight;
    double lambda_ref_nm;
    double src_pt[3];
    double src_na;
    uint64_t sphere_mask;
    uint64_t ext_mask; // surfaces whose extrema a kExt trace reduces
    // device count of the variants to trace (NULL: all V): blocks of variants >= *live exit at
    // once, so that a launch sized for V serves a captured LM cycle whose count the device sets
    const int32_t* live;
    int64_t rays, trace_rows, stride;
    double gl_u[MKO_MAX_RINGS], gl_w[MKO_MAX_RINGS];
    double field_weight[kMaxFields];
    double wavelength_weight[kMaxWavelengths];
    uint8_t pupil_mode[kMaxFields];
};

// Adjoint column map: variable index of curvature[s] / thickness[s] (-1 if not a variable).
struct ParamMap {
    int P;
    // 32-bit entries (here and in glass_col): the reverse sweeps index them by the (uniform)
    // surface, which scalar loads from the kernel arguments serve only at dword granularity
    int32_t curv_col[MKO_MAX_SURFACES];
    int32_t thick_col[MKO_MAX_SURFACES];
    // glass variables (AdjointParameterMap::glass / glass_slope, ray_jacobian.hpp:28-38): the
    // variables of (n0, nu1, nu2) of the medium after surface s, and the Buchdahl coordinate
    // w_l of each wavelength (dn/d(n0, nu1, nu2) = 1, w_l, w_l^2)
    int glass;
    int32_t glass_col[MKO_MAX_SURFACES][3];
    double omega[kMaxWavelengths];
    // columns that no ray's sweep reaches (bit p): the curvature of a stop or plane, the index of
    // the medium before the first surface
    uint64_t unswept[2];
};

// ---- tuple geometry ------------------------------------------------------------------------

struct Tuple {
    int v, f, l, n, M;
    int64_t offset;
    double scale, pscale;
};

__device__ __forceinline__ Tuple tuple_of(const TraceParams& P, int block) {
    Tuple t;
    t.v = block / P.T;
    const int tt = block - t.v * P.T;
    t.f = tt / P.L;
    t.l = tt - t.f * P.L;
    int64_t off = 0;
    for (int f = 0; f < t.f; ++f)
        off += int64_t(P.L) * P.rings * (P.pupil_mode[f] == MKO_PUPIL_AXIS ? 1 : P.spokes);
    t.M = P.pupil_mode[t.f] == MKO_PUPIL_AXIS ? 1 : P.spokes;
    t.n = P.rings * t.M;
    t.offset = off + int64_t(t.l) * t.n;
    // tuple_weight / residual_scale / penalty_scale (ray_residual.hpp:301-385): no a*b+c,
    // correctly rounded division and square root, hence bitwise equal to the host values.
    const double wf = P.field_weight[t.f];
    const double wl = P.wavelength_weight[t.l];
    double w = 0.0;
    if (wf > 0.0 && wl > 0.0) {
        double sf = 0.0, sl = 0.0;
        for (int i = 0; i < P.F; ++i) sf += P.field_weight[i];
        for (int i = 0; i < P.L; ++i) sl += P.wavelength_weight[i];
        w = __dmul_rn(__ddiv_rn(wf, sf), __ddiv_rn(wl, sl));
    }
    t.scale = w > 0.0 ? __ddiv_rn(__dsqrt_rn(w), __dmul_rn(P.lambda_ref_nm, 1e-6)) : 0.0;
    t.pscale = w > 0.0 ? __dsqrt_rn(__dmul_rn(P.fail_weight, w)) : 0.0;
    return t;
}

struct Sample {
    double rho, sphi, cphi, weight, rootw;
};

// PupilQuadrature::sample (quadrature.hpp:71-92): ring-major index k = i * M + j; ring i gives
// the radius and the weights, spoke j the angle.
__device__ __forceinline__ void ring_of(const TraceParams& P, const Tuple& t, int i, Sample& s) {
    s.rho = __dsqrt_rn(P.gl_u[i]);
    s.weight = __ddiv_rn(P.gl_w[i], double(t.M));
    s.rootw = __dsqrt_rn(s.weight);
}
__device__ __forceinline__ void spoke_of(const TraceParams& P, const Tuple& t, int j, Sample& s) {
    const uint8_t mode = P.pupil_mode[t.f];
    double phi = 0.0;
    if (mode == MKO_PUPIL_HALF)
        phi = __ddiv_rn(__dmul_rn(double(2 * j + 1), kPi), double(2 * t.M));
    else if (mode == MKO_PUPIL_FULL)
        phi = __ddiv_rn(__dmul_rn(double(2 * j + 1), kPi), double(t.M));
    if (mode == MKO_PUPIL_AXIS) {
        s.sphi = 0.0;
        s.cphi = 1.0;
    } else {
        sincos(phi, &s.sphi, &s.cphi);
    }
}
__device__ __forceinline__ Sample sample_of(const TraceParams& P, const Tuple& t, int k) {
    const int i = k / t.M;
    const int j = k - i * t.M;
    Sample s;
    ring_of(P, t, i, s);
    spoke_of(P, t, j, s);
    return s;
}

// The tuple's ring and spoke values in LDS, formed once per workgroup by the functions above (the
// same bits as sample_of): a ray's sample is then two table reads instead of a square root, a
// division and an FP64 sincos per ray. Tuples with more spokes than the table holds compute
// their samples per ray.
constexpr int kTableSpokes = 128;
struct SampleTable {
    double rho[MKO_MAX_RINGS], weight[MKO_MAX_RINGS], rootw[MKO_MAX_RINGS];
    double sphi[kTableSpokes], cphi[kTableSpokes];
};
// The caller's next __syncthreads publishes the table.
__device__ __forceinline__ void stage_samples(const TraceParams& P, const Tuple& t,
                                              SampleTable& T) {
    if (t.M > kTableSpokes) return;
    const int x = threadIdx.x;
    if (x < P.rings) {
        Sample s;
        ring_of(P, t, x, s);
        T.rho[x] = s.rho;
        T.weight[x] = s.weight;
        T.rootw[x] = s.rootw;
    }
    for (int j = x; j < t.M; j += int(blockDim.x)) {
        Sample s;
        spoke_of(P, t, j, s);
        T.sphi[j] = s.sphi;
        T.cphi[j] = s.cphi;
    }
}
__device__ __forceinline__ Sample sample_at(const TraceParams& P, const Tuple& t,
                                            const SampleTable& T, int k) {
    if (t.M > kTableSpokes) return sample_of(P, t, k);
    const int i = k / t.M;
    const int j = k - i * t.M;
    return Sample{T.rho[i], T.sphi[j], T.cphi[j], T.weight[i], T.rootw[i]};
}

// Surface table of (variant, wavelength) in LDS for the df64 trace.
struct PlainLds {
    double c[MKO_MAX_SURFACES];  // effective curvature (0 for stop/plane)
    double t[MKO_MAX_SURFACES];  // thickness[s]
    double n[MKO_MAX_SURFACES];  // index[s][l]
    double mu[MKO_MAX_SURFACES]; // n[s-1] / n[s]
};

// Step table of (variant, wavelength): L[s] the step to surface s, L[S].t the working distance.
// The caller's next __syncthreads publishes it.
using mkod::Step;
__device__ __forceinline__ Step step_at(const TraceParams& P, int v, int l, int s) {
    const size_t vs = size_t(v) * P.S + s;
    Step k{};
    if (s > 0) k.t = P.thickness[vs - 1];
    if (s < P.S) {
        k.c = ((P.sphere_mask >> s) & 1ull) ? P.curvature[vs] : 0.0;
        k.n = P.index[vs * P.L + l];
        k.cna = k.c * (k.n * k.n);
        if (s > 0) {
            const double nb = P.index[(vs - 1) * P.L + l];
            k.n2 = nb * nb;
            k.ni2 = __ddiv_rn(-1.0, k.n2);
            k.cn2 = k.c * k.n2;
            k.dn2 = (k.n - nb) * (k.n + nb);
        }
    }
    return k;
}
__device__ __forceinline__ void stage_steps(const TraceParams& P, int v, int l, Step* L) {
    for (int s = threadIdx.x; s <= P.S; s += int(blockDim.x)) L[s] = step_at(P, v, l, s);
}

// The trace's table by its number type: the step table (double), the plain one (df64).
template <class R>
struct TraceTable;
template <>
struct TraceTable<double> {
    Step k[MKO_MAX_SURFACES + 1];
    using Ptr = const Step*;
    __device__ __forceinline__ Ptr ptr() const { return k; }
    // synchronises
    __device__ __forceinline__ void stage(const TraceParams& P, const Tuple& t) {
        stage_steps(P, t.v, t.l, k);
        __syncthreads();
    }
};
template <>
struct TraceTable<mkod::df64> {
    PlainLds p;
    using Ptr = const PlainLds*;
    __device__ __forceinline__ Ptr ptr() const { return &p; }
    __device__ __forceinline__ void stage(const TraceParams& P, const Tuple& t) {
        const int s = threadIdx.x;
        if (s < P.S) {
            const size_t vs = size_t(t.v) * P.S + s;
            p.c[s] = ((P.sphere_mask >> s) & 1ull) ? P.curvature[vs] : 0.0;
            p.t[s] = P.thickness[vs];
            p.n[s] = P.index[vs * P.L + t.l];
        }
        __syncthreads();
        if (s >= 1 && s < P.S) p.mu[s] = __ddiv_rn(p.n[s - 1], p.n[s]);
        __syncthreads();
    }
};
__device__ __forceinline__ double index_after(const Step* L, int s) { return L[s].n; }
__device__ __forceinline__ double index_after(const PlainLds* L, int s) { return L->n[s]; }
__device__ __forceinline__ double working_distance(const Step* L, int S) { return L[S].t; }
__device__ __forceinline__ double working_distance(const PlainLds* L, int S) { return L->t[S - 1]; }

__device__ __forceinline__ Ray source_ray(const TraceParams& P, const Tuple& t, const Sample& s,
                                          double a, double sin_t, double cos_t, double n0) {
    Ray r;
    if (P.source == MKO_SOURCE_POINT) {
        const double sin_max = P.src_na / n0;
        const double sr = sin_max * s.rho;
        r.p = V3<double>{P.src_pt[0], P.src_pt[1], P.src_pt[2]};
        r.d = V3<double>{sr * s.sphi, sr * s.cphi, __dsqrt_rn((1.0 - sr) * (1.0 + sr))};
        r.opl = 0.0;
        return r;
    }
    const double rad = a * s.rho;
    r.p = V3<double>{rad * s.sphi, rad * s.cphi, 0.0};
    r.d = V3<double>{0.0, sin_t, cos_t};
    r.opl = mkod::dot(r.p, r.d);
    return r;
}

// Record of one ray's states for the reverse sweep of a ray with soft continuations
// (AdjointRecord, adjoint_record.hpp:66): positions and optical direction cosines.
struct Record {
    V3<double> p[MKO_MAX_SURFACES], P[MKO_MAX_SURFACES];
    uint8_t branch[MKO_MAX_SURFACES];
    uint8_t image_branch;
    int count;
    __device__ __forceinline__ void put(int s, V3<double> q, V3<double> mom, uint8_t b) {
        p[s] = q;
        P[s] = mom;
        branch[s] = b;
        count = s + 1;
    }
};

struct NoRecord {
    uint8_t image_branch;
};

// Last state of a forward trace (the state on surface S-1, which the reference-sphere step starts
// from); the reverse sweep traces the ray backwards from there. The traces put it once, after the
// last surface: a ray that fails on the way leaves it unset, and the loop carries no copy of the
// state.
struct LastState {
    V3<double> p, d;
    uint8_t image_branch;
};

// One ray through the surfaces, r in its number type: step() takes r from surface s - 1 to s,
// cos_incidence() is cos I there (of a ray that step() found Ok), finish() leaves r's direction of
// unit length. In double, r.d holds the optical direction cosines on the way.
template <class R>
struct Tracer;
template <>
struct Tracer<double> {
    double a = 0.0; // P . N
    __device__ __forceinline__ void begin(const Step* L, Ray& r) {
        const double n0 = L[0].n;
        r.d = V3<double>{n0 * r.d.x, n0 * r.d.y, n0 * r.d.z};
    }
    template <bool kSoft, bool kCos>
    __device__ __forceinline__ uint8_t step(const Step* L, int s, Ray& r, Soft& soft,
                                            uint8_t& branch) {
        if constexpr (kSoft) {
            return mkod::momentum_step_soft(r.p, r.d, r.opl, L[s], L[s - 1].n, a, soft, branch);
        } else {
            branch = mkod::kBranchRegular;
            return mkod::momentum_step(r.p, r.d, r.opl, L[s], a);
        }
    }
    // (P . N) / n, 1 / n = n / n^2
    __device__ __forceinline__ double cos_incidence(const Step* L, int s, const Ray&) const {
#pragma clang fp contract(off)
        return a * (L[s - 1].n * -L[s].ni2);
    }
    __device__ __forceinline__ void finish(const Step* L, int S, Ray& r) const {
        const double rn = mkod::rev_rcp(L[S - 1].n);
        r.d = V3<double>{rn * r.d.x, rn * r.d.y, rn * r.d.z};
    }
};
template <>
struct Tracer<mkod::df64> {
    using R = mkod::df64;
    V3<double> before{}; // direction before the surface (kCos)
    __device__ __forceinline__ void begin(const PlainLds*, mkod::RayT<R>&) {}
    template <bool kSoft, bool kCos>
    __device__ __forceinline__ uint8_t step(const PlainLds* L, int s, mkod::RayT<R>& r, Soft& soft,
                                            uint8_t& branch) {
        using mkod::num;
        using mkod::to_double;
        if constexpr (kCos)
            before = V3<double>{to_double(r.d.x), to_double(r.d.y), to_double(r.d.z)};
        return mkod::surface_step<kSoft>(r, num<R>(L->c[s]), num<R>(L->t[s - 1]),
                                         num<R>(L->n[s - 1]), num<R>(L->mu[s]), soft, branch);
    }
    // d_before . N, N = (-c x, -c y, 1 - c z)
    __device__ __forceinline__ double cos_incidence(const PlainLds* L, int s,
                                                    const mkod::RayT<R>& r) const {
#pragma clang fp contract(off)
        const double c = L->c[s];
        return before.x * (-c * mkod::to_double(r.p.x)) + before.y * (-c * mkod::to_double(r.p.y)) +
               before.z * (1.0 - c * mkod::to_double(r.p.z));
    }
    __device__ __forceinline__ void finish(const PlainLds*, int, mkod::RayT<R>&) const {}
};

// The reference sphere from the state on the last surface: final status.
template <bool kSoft, class R, class Table, class Rec>
__device__ __forceinline__ uint8_t reference_end(const TraceParams& P, Table L, mkod::RayT<R>& r,
                                                 V3<double> M, double kappa, Soft& soft, Rec& rec) {
    using mkod::num;
    if (!(r.d.z > num<R>(0.0))) return MKO_STATUS_BACKWARD;
    uint8_t rb = 0;
    const uint8_t rst = mkod::reference_step<kSoft>(
        r, V3<R>{num<R>(M.x), num<R>(M.y), num<R>(M.z)}, num<R>(kappa), P.ref_kind,
        num<R>(index_after(L, P.S - 1)), soft, rb);
    if (!mkod::in_piston(rst)) return rst;
    rec.image_branch = rb;
    return kSoft ? soft.first : uint8_t(MKO_STATUS_OK);
}

// trace_to_reference_sphere (reference_sphere.hpp:183-222) over the LDS table, in the number
// type R of the ray (double, or df64 for MKO_PRECISION_DF64). Returns the final status;
// soft.penalty holds the accumulated penalty.
template <bool kSoft, class R, class Table, class Rec>
__device__ __forceinline__ uint8_t trace_ray(const TraceParams& P, Table L, mkod::RayT<R>& r,
                                             V3<double> M, double kappa, Soft& soft, Rec& rec) {
    constexpr bool kRecord = std::is_same_v<Rec, Record>;
    Tracer<R> tr;
    tr.begin(L, r);
    if constexpr (kRecord) rec.put(0, r.p, r.d, mkod::kBranchRegular);
    for (int s = 1; s < P.S; ++s) {
        uint8_t branch = 0;
        const uint8_t st = tr.template step<kSoft, false>(L, s, r, soft, branch);
        if (st != MKO_STATUS_OK) return st;
        if constexpr (kRecord) rec.put(s, r.p, r.d, branch);
    }
    tr.finish(L, P.S, r);
    if constexpr (std::is_same_v<Rec, LastState>) {
        rec.p = r.p;
        rec.d = r.d;
    }
    return reference_end<kSoft>(P, L, r, M, kappa, soft, rec);
}

// The start ray in the trace's number type (computed in double, then converted).
template <class R>
__device__ __forceinline__ mkod::RayT<R> ray_as(const Ray& r) {
    using mkod::num;
    return mkod::RayT<R>{V3<R>{num<R>(r.p.x), num<R>(r.p.y), num<R>(r.p.z)},
                         V3<R>{num<R>(r.d.x), num<R>(r.d.y), num<R>(r.d.z)}, num<R>(r.opl)};
}

// ---- surface extrema (SurfaceExtrema, include/mikroptim/trace/surface_extrema.hpp:47-110) -----

// height^2 = x^2 + y^2 at the intersection, each product and sum rounded on its own
// (RaySurfaceRecord::surface)
__device__ __forceinline__ double height_sq(double x, double y) {
#pragma clang fp contract(off)
    return x * x + y * y;
}

// trace_ray with the surface extrema of the wave's rays: at every surface s in P.ext_mask (0 =
// start state; the other surfaces keep the neutral 0 / 1),
// the largest height^2 and the smallest cos I over the wave's lanes whose ray is `alive` (has
// passed every surface so far) are reduced across the wave; lane s keeps surface s's values in
// eh / ec (S <= 64 = wave width), replacing them (merge = false) or folding them in (merge =
// true). Every lane of the wave calls this with the same P.S (uniform control flow around the
// cross-lane reductions); lanes without a ray pass alive = false.
template <bool kSoft, class R, class Table, class Rec>
__device__ __forceinline__ uint8_t trace_ray_ext(const TraceParams& P, Table L, mkod::RayT<R>& r,
                                                 V3<double> M, double kappa, Soft& soft, bool alive,
                                                 int lane, double& eh, double& ec, bool merge,
                                                 Rec& rec) {
    using mkod::to_double;
    auto reduce = [&](int s, double h, double c) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const double oh = __shfl_xor(h, off, 64);
            const double oc = __shfl_xor(c, off, 64);
            h = oh > h ? oh : h;
            c = oc < c ? oc : c;
        }
        if (lane == s) {
            eh = merge ? (h > eh ? h : eh) : h;
            ec = merge ? (c < ec ? c : ec) : c;
        }
    };
    uint8_t st = MKO_STATUS_OK;
    {
        double h = 0.0, c = 1.0;
        if (alive) {
            h = height_sq(to_double(r.p.x), to_double(r.p.y));
            c = to_double(r.d.z);
        }
        if (P.ext_mask & 1ull) reduce(0, h, c);
    }
    Tracer<R> tr;
    tr.begin(L, r);
    for (int s = 1; s < P.S; ++s) {
        double h = 0.0, c = 1.0;
        if (alive) {
            uint8_t branch = 0;
            const uint8_t sst = tr.template step<kSoft, true>(L, s, r, soft, branch);
            if (sst != MKO_STATUS_OK) {
                alive = false;
                st = sst;
            } else {
                h = height_sq(to_double(r.p.x), to_double(r.p.y));
                c = tr.cos_incidence(L, s, r);
            }
        }
        if ((P.ext_mask >> s) & 1ull) reduce(s, h, c); // uniform: P.ext_mask is a kernel argument
    }
    if (!alive) return st;
    tr.finish(L, P.S, r);
    if constexpr (std::is_same_v<Rec, LastState>) {
        rec.p = r.p;
        rec.d = r.d;
    }
    return reference_end<kSoft>(P, L, r, M, kappa, soft, rec);
}

// A wave-uniform value, into scalar registers.
__device__ __forceinline__ double first_lane(double x) {
    const int lo = __builtin_amdgcn_readfirstlane(__double2loint(x));
    const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(x));
    return __hiloint2double(hi, lo);
}

// ---- deterministic block reductions -----------------------------------------------------------

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

template <class T>
__device__ __forceinline__ T block_sum(T v, T* lds) {
    v = wave_sum(v);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) lds[wave] = v;
    __syncthreads();
    T total = lds[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) total += lds[w];
    __syncthreads();
    return total;
}

// ---- RESIDUALS / MERIT ----------------------------------------------------------------------

// Mode 0: RESIDUALS (residual rows, penalty rows, OPD, status). Mode 1: MERIT partials per
// (variant, tuple): sum r^2 + sum p^2, failed and hard-failed counts. R: number type of the ray
// trace (double or df64); OPL, piston and residuals are formed in double.
__device__ __forceinline__ int64_t state_index(const mko_internal::RayStates& rs, int v, int c,
                                               int64_t row) {
    const int64_t slot = rs.slot ? rs.slot[v] : int64_t(rs.slot_offset) + v;
    return (int64_t(c) * rs.slots + slot) * rs.rays + row;
}

// kExt: also the surface extrema of the tuple's rays with status Ok, ext_partial[block][S][2]
// (largest height^2, smallest cos I); a wave that holds a ray with another status traces its
// valid rays a second time for them.
template <int kMode, bool kSoft, int kRpl, class R, bool kStates = false, bool kExt = false>
__global__ __launch_bounds__(kBlock) void trace_kernel(TraceParams P, double* residuals,
                                                       double* opd, uint8_t* status,
                                                       double* partial, int* pfailed,
                                                       int* phard,
                                                       mko_internal::RayStates states,
                                                       double* ext_partial) {
    __shared__ TraceTable<R> table;
    __shared__ SampleTable ST;
    __shared__ double red[kWaves];
    __shared__ int ired[kWaves];
    if (P.live && int(blockIdx.x) / P.T >= *P.live) return;
    const Tuple t = tuple_of(P, blockIdx.x);
    stage_samples(P, t, ST);
    table.stage(P, t);
    const typename TraceTable<R>::Ptr L = table.ptr();
    const size_t vf = size_t(t.v) * P.F + t.f;
    const double a = P.pupil_radius[t.v];
    double sin_t, cos_t;
    sincos(P.field_angle[vf], &sin_t, &cos_t);
    const V3<double> M{0.0, P.field_target[vf], working_distance(L, P.S)};
    const double kappa = P.ref_kind != MKO_REF_LAST_SURFACE ? P.reference_curvature[vf] : 0.0;

    // when the spoke count divides the workgroup, lane x keeps spoke x mod M in every ray slot i
    // and its ring advances by 256 / M per slot: the samples without a division per ray
    const bool lane_spoke = kBlock % t.M == 0 && t.M <= kTableSpokes;
    const int ring0 = int(threadIdx.x) / t.M, spoke0 = int(threadIdx.x) - ring0 * t.M;
    const int ring_step = kBlock / t.M;
    auto sample_slot = [&](int i, int k) {
        if (!lane_spoke) return sample_at(P, t, ST, k);
        const int ring = ring0 + i * ring_step;
        return Sample{ST.rho[ring], ST.sphi[spoke0], ST.cphi[spoke0], ST.weight[ring],
                      ST.rootw[ring]};
    };
    double opl[kRpl], pen[kRpl];
    uint8_t st[kRpl];
    double sw = 0.0, swo = 0.0;
    const int lane = threadIdx.x & 63;
    double eh = 0.0, ec = 1.0; // surface `lane`'s extrema over this wave's valid rays
#pragma unroll
    for (int i = 0; i < kRpl; ++i) {
        const int k = threadIdx.x + i * kBlock;
        st[i] = MKO_STATUS_UNSUPPORTED;
        opl[i] = 0.0;
        pen[i] = 0.0;
        if constexpr (kExt) {
            const bool have = k < t.n;
            Sample s{};
            Ray r0{};
            if (have) {
                s = sample_slot(i, k);
                r0 = source_ray(P, t, s, a, sin_t, cos_t, index_after(L, 0));
            }
            mkod::RayT<R> r = ray_as<R>(r0);
            Soft soft{0.0, MKO_STATUS_OK};
            double pend_h = 0.0, pend_c = 1.0;
            std::conditional_t<kStates, LastState, NoRecord> rec{};
            const uint8_t sti = trace_ray_ext<kSoft>(P, L, r, M, kappa, soft, have, lane,
                                                            pend_h, pend_c, false, rec);
            const uint64_t have_mask = __ballot(have);
            const uint64_t ok_mask = __ballot(have && sti == MKO_STATUS_OK);
            if (ok_mask == have_mask) {
                if (lane < P.S) {
                    eh = pend_h > eh ? pend_h : eh;
                    ec = pend_c < ec ? pend_c : ec;
                }
            } else {
                // some ray of the wave did not end with status Ok: its earlier surfaces must not
                // count, so the wave's valid rays are traced again and folded in directly
                mkod::RayT<R> rr = ray_as<R>(r0);
                Soft s2{0.0, MKO_STATUS_OK};
                NoRecord nr;
                trace_ray_ext<kSoft>(P, L, rr, M, kappa, s2, have && sti == MKO_STATUS_OK,
                                            lane, eh, ec, true, nr);
            }
            if (have) {
                st[i] = sti;
                if constexpr (kStates) {
                    const int64_t row = t.offset + k;
                    const bool okr = sti == MKO_STATUS_OK;
                    if (okr) {
                        states.data[state_index(states, t.v, 0, row)] = rec.p.x;
                        states.data[state_index(states, t.v, 1, row)] = rec.p.y;
                        states.data[state_index(states, t.v, 2, row)] = rec.p.z;
                        states.data[state_index(states, t.v, 3, row)] = rec.d.x;
                        states.data[state_index(states, t.v, 4, row)] = rec.d.y;
                        states.data[state_index(states, t.v, 5, row)] = rec.d.z;
                    }
                    states.data[state_index(states, t.v, 6, row)] =
                        okr ? mkod::to_double(r.opl) : __builtin_nan("");
                }
                opl[i] = mkod::in_piston(sti) ? mkod::to_double(r.opl) : 0.0;
                pen[i] = soft.penalty;
                if (mkod::in_piston(sti)) {
                    sw += s.weight;
                    swo += s.weight * opl[i];
                }
            }
            continue;
        }
        if (k < t.n) {
            const Sample s = sample_slot(i, k);
            mkod::RayT<R> r = ray_as<R>(source_ray(P, t, s, a, sin_t, cos_t, index_after(L, 0)));
            Soft soft{0.0, MKO_STATUS_OK};
            if constexpr (kStates) {
                LastState last;
                last.image_branch = 0;
                st[i] = trace_ray<kSoft>(P, L, r, M, kappa, soft, last);
                const int64_t row = t.offset + k;
                const bool okr = st[i] == MKO_STATUS_OK;
                if (okr) {
                    states.data[state_index(states, t.v, 0, row)] = last.p.x;
                    states.data[state_index(states, t.v, 1, row)] = last.p.y;
                    states.data[state_index(states, t.v, 2, row)] = last.p.z;
                    states.data[state_index(states, t.v, 3, row)] = last.d.x;
                    states.data[state_index(states, t.v, 4, row)] = last.d.y;
                    states.data[state_index(states, t.v, 5, row)] = last.d.z;
                }
                states.data[state_index(states, t.v, 6, row)] =
                    okr ? mkod::to_double(r.opl) : __builtin_nan("");
            } else {
                NoRecord nr;
                st[i] = trace_ray<kSoft>(P, L, r, M, kappa, soft, nr);
            }
            // a ray's OPL counts only with an in-piston status; selecting it here leaves the ray
            // dead on the surface loop's failure exits (no copies of it kept for them)
            opl[i] = mkod::in_piston(st[i]) ? mkod::to_double(r.opl) : 0.0;
            pen[i] = soft.penalty;
            if (mkod::in_piston(st[i])) {
                sw += s.weight;
                swo += s.weight * opl[i];
            }
        }
    }
    const double w_ok = block_sum(sw, red);
    const double sum = block_sum(swo, red);
    const bool valid = w_ok > 0.0;
    const double piston = valid ? sum / w_ok : 0.0;
    double r2 = 0.0, p2 = 0.0;
    int nfail = 0, nhard = 0;
#pragma unroll
    for (int i = 0; i < kRpl; ++i) {
        const int k = threadIdx.x + i * kBlock;
        if (k < t.n) {
            const Sample s = sample_slot(i, k);
            const bool ok = valid && mkod::in_piston(st[i]);
            const double e = ok ? opl[i] - piston : 0.0;
            const double r = t.scale * s.rootw * e;
            double pr = 0.0;
            if (kSoft) {
                const double fp = st[i] == MKO_STATUS_OK ? 0.0
                                  : mkod::is_soft(st[i]) ? pen[i]
                                                         : pen[i] + 1.0;
                pr = t.pscale * s.rootw * fp;
            }
            const int64_t row = t.offset + k;
            if (kMode == 0) {
                const size_t base = size_t(t.v) * P.stride;
                residuals[base + row] = r;
                if (kSoft) residuals[base + P.rays + row] = pr;
                if (opd) opd[size_t(t.v) * P.rays + row] = e;
                if (status) status[size_t(t.v) * P.rays + row] = st[i];
            } else {
                r2 += r * r;
                p2 += pr * pr;
                nfail += st[i] != MKO_STATUS_OK;
                nhard += !mkod::in_piston(st[i]);
            }
        }
    }
    if (kMode == 1) {
        const double tr2 = block_sum(r2, red);
        const double tp2 = kSoft ? block_sum(p2, red) : 0.0;
        const int tf = block_sum(nfail, ired);
        const int th = block_sum(nhard, ired);
        if (threadIdx.x == 0) {
            const size_t idx = size_t(t.v) * P.T + size_t(blockIdx.x - t.v * P.T);
            partial[idx] = kSoft ? tr2 + tp2 : tr2;
            pfailed[idx] = tf;
            phard[idx] = th;
        }
    }
    if constexpr (kExt) {
        __shared__ double ext_w[kWaves][MKO_MAX_SURFACES][2];
        const int wave = threadIdx.x >> 6;
        if (lane < P.S) {
            ext_w[wave][lane][0] = eh;
            ext_w[wave][lane][1] = ec;
        }
        __syncthreads();
        if (int(threadIdx.x) < P.S) {
            double h = ext_w[0][threadIdx.x][0], c = ext_w[0][threadIdx.x][1];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) {
                const double hw = ext_w[w][threadIdx.x][0], cw = ext_w[w][threadIdx.x][1];
                h = hw > h ? hw : h;
                c = cw < c ? cw : c;
            }
            double* out = ext_partial + (size_t(blockIdx.x) * P.S + threadIdx.x) * 2;
            out[0] = h;
            out[1] = c;
        }
    }
}

// ---- tuple packs: consecutive tuples of a variant share a workgroup -------------------------

// Step tables of the pack's tuples (tuple t0 + j at Ls + j (S + 1)); as stage_steps per tuple.
__device__ __forceinline__ void stage_steps_pack(const TraceParams& P, int v, int t0, int tpb,
                                                 Step* Ls) {
    const int n = tpb * (P.S + 1);
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
        const int j = e / (P.S + 1), s = e - j * (P.S + 1);
        const int tt = t0 + j;
        if (tt < P.T) Ls[e] = step_at(P, v, tt - (tt / P.L) * P.L, s);
    }
    __syncthreads();
}

// Sum over a pack segment of `seg` lanes (a power of two, 32 ... 256): for seg >= 64 the wave
// sums of the segment's waves added in wave order, for seg < 64 the xor butterfly over the
// segment's lanes (offsets seg / 2 ... 1). The same tree as block_sum of one tuple per workgroup,
// whose other lanes (and waves) hold zeros: the steps it has beyond the segment add exact zeros,
// so the sums are equal bit for bit.
template <class T>
__device__ __forceinline__ T seg_sum(T v, int seg, T* lds) {
    if (seg >= 64) {
        v = wave_sum(v);
        const int wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0) lds[wave] = v;
        __syncthreads();
        const int w0 = (int(threadIdx.x) / seg) * (seg / 64);
        T total = lds[w0];
        for (int w = 1; w < seg / 64; ++w) total += lds[w0 + w];
        __syncthreads();
        return total;
    }
    for (int off = seg / 2; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// RESIDUALS (kMode 0) / MERIT partials (kMode 1) of tuples of at most `seg` rays (seg 32, 64 or
// 128), 256 / seg consecutive tuples of one variant per workgroup (make_tuple_packs,
// include/mikroptim/cuda/tuple_packs.hpp:61, with a pack size fixed per launch): tuple t0 + j
// on lanes [j seg, (j + 1) seg), one ray per lane, its step table at Ls + j (S + 1). Every value is
// the one trace_kernel computes for the tuple alone (FP64 trace, no extrema).
template <int kMode, bool kSoft, bool kStates>
__global__ __launch_bounds__(kBlock) void trace_pack_kernel(TraceParams P, int seg,
                                                            double* residuals, double* opd,
                                                            uint8_t* status, double* partial,
                                                            int* pfailed, int* phard,
                                                            mko_internal::RayStates states) {
    extern __shared__ __align__(16) unsigned char pack_lds[];
    Step* Ls = reinterpret_cast<Step*>(pack_lds);
    __shared__ double red[kWaves];
    __shared__ int ired[kWaves];
    const int tpb = kBlock / seg;
    const int bpv = (P.T + tpb - 1) / tpb;
    const int v = int(blockIdx.x) / bpv;
    const int t0 = (int(blockIdx.x) - v * bpv) * tpb;
    if (P.live && v >= *P.live) return;
    stage_steps_pack(P, v, t0, tpb, Ls);
    const int j = int(threadIdx.x) / seg, k = int(threadIdx.x) - j * seg;
    const int tt = t0 + j;
    const bool in_pack = tt < P.T;
    const Step* L = Ls + j * (P.S + 1);
    const Tuple t = tuple_of(P, v * P.T + (in_pack ? tt : 0));
    const size_t vf = size_t(t.v) * P.F + t.f;
    const double a = P.pupil_radius[t.v];
    double sin_t, cos_t;
    sincos(P.field_angle[vf], &sin_t, &cos_t);
    const V3<double> M{0.0, P.field_target[vf], L[P.S].t};
    const double kappa = P.ref_kind != MKO_REF_LAST_SURFACE ? P.reference_curvature[vf] : 0.0;
    const bool have = in_pack && k < t.n;
    double opl = 0.0, pen = 0.0, sw = 0.0, swo = 0.0;
    uint8_t st = MKO_STATUS_UNSUPPORTED;
    Sample smp{};
    if (have) {
        smp = sample_of(P, t, k);
        mkod::RayT<double> r = source_ray(P, t, smp, a, sin_t, cos_t, L[0].n);
        Soft soft{0.0, MKO_STATUS_OK};
        if constexpr (kStates) {
            LastState last;
            last.image_branch = 0;
            st = trace_ray<kSoft>(P, L, r, M, kappa, soft, last);
            const int64_t row = t.offset + k;
            const bool okr = st == MKO_STATUS_OK;
            if (okr) {
                states.data[state_index(states, t.v, 0, row)] = last.p.x;
                states.data[state_index(states, t.v, 1, row)] = last.p.y;
                states.data[state_index(states, t.v, 2, row)] = last.p.z;
                states.data[state_index(states, t.v, 3, row)] = last.d.x;
                states.data[state_index(states, t.v, 4, row)] = last.d.y;
                states.data[state_index(states, t.v, 5, row)] = last.d.z;
            }
            states.data[state_index(states, t.v, 6, row)] = okr ? r.opl : __builtin_nan("");
        } else {
            NoRecord nr;
            st = trace_ray<kSoft>(P, L, r, M, kappa, soft, nr);
        }
        opl = r.opl;
        pen = soft.penalty;
        if (mkod::in_piston(st)) {
            sw += smp.weight;
            swo += smp.weight * opl;
        }
    }
    const double w_ok = seg_sum(sw, seg, red);
    const double sum = seg_sum(swo, seg, red);
    const bool valid = w_ok > 0.0;
    const double piston = valid ? sum / w_ok : 0.0;
    double r2 = 0.0, p2 = 0.0;
    int nfail = 0, nhard = 0;
    if (have) {
        const bool ok = valid && mkod::in_piston(st);
        const double e = ok ? opl - piston : 0.0;
        const double r = t.scale * smp.rootw * e;
        double pr = 0.0;
        if (kSoft) {
            const double fp = st == MKO_STATUS_OK ? 0.0 : mkod::is_soft(st) ? pen : pen + 1.0;
            pr = t.pscale * smp.rootw * fp;
        }
        const int64_t row = t.offset + k;
        if (kMode == 0) {
            const size_t base = size_t(t.v) * P.stride;
            residuals[base + row] = r;
            if (kSoft) residuals[base + P.rays + row] = pr;
            if (opd) opd[size_t(t.v) * P.rays + row] = e;
            if (status) status[size_t(t.v) * P.rays + row] = st;
        } else {
            r2 = r * r;
            p2 = pr * pr;
            nfail = st != MKO_STATUS_OK;
            nhard = !mkod::in_piston(st);
        }
    }
    if (kMode == 1) {
        const double tr2 = seg_sum(r2, seg, red);
        const double tp2 = kSoft ? seg_sum(p2, seg, red) : 0.0;
        const int tf = seg_sum(nfail, seg, ired);
        const int th = seg_sum(nhard, seg, ired);
        if (k == 0 && in_pack) {
            const size_t idx = size_t(v) * P.T + size_t(tt);
            partial[idx] = kSoft ? tr2 + tp2 : tr2;
            pfailed[idx] = tf;
            phard[idx] = th;
        }
    }
}

// Extrema of every variant from the tuple partials: out[v][s] = {sqrt(max height^2), min cos I}
// over the variant's tuples (extrema_finalize_kernel of the reference, wavefront_block.hpp:414).
__global__ void extrema_finalize_kernel(int V, int T, int S, const double* partial, double* out) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= int64_t(V) * S) return;
    const int64_t v = i / S, s = i - v * S;
    double h = 0.0, c = 1.0;
    for (int t = 0; t < T; ++t) {
        const double* p = partial + ((v * T + t) * S + s) * 2;
        h = p[0] > h ? p[0] : h;
        c = p[1] < c ? p[1] : c;
    }
    out[i * 2] = __dsqrt_rn(h);
    out[i * 2 + 1] = c;
}

// Check of the candidate rays after the differences' traces, one thread per run: on every height
// surface the candidates' largest height over the run's per_run points (ex [runs * per_run][S][2])
// moved by at most D from the run's (ex0); the other rays lie below (1 - delta) of the run's
// largest height at its point and would have to move by more than K D to reach the candidates'
// smallest; likewise for the smallest cos I on the incidence surfaces (the others above
// cmin + delta (1 - cmin)). flag[r] = 1 where that margin is missing or the list overflowed.
__global__ void extrema_check_kernel(int runs, int per_run, int S, uint64_t hmask, uint64_t cmask,
                                     double delta, const double* ex, const double* ex0,
                                     const int* others, const int* overflow, double K,
                                     int* flag) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= runs) return;
    int bad = overflow[r];
    if (!bad && others[r] > 0) {
        for (int s = 0; s < S; ++s) {
            if (!(((hmask | cmask) >> s) & 1ull)) continue;
            const double h0 = ex0[(size_t(r) * S + s) * 2], c0 = ex0[(size_t(r) * S + s) * 2 + 1];
            double dh = 0.0, dc = 0.0, hmin = h0, cmax = c0;
            for (int j = 0; j < per_run; ++j) {
                const double* e = ex + ((size_t(r) * per_run + j) * S + s) * 2;
                dh = fmax(dh, fabs(e[0] - h0));
                dc = fmax(dc, fabs(e[1] - c0));
                hmin = fmin(hmin, e[0]);
                cmax = fmax(cmax, e[1]);
            }
            if (((hmask >> s) & 1ull) && !((1.0 - delta) * h0 + K * dh < hmin)) bad = 1;
            if (((cmask >> s) & 1ull) && !(c0 + delta * (1.0 - c0) - K * dc > cmax)) bad = 1;
        }
    }
    flag[r] = bad;
}

// ---- candidate rays of the constraint rows' central differences ----------------------------

// Per-ray candidates at the runs' points: one 256-lane workgroup per (run, tuple) of the points'
// batch (variant = run), each ray traced as trace_ray_ext traces it. A ray is a candidate where it
// does not end with status Ok (at a difference point it may), or where on a height surface
// (hmask) its height reaches (1 - delta) of the run's largest, or on an incidence surface (cmask)
// its cos I lies within delta (1 - cos) of the run's smallest (ex0 [runs][S][2]). flags [runs *
// rays] (1 = candidate), tcount [runs][T] candidates per tuple, others [runs] (atomic count of the
// non-candidates).
template <bool kSoft>
__global__ __launch_bounds__(kBlock) void ray_candidates_kernel(TraceParams P, uint64_t hmask,
                                                               uint64_t cmask, double delta,
                                                               const double* ex0, uint8_t* flags,
                                                               int* tcount, int* others) {
    __shared__ Step L[MKO_MAX_SURFACES + 1];
    __shared__ SampleTable ST;
    __shared__ double thr[2][MKO_MAX_SURFACES];
    __shared__ int red[kWaves];
    const Tuple t = tuple_of(P, blockIdx.x);
    if (int(threadIdx.x) < P.S) {
        const double hmax = ex0[(size_t(t.v) * P.S + threadIdx.x) * 2];
        const double cmin = ex0[(size_t(t.v) * P.S + threadIdx.x) * 2 + 1];
        thr[0][threadIdx.x] = (1.0 - delta) * hmax;
        thr[1][threadIdx.x] = cmin + delta * (1.0 - cmin);
    }
    stage_samples(P, t, ST);
    stage_steps(P, t.v, t.l, L);
    __syncthreads();
    const size_t vf = size_t(t.v) * P.F + t.f;
    const double a = P.pupil_radius[t.v];
    double sin_t, cos_t;
    sincos(P.field_angle[vf], &sin_t, &cos_t);
    const V3<double> M{0.0, P.field_target[vf], L[P.S].t};
    const double kappa = P.ref_kind != MKO_REF_LAST_SURFACE ? P.reference_curvature[vf] : 0.0;
    const uint64_t mask = hmask | cmask;
    int cands = 0, rest = 0;
    for (int k = threadIdx.x; k < t.n; k += kBlock) {
        const Sample smp = sample_at(P, t, ST, k);
        mkod::RayT<double> r = ray_as<double>(source_ray(P, t, smp, a, sin_t, cos_t, L[0].n));
        Soft soft{0.0, MKO_STATUS_OK};
        bool cand = false;
        auto mark = [&](int sf, double x, double y, double ci) {
            if (!((mask >> sf) & 1ull)) return;
            if (((hmask >> sf) & 1ull) && __dsqrt_rn(height_sq(x, y)) >= thr[0][sf]) cand = true;
            if (((cmask >> sf) & 1ull) && ci <= thr[1][sf]) cand = true;
        };
        mark(0, r.p.x, r.p.y, r.d.z);
        uint8_t st = MKO_STATUS_OK;
        Tracer<double> tr;
        tr.begin(L, r);
        for (int sf = 1; sf < P.S; ++sf) {
            uint8_t branch = 0;
            const uint8_t sst = tr.step<kSoft, true>(L, sf, r, soft, branch);
            if (sst != MKO_STATUS_OK) {
                st = sst;
                break;
            }
            mark(sf, r.p.x, r.p.y, tr.cos_incidence(L, sf, r));
        }
        if (st == MKO_STATUS_OK) {
            NoRecord nr;
            tr.finish(L, P.S, r);
            st = reference_end<kSoft>(P, static_cast<const Step*>(L), r, M, kappa, soft, nr);
        }
        if (st != MKO_STATUS_OK) cand = true;
        flags[size_t(t.v) * P.rays + t.offset + k] = cand ? 1 : 0;
        cands += cand;
        rest += !cand;
    }
    const int tc = block_sum(cands, red);
    const int tr = block_sum(rest, red);
    if (threadIdx.x == 0) {
        tcount[blockIdx.x] = tc;
        if (tr) atomicAdd(others + t.v, tr);
    }
}

// Ordered candidate list of each run (one 1024-thread workgroup per run): the rows with a flag in
// ascending order (so grouped by tuple), list [runs][cap]; tstart [runs][T + 1] the tuples'
// first entries; overflow[run] = 1 where more than cap rays are candidates.
__global__ __launch_bounds__(1024) void candidate_list_kernel(int T, int64_t rays, int cap,
                                                              const uint8_t* flags,
                                                              const int* tcount, int* tstart,
                                                              int* list, int* overflow) {
    __shared__ int32_t wave_total[16];
    __shared__ int32_t base_s;
    const int r = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) {
        int acc = 0;
        for (int t = 0; t < T; ++t) {
            tstart[size_t(r) * (T + 1) + t] = acc;
            acc += tcount[size_t(r) * T + t];
        }
        tstart[size_t(r) * (T + 1) + T] = acc;
        overflow[r] = acc > cap ? 1 : 0;
        base_s = 0;
    }
    __syncthreads();
    if (tstart[size_t(r) * (T + 1) + T] > cap) return;
    const uint8_t* f = flags + size_t(r) * rays;
    for (int64_t start = 0; start < rays; start += 1024) {
        const int64_t e = start + tid;
        const bool pick = e < rays && f[e] != 0;
        const uint64_t m = __ballot(pick);
        const int before = __popcll(m & ((uint64_t(1) << lane) - 1));
        if (lane == 0) wave_total[wave] = __popcll(m);
        __syncthreads();
        int offset = base_s;
        for (int w = 0; w < wave; ++w) offset += wave_total[w];
        if (pick) list[size_t(r) * cap + offset + before] = int(e);
        __syncthreads();
        if (tid == 0) {
            int sum = 0;
            for (int w = 0; w < 16; ++w) sum += wave_total[w];
            base_s += sum;
        }
        __syncthreads();
    }
}

// The extrema [V][S][2] of the differences' batch over the candidate rays of each variant's run
// (run = v / per_run): one wavefront per variant, the tuples holding candidates in order, their
// rays traced and reduced exactly as trace_kernel's extrema trace (trace_ray_ext; a wave with a
// ray that does not end Ok traces its valid rays again), then sqrt of the largest height^2 and
// the smallest cos I (extrema_finalize_kernel). Equal to the extrema over every ray wherever the
// extremal ray of each surface is a candidate.
template <bool kSoft>
__global__ __launch_bounds__(64) void candidate_extrema_kernel(TraceParams P, int per_run,
                                                               int cap, const int* tstart,
                                                               const int* list, double* ext) {
    __shared__ Step steps[MKO_MAX_SURFACES + 1];
    const Step* L = steps;
    const int v = blockIdx.x;
    const int run = v / per_run;
    const int lane = threadIdx.x;
    const int* ts = tstart + size_t(run) * (P.T + 1);
    const int* lst = list + size_t(run) * cap;
    double eh = 0.0, ec = 1.0;
    // an overflowed list was not written: neutral extrema (the check sends the chunk to the
    // whole trace)
    const int ntuples = ts[P.T] > cap ? 0 : P.T;
    for (int tt = 0; tt < ntuples; ++tt) {
        const int lo = ts[tt], hi = ts[tt + 1];
        if (lo == hi) continue; // uniform across the wave
        const Tuple t = tuple_of(P, v * P.T + tt);
        stage_steps(P, t.v, t.l, steps);
        __syncthreads();
        const size_t vf = size_t(t.v) * P.F + t.f;
        const double a = P.pupil_radius[t.v];
        double sin_t, cos_t;
        sincos(P.field_angle[vf], &sin_t, &cos_t);
        const V3<double> M{0.0, P.field_target[vf], L[P.S].t};
        const double kappa = P.ref_kind != MKO_REF_LAST_SURFACE ? P.reference_curvature[vf] : 0.0;
        for (int base = lo; base < hi; base += 64) {
            const int e = base + lane;
            const bool have = e < hi;
            Sample smp{};
            Ray r0{};
            if (have) {
                const int k = int(int64_t(lst[e]) - t.offset);
                smp = sample_of(P, t, k);
                r0 = source_ray(P, t, smp, a, sin_t, cos_t, L[0].n);
            }
            mkod::RayT<double> r = ray_as<double>(r0);
            Soft soft{0.0, MKO_STATUS_OK};
            double pend_h = 0.0, pend_c = 1.0;
            NoRecord rec;
            const uint8_t sti = trace_ray_ext<kSoft>(
                P, L, r, M, kappa, soft, have, lane, pend_h, pend_c, false, rec);
            const uint64_t have_mask = __ballot(have);
            const uint64_t ok_mask = __ballot(have && sti == MKO_STATUS_OK);
            if (ok_mask == have_mask) {
                if (lane < P.S) {
                    eh = pend_h > eh ? pend_h : eh;
                    ec = pend_c < ec ? pend_c : ec;
                }
            } else {
                mkod::RayT<double> rr = ray_as<double>(r0);
                Soft s2{0.0, MKO_STATUS_OK};
                NoRecord nr;
                trace_ray_ext<kSoft>(P, L, rr, M, kappa, s2,
                                                     have && sti == MKO_STATUS_OK, lane, eh, ec,
                                                     true, nr);
            }
        }
        __syncthreads(); // L is restaged for the next tuple
    }
    if (lane < P.S) {
        ext[(size_t(v) * P.S + lane) * 2] = __dsqrt_rn(eh);
        ext[(size_t(v) * P.S + lane) * 2 + 1] = ec;
    }
}

// Constraint rows of every variant (one thread per variant), rows[v * stride + offset + k] for
// the `count` items in row order; extrema [V][S][2] for the items that need them.
__global__ void constraint_rows_kernel(int V, int S, int F, const double* curvature,
                                       const double* thickness, const double* paraxial_index,
                                       const double* pupil_radius, const double* field_angle,
                                       const double* field_target, uint64_t sphere_mask,
                                       const mko_constraint* items, int count, int need_paraxial,
                                       const double* extrema, double* rows, int64_t stride,
                                       int64_t offset, const double* buchdahl,
                                       const double* glass_hull) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const mkoc::VariantRows vr{curvature + size_t(v) * S,
                               thickness + size_t(v) * S,
                               paraxial_index ? paraxial_index + size_t(v) * S : nullptr,
                               sphere_mask,
                               pupil_radius[v],
                               S,
                               field_angle + size_t(v) * F,
                               field_target + size_t(v) * F,
                               F,
                               buchdahl ? buchdahl + size_t(v) * S * 4 : nullptr,
                               glass_hull};
    mkoc::Paraxial p{1.0, 0.0, 0.0, 0.0, false, false, 0.0, 0.0, 0.0};
    if (need_paraxial) p = mkoc::paraxial(vr.c, vr.t, vr.n, S);
    const double* ext = extrema ? extrema + size_t(v) * S * 2 : nullptr;
    double* out = rows + size_t(v) * stride + offset;
    for (int k = 0; k < count; ++k) out[k] = mkoc::row(items[k], vr, p, ext);
}

// Normal equations of the constraint rows added to a run's A [P][P] and g [P] (the fused
// mixed-precision path forms no J): A(p, q) += sum_e Je(p, e) Je(q, e), g(p) += sum_e Je(p, e)
// re(e), one workgroup per run, Je [runs][P][E], re [runs][E].
__global__ void extra_normal_kernel(int P, int E, const double* Je, const double* re, double* a,
                                    double* g) {
    const int run = blockIdx.x;
    const double* J = Je + size_t(run) * P * E;
    const double* r = re + size_t(run) * E;
    for (int i = threadIdx.x; i < P * (P + 1); i += blockDim.x) {
        const int p = i / (P + 1), q = i - p * (P + 1);
        const double* u = J + size_t(p) * E;
        const double* w = q < P ? J + size_t(q) * E : r;
        double acc = 0.0;
        for (int e = 0; e < E; ++e) acc = fma(u[e], w[e], acc);
        if (q < P) a[(size_t(run) * P + p) * P + q] += acc;
        else g[size_t(run) * P + p] += acc;
    }
}

// Sums of squares of the constraint rows per variant (extra_merit_values,
// src/optim/levenberg_marquardt.cpp:659; trace_extra_merit, src/optim/trace_extra_residuals.cpp:96):
// e[v] = (extra ? extra[v] + : ) sum_{k < E} r_k^2, t[v] = sum_{E <= k < E + Et} r_k^2, ascending.
__global__ void rows_merit_kernel(int V, const double* rows, int64_t stride, int64_t offset, int E,
                                  int Et, const double* extra, double* e_sum, double* t_sum) {
#pragma clang fp contract(off)
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const double* r = rows + size_t(v) * stride + offset;
    double e = 0.0;
    for (int k = 0; k < E; ++k) e = e + r[k] * r[k];
    if (e_sum) e_sum[v] = extra ? extra[v] + e : e;
    double t = 0.0;
    for (int k = E; k < E + Et; ++k) t = t + r[k] * r[k];
    if (t_sum) t_sum[v] = t;
}

// merit[v] = sum over tuples in (f, l) order + extra[v] (merit_finalize_kernel, merit.cu:207). A
// wave per variant, 4 to a workgroup: the partials of 64 tuples in one load, added in tuple order
// from the lanes' registers (a thread per variant waited for each tuple's three loads: 256 variants
// of 35 tuples 21 -> 5 us).
__global__ __launch_bounds__(256) void merit_finalize_kernel(
    int V, int T, const double* partial, const int* pfailed, const int* phard, const double* extra,
    const double* traced, double* merit, int64_t* failed, int64_t* hard, const int32_t* live) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const int v = int(blockIdx.x) * 4 + int(threadIdx.x >> 6);
    if (v >= V || (live && v >= *live)) return;
    double s = 0.0;
    int64_t f = 0, h = 0;
    for (int t0 = 0; t0 < T; t0 += 64) {
        const int t = t0 + lane;
        const size_t at = size_t(v) * T + t;
        const double x = t < T ? partial[at] : 0.0;
        f += t < T ? pfailed[at] : 0;
        h += t < T ? phard[at] : 0;
        const int n = min(64, T - t0);
        const int lo = __double2loint(x), hi = __double2hiint(x);
        for (int i = 0; i < n; ++i)
            s += __hiloint2double(__builtin_amdgcn_readlane(hi, i),
                                  __builtin_amdgcn_readlane(lo, i));
    }
    f = wave_sum(f);
    h = wave_sum(h);
    if (lane != 0) return;
    // (ray merit + sum e^2) + sum t^2 (CpuLmBackend::merit, levenberg_marquardt.cpp:866-888)
    double m = extra ? s + extra[v] : s;
    if (traced) m = m + traced[v];
    merit[v] = m;
    failed[v] = f;
    hard[v] = h;
}

// ---- FP32 prefilter (prefilter_kernel, src/cuda/prefilter.cu:87; per ray prefilter_ray,
// include/mikroptim/merit/prefilter_ray.hpp:171-249) ---------------------------------------------
// The only float path: its values select multistart variants and never enter a merit, residual
// or Jacobian. Each ray is traced in float (hard failure) and carries its boundary margin: the
// smallest distance of the tracer's checks from their failure boundary, as a cosine (d_z before a
// transfer, cos I = sqrt(D) at the sphere, cos I' = sqrt(k) after refraction, the reference
// sphere's discriminant and denominator); for a failed ray the size of the violated check.

// Surface table of a (variant, wavelength) in LDS: row s >= 1 the step to surface s, row 0 the
// image side.
struct PfStep {
    float c, t, n, mu; // effective curvature, thickness and index before the surface, n / n'
};
static_assert(sizeof(PfStep) == mko_internal::kPrefilterStepBytes);

// Quotient and root in 4 and 6 instructions (the correctly rounded ones of the compiler take
// about 10 and 15 and were half of the trace): the hardware's estimate and one step on the residual,
// within 1 ulp. The root of a number below the smallest normal one is that one's.
__device__ __forceinline__ float pf_div(float a, float b) {
    const float y = __builtin_amdgcn_rcpf(b);
    const float q = a * y;
    return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}
__device__ __forceinline__ float pf_sqrt(float x) {
    const float v = x < 1.17549435e-38f ? 1.17549435e-38f : x; // NaN stays
    const float y = __builtin_amdgcn_rsqf(v);
    const float r = v * y;
    return __builtin_fmaf(__builtin_fmaf(-r, r, v), 0.5f * y, r);
}

// NaN in either sticks: no margin compares above eta then (uncertain).
__device__ __forceinline__ float pf_min_margin(float acc, float x) {
    return __builtin_elementwise_minimum(acc, x);
}
__device__ __forceinline__ float pf_fail_linear(float x) { return -x > 0.0f ? -x : 0.0f; }
__device__ __forceinline__ float pf_fail_root(float q) {
    return -q > 0.0f ? __builtin_sqrtf(-q) : 0.0f;
}

struct PfRay {
    uint8_t status;
    float opl, margin;
};

__device__ __forceinline__ PfRay pf_trace(const PfStep* L, int S, V3<float> p, V3<float> d,
                                          float opl, V3<float> M, float n_image, int kind,
                                          float kappa) {
    using mkod::cross;
    using mkod::dot;
    PfRay out{MKO_STATUS_OK, 0.0f, 0.0f};
    float margin = 1.0f;
    for (int s = 1; s < S; ++s) {
        const PfStep e = L[s];
        if (!(d.z > 0.0f)) {
            out.status = MKO_STATUS_BACKWARD;
            out.margin = pf_fail_linear(d.z);
            return out;
        }
        const float dz = d.z;
        p.z -= e.t;
        const float s0 = pf_div(-p.z, dz);
        p.x += s0 * d.x;
        p.y += s0 * d.y;
        p.z = 0.0f;
        const float H = e.c * (p.x * p.x + p.y * p.y);
        const float B = dz - e.c * (p.x * d.x + p.y * d.y);
        const float D = B * B - e.c * H;
        const float denom = D < 0.0f ? 0.0f : B + pf_sqrt(D);
        if (D < 0.0f || !(denom > 0.0f)) {
            const float a = pf_fail_root(D), b = pf_fail_linear(B);
            out.status = MKO_STATUS_MISSED;
            out.margin = a > b ? a : b;
            return out;
        }
        const float sh = pf_div(H, denom);
        p = p + sh * d;
        opl += e.n * (s0 + sh);
        const V3<float> N{-e.c * p.x, -e.c * p.y, 1.0f - e.c * p.z};
        const float cosI = dot(d, N);
        const float k = 1.0f - e.mu * e.mu * (1.0f - cosI * cosI);
        if (k < 0.0f) {
            out.status = MKO_STATUS_TIR;
            out.margin = pf_fail_root(k);
            return out;
        }
        d = e.mu * d + (pf_sqrt(k) - e.mu * cosI) * N;
        margin = pf_min_margin(pf_min_margin(margin, dz), cosI);
        margin = pf_min_margin(margin, dot(d, N));
    }
    if (!(d.z > 0.0f)) {
        out.status = MKO_STATUS_BACKWARD;
        out.margin = pf_fail_linear(d.z);
        return out;
    }
    margin = pf_min_margin(margin, d.z);
    if (kind != MKO_REF_LAST_SURFACE) {
        const V3<float> q = p - M;
        const V3<float> ci = cross(q, d);
        const float t = -dot(ci, ci);
        const float disc = 1.0f + kappa * kappa * t;
        const float b = -dot(q, d);
        float step = 0.0f;
        const bool ok = disc >= 0.0f;
        if (ok) step = b - kappa * t / (__builtin_sqrtf(disc) + 1.0f);
        if (!ok || (!(step >= 0.0f) && !(step < 0.0f))) {
            out.status = MKO_STATUS_MISSED;
            out.margin = disc < 0.0f ? pf_fail_root(disc) : 0.0f;
            return out;
        }
        out.opl = opl + n_image * step;
        out.margin = pf_min_margin(margin, __builtin_sqrtf(disc));
        return out;
    }
    const float r2 = dot(M, M);
    const float inv_r = r2 > 0.0f ? 1.0f / __builtin_sqrtf(r2) : 1.0f;
    const V3<float> q = p - M;
    const float bq = -dot(q, d);
    const float g = dot(p, p - 2.0f * M);
    const float disc = bq * bq - g;
    const float sigma = M.z >= 0.0f ? 1.0f : -1.0f;
    const float root = disc > 0.0f ? __builtin_sqrtf(disc) : 0.0f;
    const float den = sigma * (bq + sigma * root) * inv_r;
    bool ok = !(disc < 0.0f);
    float s_ref = 0.0f;
    if (ok) {
        const float rt = __builtin_sqrtf(disc);
        const bool real_image = M.z >= 0.0f;
        const float dn = real_image ? bq + rt : bq - rt;
        ok = real_image ? dn > 0.0f : dn < 0.0f;
        if (ok) s_ref = g / dn;
    }
    if (!ok) {
        const float a = pf_fail_root(disc * inv_r * inv_r);
        const float c = disc >= 0.0f ? pf_fail_linear(den) : 0.0f;
        out.status = MKO_STATUS_MISSED;
        out.margin = a > c ? a : c;
        return out;
    }
    margin = pf_min_margin(margin, root * inv_r);
    margin = pf_min_margin(margin, den);
    out.opl = opl + n_image * s_ref;
    out.margin = margin;
    return out;
}

__device__ __forceinline__ float block_max_f(float v, float* lds) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) lds[wave] = v;
    __syncthreads();
    float m = lds[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) m = lds[w] > m ? lds[w] : m;
    __syncthreads();
    return m;
}

// OPL relative to the axial optical length (prefilter_opl_offset), classes 0 certain valid / 1
// certain failed / 2, 3 uncertain (margin <= eta), the piston over the certain-valid rays and the
// tuple's sum of squared residuals; partials per tuple: merit (as double), largest optical length,
// counts [3] (certain failed, uncertain valid, uncertain failed).
// A multistart's tuples are small (6 to some hundred rays of a few surfaces), so what bounds it is
// the instruction issue, of which a workgroup per tuple spent two thirds on idle waves, on the
// tuple's weights and on every ray's sine and cosine. A workgroup takes one (field, wavelength) of
// 256 / Q variants, Q lanes per variant: the spokes' and rings' samples and the weight are formed
// once for all and the surface tables sit side by side (an odd stride spreads them over the banks).
// The rays' path lengths and classes wait in LDS for the sums, which q <= Q lanes of the variant
// form, without a barrier where Q = q (kWide: q = 256, sums over the workgroup). q depends on the
// tuple's size alone, so the sums' order, hence their bits, are the same in every batch; Q is
// larger where the batch is too small for the chip (prefilter_stats). 20000 variants of 9 tuples
// of up to 72 rays and 3 surfaces: 637 -> 113 us.
template <bool kWide>
__global__ __launch_bounds__(kBlock) void prefilter_kernel(TraceParams P, int Q, int q, float eta,
                                                           double* pmerit, float* plength,
                                                           int* pcounts) {
    extern __shared__ __align__(16) unsigned char pf_lds[];
    __shared__ float rho_l[MKO_MAX_RINGS], w_l[MKO_MAX_RINGS], scale_l;
    __shared__ float fred[kWaves];
    __shared__ int ired[kWaves];
    const int G = kBlock / Q, pitch = P.S | 1;
    const int group = int(blockIdx.x) / P.T, tt = int(blockIdx.x) - group * P.T;
    const int v0 = group * G, f = tt / P.L, l = tt - f * P.L;
    const int tid = threadIdx.x;
    const uint8_t mode = P.pupil_mode[f];
    const int M = mode == MKO_PUPIL_AXIS ? 1 : P.spokes, n = P.rings * M;
    PfStep* steps = reinterpret_cast<PfStep*>(pf_lds);        // [G][pitch]
    float2* spoke = reinterpret_cast<float2*>(steps + G * pitch); // [M]
    float* opl_l = reinterpret_cast<float*>(spoke + M);           // [G][rays]
    const int rays = mko_internal::prefilter_slots(n, q);
    uint8_t* cls_l = reinterpret_cast<uint8_t*>(opl_l + G * rays); // [G][rays]
    for (int e = tid; e < G * P.S; e += kBlock) {
        const int g = e / P.S, s = e - g * P.S;
        if (v0 + g >= P.V) break;
        const size_t vs = size_t(v0 + g) * P.S + s;
        PfStep k{};
        const float na = float(P.index[vs * P.L + l]);
        if (s > 0) {
            k.c = ((P.sphere_mask >> s) & 1ull) ? float(P.curvature[vs]) : 0.0f;
            k.t = float(P.thickness[vs - 1]);
            k.n = float(P.index[(vs - 1) * P.L + l]);
            k.mu = k.n / na;
        } else {
            const size_t last = vs + P.S - 1;
            k.t = float(P.thickness[last]);
            k.n = float(P.index[last * P.L + l]);
        }
        steps[g * pitch + s] = k;
    }
    const float pi = float(kPi);
    for (int j = tid; j < M; j += kBlock) {
        const float phi = mode == MKO_PUPIL_HALF   ? float(2 * j + 1) * pi / float(2 * M)
                          : mode == MKO_PUPIL_FULL ? float(2 * j + 1) * pi / float(M)
                                                   : 0.0f;
        spoke[j] = make_float2(sinf(phi), cosf(phi));
    }
    if (tid < P.rings) {
        rho_l[tid] = __builtin_sqrtf(float(P.gl_u[tid]));
        w_l[tid] = float(P.gl_w[tid]) / float(M);
    }
    if (tid >= kBlock - 64) { // one wave
        const Tuple t = tuple_of(P, tt);
        if (tid == kBlock - 1) scale_l = float(t.scale);
    }
    __syncthreads();
    const int mine = tid / Q, lane = tid & (Q - 1);
    const bool in = v0 + mine < P.V;
    const int v = in ? v0 + mine : P.V - 1;
    const PfStep* L = steps + (v - v0) * pitch;
    opl_l += mine * rays;
    cls_l += mine * rays;
    float offset = 0.0f;
    for (int s = 1; s < P.S; ++s) offset += L[s].n * L[s].t;
    const size_t vf = size_t(v) * P.F + f;
    const float a = float(P.pupil_radius[v]);
    const float th = float(P.field_angle[vf]);
    const float sth = sinf(th), cth = cosf(th);
    const V3<float> center{0.0f, float(P.field_target[vf]), L[0].t};
    const float n_image = L[0].n;
    const float kappa = P.ref_kind != MKO_REF_LAST_SURFACE ? float(P.reference_curvature[vf]) : 0.0f;
    // ray k = ri M + j of the lane: lane, lane + stride, ...
    int ri, j, step_r, step_j;
    const auto first_ray = [&](int stride) {
        step_r = stride / M;
        step_j = stride - step_r * M;
        ri = lane / M;
        j = lane - ri * M;
    };
    const auto next_ray = [&] {
        ri += step_r;
        j += step_j;
        if (j >= M) {
            j -= M;
            ++ri;
        }
    };
    first_ray(Q);
    for (int k = lane; in && k < n; k += Q, next_ray()) {
        const float rho = rho_l[ri];
        const float sp = spoke[j].x, cp = spoke[j].y;
        V3<float> p, d;
        float o;
        if (P.source == MKO_SOURCE_POINT) {
            const float sin_max = float(P.src_na) / L[1].n;
            const float sr = sin_max * rho;
            p = V3<float>{float(P.src_pt[0]), float(P.src_pt[1]), float(P.src_pt[2])};
            d = V3<float>{sr * sp, sr * cp, __builtin_sqrtf((1.0f - sr) * (1.0f + sr))};
            o = 0.0f;
        } else {
            const float r = a * rho;
            p = V3<float>{r * sp, r * cp, 0.0f};
            d = V3<float>{0.0f, sth, cth};
            o = mkod::dot(p, d);
        }
        const PfRay rr = pf_trace(L, P.S, p, d, o - offset, center, n_image, P.ref_kind, kappa);
        const bool ok = rr.status == MKO_STATUS_OK;
        const bool certain = rr.margin > eta;
        opl_l[k] = rr.opl;
        cls_l[k] = uint8_t(ok ? (certain ? 0 : 2) : (certain ? 1 : 3));
    }
    if (Q != q) __syncthreads();
    const bool sums = in && lane < q;
    float wok = 0.0f, wopl = 0.0f, optical = 0.0f;
    int fail_unsure = 0, nuf = 0; // certain failed + 2^16 uncertain valid, uncertain failed
    first_ray(q);
    for (int k = lane; sums && k < n; k += q, next_ray()) {
        const float opl = opl_l[k];
        const int c = cls_l[k];
        if (c == 0) {
            const float w = w_l[ri];
            wok += w;
            wopl += w * opl;
            const float len = fabsf(offset) + fabsf(opl);
            optical = len > optical ? len : optical;
        }
        fail_unsure += c == 1 ? 1 : c == 2 ? 1 << 16 : 0;
        nuf += c == 3;
    }
    const auto sum = [&](auto x, auto* lds) {
        if constexpr (kWide) return block_sum(x, lds);
        for (int off = q >> 1; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
        return x;
    };
    const float w_ok = sum(wok, fred);
    const float sum_o = sum(wopl, fred);
    const bool valid = w_ok > 0.0f;
    const float piston = valid ? sum_o / w_ok : 0.0f;
    const float scale = scale_l;
    float r2 = 0.0f;
    first_ray(q);
    for (int k = lane; sums && valid && k < n; k += q, next_ray()) {
        const float e = cls_l[k] == 0 ? opl_l[k] - piston : 0.0f;
        const float r = scale * __builtin_sqrtf(w_l[ri]) * e;
        r2 += r * r;
    }
    const float tr2 = sum(r2, fred);
    float tl = optical;
    if constexpr (kWide) tl = block_max_f(optical, fred);
    else
        for (int off = q >> 1; off >= 1; off >>= 1) {
            const float o = __shfl_xor(tl, off, 64);
            tl = o > tl ? o : tl;
        }
    const int tfu = sum(fail_unsure, ired);
    const int tuf = sum(nuf, ired);
    if (lane == 0 && in) {
        const size_t at = size_t(v) * P.T + tt;
        pmerit[at] = double(tr2);
        plength[at] = tl;
        pcounts[at * 3] = tfu & 0xffff;
        pcounts[at * 3 + 1] = tfu >> 16;
        pcounts[at * 3 + 2] = tuf;
    }
}

// Per variant: merit = sum of the tuple partials (double, tuple order), optical length = max,
// counts summed (the second stage of the reference's prefilter).
__global__ void prefilter_finalize_kernel(int V, int T, const double* pmerit,
                                          const float* plength, const int* pcounts,
                                          double* merit, double* optical, int64_t* failed,
                                          int64_t* uncertain_ok, int64_t* uncertain_failed) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    double m = 0.0;
    float len = 0.0f;
    int64_t f = 0, uo = 0, uf = 0;
    for (int t = 0; t < T; ++t) {
        const size_t i = size_t(v) * T + t;
        m += pmerit[i];
        len = plength[i] > len ? plength[i] : len;
        f += pcounts[i * 3];
        uo += pcounts[i * 3 + 1];
        uf += pcounts[i * 3 + 2];
    }
    merit[v] = m;
    optical[v] = double(len);
    failed[v] = f;
    uncertain_ok[v] = uo;
    uncertain_failed[v] = uf;
}

// ---- FD batch and FD difference -------------------------------------------------------------

// Builds the 2P+1 FD variants of each run from its template variant: variant 0 = x0,
// 2k+1 = x0 + d+_k e_k, 2k+2 = x0 + d-_k e_k (write_fd_variants, variant_generator.cpp:240).
// The template's per-variant arrays are copied, then the variables written.
struct BatchPtrs {
    double* curvature;
    double* thickness;
    double* index;
    double* pupil_radius;
    double* field_angle;
    double* field_target;
    double* reference_curvature;
    double* paraxial_index;
    double* buchdahl;
};
struct ConstBatchPtrs {
    const double* curvature;
    const double* thickness;
    const double* index;
    const double* pupil_radius;
    const double* field_angle;
    const double* field_target;
    const double* reference_curvature;
    const double* paraxial_index;
    const double* buchdahl;
};

// Buchdahl coordinate w of each wavelength and (at [L]) of lambda_ref, computed on the host from
// the batch's wavelengths (valid = 0: not available).
struct OmegaTable {
    double w[kMaxWavelengths + 1];
    int valid;
};

__global__ void point_batch_kernel(ConstBatchPtrs src, BatchPtrs dst, int runs, int per_run,
                                   const int32_t* template_index, int template_per_run, int S,
                                   int L, int F, int P, const int* var_type,
                                   const int* var_surface, const int* var_component,
                                   const double* x0, const double* plus, const double* minus,
                                   const int32_t* live, OmegaTable om) {
    const int vv = blockIdx.x; // destination variant
    const int run = vv / per_run;
    const int j = vv - run * per_run;
    if (run >= runs || (live && run >= *live)) return;
    const int from = template_index ? template_index[run] : template_per_run ? run : 0;
    for (int i = threadIdx.x; i < S; i += blockDim.x) {
        dst.curvature[size_t(vv) * S + i] = src.curvature[size_t(from) * S + i];
        dst.thickness[size_t(vv) * S + i] = src.thickness[size_t(from) * S + i];
        if (src.paraxial_index && dst.paraxial_index)
            dst.paraxial_index[size_t(vv) * S + i] = src.paraxial_index[size_t(from) * S + i];
    }
    for (int i = threadIdx.x; i < S * L; i += blockDim.x)
        dst.index[size_t(vv) * S * L + i] = src.index[size_t(from) * S * L + i];
    for (int i = threadIdx.x; i < F; i += blockDim.x) {
        dst.field_angle[size_t(vv) * F + i] = src.field_angle[size_t(from) * F + i];
        dst.field_target[size_t(vv) * F + i] = src.field_target[size_t(from) * F + i];
        if (src.reference_curvature)
            dst.reference_curvature[size_t(vv) * F + i] = src.reference_curvature[size_t(from) * F + i];
    }
    if (threadIdx.x == 0) dst.pupil_radius[vv] = src.pupil_radius[from];
    if (src.buchdahl && dst.buchdahl)
        for (int i = threadIdx.x; i < 4 * S; i += blockDim.x)
            dst.buchdahl[size_t(vv) * 4 * S + i] = src.buchdahl[size_t(from) * 4 * S + i];
    __syncthreads();
    // variables: x0 of the run, component k replaced for FD variants
    const int kk = j == 0 ? -1 : (j - 1) / 2;
    bool glass = false;
    for (int k = threadIdx.x; k < P; k += blockDim.x) {
        glass = glass || var_type[k] == MKO_VAR_GLASS;
        double x = x0[size_t(run) * P + k];
        if (k == kk) x = (j & 1) ? plus[size_t(run) * P + k] : minus[size_t(run) * P + k];
        const int s = var_surface[k];
        if (var_type[k] == MKO_VAR_CURVATURE)
            dst.curvature[size_t(vv) * S + s] = x;
        else if (var_type[k] == MKO_VAR_GLASS) {
            if (dst.buchdahl && var_component)
                dst.buchdahl[(size_t(vv) * S + s) * 4 + var_component[k]] = x;
        } else
            dst.thickness[size_t(vv) * S + s] = x;
    }
    if (!__any(glass)) return; // one wavefront
    __syncthreads();
    // index of the glass-variable surfaces from their Buchdahl coefficients
    // (VariableSet::apply, variable_set.cpp:271-284; buchdahl_index, dispersion.hpp:93);
    // without coefficients or wavelengths the index becomes NaN (the trace then fails loudly)
    for (int k = threadIdx.x; k < P; k += blockDim.x) {
        if (var_type[k] != MKO_VAR_GLASS || !var_component || var_component[k] != 0) continue;
        const int s = var_surface[k];
        const bool ok = om.valid && dst.buchdahl != nullptr;
        const double* c = ok ? dst.buchdahl + (size_t(vv) * S + s) * 4 : nullptr;
        for (int l = 0; l <= L; ++l) {
#pragma clang fp contract(off)
            double n = __builtin_nan("");
            if (ok) {
                const double w = om.w[l];
                n = c[0] + w * (c[1] + w * (c[2] + w * c[3]));
            }
            if (l < L) dst.index[(size_t(vv) * S + s) * L + l] = n;
            else if (dst.paraxial_index) dst.paraxial_index[size_t(vv) * S + s] = n;
        }
    }
}

// fd_derivative (fd_formula.hpp:39) from the residual at the point and at its two differences. The
// contraction is spelled out, so every kernel that inlines it computes the same bits.
__device__ __forceinline__ double fd_derivative(double a0, double aa, double ab, double da,
                                                double db, uint8_t stencil) {
#pragma clang fp contract(off)
    if (stencil == MKO_STENCIL_ONE_SIDED) {
        const double ga = aa - a0, gb = ab - a0;
        return __builtin_fma(db * db, ga, -(da * da * gb)) / (da * db * (db - da));
    }
    return (aa - ab) / (da - db);
}

// J[i][k][r] = fd_derivative (fd_formula.hpp:39) from the FD residuals; block (i, P) copies r0.
// Status changes per (i, k): rays whose Ok-ness differs between x0 and either point.
__global__ __launch_bounds__(kBlock) void fd_difference_kernel(
    const double* res, int64_t stride, const uint8_t* st, int64_t rays, int runs, int P,
    int64_t rows, const double* step_plus, const double* step_minus, const uint8_t* stencil,
    double* J, double* r0, int64_t* changes, int64_t jstride, int64_t joffset) {
    __shared__ int ired[kWaves];
    const int i = blockIdx.x / (P + 1);
    const int k = blockIdx.x - i * (P + 1);
    const int n = 2 * P + 1;
    const size_t v0 = size_t(i) * n;
    const double* r_0 = res + v0 * stride;
    if (k == P) {
        for (int64_t r = threadIdx.x; r < rows; r += kBlock)
            r0[size_t(i) * jstride + joffset + r] = r_0[r];
        return;
    }
    const double* ra = res + (v0 + 2 * k + 1) * stride;
    const double* rb = res + (v0 + 2 * k + 2) * stride;
    const double da = step_plus[size_t(i) * P + k];
    const double db = step_minus[size_t(i) * P + k];
    const uint8_t sten = stencil[size_t(i) * P + k];
    double* col = J + (size_t(i) * P + k) * jstride + joffset;
    for (int64_t r = threadIdx.x; r < rows; r += kBlock) {
        col[r] = fd_derivative(r_0[r], ra[r], rb[r], da, db, sten);
    }
    if (!st) return;
    int c = 0;
    const uint8_t* s0 = st + v0 * rays;
    const uint8_t* sa = st + (v0 + 2 * k + 1) * rays;
    const uint8_t* sb = st + (v0 + 2 * k + 2) * rays;
    for (int64_t r = threadIdx.x; r < rays; r += kBlock) {
        const bool ok0 = s0[r] == MKO_STATUS_OK;
        c += ((sa[r] == MKO_STATUS_OK) != ok0) || ((sb[r] == MKO_STATUS_OK) != ok0);
    }
    const int total = block_sum(c, ired);
    if (threadIdx.x == 0) changes[size_t(i) * P + k] = total;
}

// ---- FD Jacobian without the differences' residuals -----------------------------------------

// The variables in the order of the first step their differences change: a curvature the step to
// its surface, a thickness the step after it (the last one only the reference sphere, first = S),
// a glass coefficient the steps to its surface and to the next one.
constexpr int kFdMaxVariables = 320;
struct FdPlan {
    int P, parts;
    int32_t var[kFdMaxVariables]; // variable | first step << 16 | glass << 24
};

// FD Jacobian of the trace rows, J[i][k][row] at jstride, and r0, one workgroup of up to 4 waves per
// (run, tuple) of the central FD batch P (runs x (2 plan.P + 1) variants). A difference of a
// variable leaves the rays alone up to the variable's surface: the workgroup takes the rays of the
// run's point through the surfaces once, and at each surface sends a copy of them through the rest
// of the system for both differences of the variables that start there. About half of the
// surface steps of tracing every variant (P = 48, 25 surfaces: 1250 instead of 2328 per ray), and
// the differences' residuals stay in registers: 32 runs x 17920 rays 3.5 + 0.2 ms (every variant
// traced, then differenced in a second kernel) -> 1.95 ms, 0.78 vector instructions per quad cycle.
// Registers capped for 4 waves per SIMD up to 512 rays per tuple in hard mode (28 bytes of spill).
// Both differences of a ray in one pass of the surface loop (two chains): 1.92 ms, not kept. Same
// step, reference sphere, sums in the order of trace_kernel's and difference formula, so J and r0 are
// those of the two kernels bit for bit.
template <bool kSoft, int kRpl>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(kSoft ? (kRpl <= 1 ? 3 : 1) : kRpl <= 2 ? 4 : 1)))
void fd_jacobian_kernel(TraceParams P, FdPlan plan,
                                                             const double* step_plus,
                                                             const double* step_minus,
                                                             const uint8_t* stencil, double* J,
                                                             double* r0, int64_t jstride) {
    extern __shared__ __align__(16) unsigned char fd_lds[];
    __shared__ SampleTable ST;
    __shared__ double red[2][4][kWaves];
    const int Pn = plan.P;
    const int tuple = int(blockIdx.x) / plan.parts;
    const int part = int(blockIdx.x) - tuple * plan.parts;
    const int run = tuple / P.T, tt = tuple - run * P.T;
    const int v0 = run * (2 * Pn + 1);
    const Tuple t = tuple_of(P, v0 * P.T + tt);
    Step* steps = reinterpret_cast<Step*>(fd_lds);
    Step* moved = steps + (P.S + 1); // [P][2 differences][2 steps], in plan order
    const Step* L = steps;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int threads = int(blockDim.x), waves = threads >> 6;
    stage_samples(P, t, ST);
    stage_steps(P, v0, t.l, steps);
    for (int e = tid; e < 4 * Pn; e += threads) {
        const int k = plan.var[e >> 2] & 0xffff, first = (plan.var[e >> 2] >> 16) & 0xff;
        const int s = first + (e & 1);
        if (s <= P.S) moved[e] = step_at(P, v0 + 2 * k + 1 + ((e >> 1) & 1), t.l, s);
    }
    __syncthreads();
    const size_t vf = size_t(t.v) * P.F + t.f;
    const double a = P.pupil_radius[t.v];
    double sin_t, cos_t;
    sincos(P.field_angle[vf], &sin_t, &cos_t);
    const V3<double> M{0.0, P.field_target[vf], L[P.S].t};
    const double kappa = P.ref_kind != MKO_REF_LAST_SURFACE ? P.reference_curvature[vf] : 0.0;

    // a ray on its way: momentum in r.d; st != Ok: it failed
    struct Way {
        Ray r;
        double pen;
        uint8_t st, first;
    };
    const auto advance = [&](Way& w, const Step& k, double nb) {
        if (w.st != MKO_STATUS_OK) return;
        double n_dot;
        if constexpr (kSoft) {
            Soft soft{w.pen, w.first};
            uint8_t branch = 0;
            w.st = mkod::momentum_step_soft(w.r.p, w.r.d, w.r.opl, k, nb, n_dot, soft, branch);
            w.pen = soft.penalty;
            w.first = soft.first;
        } else {
            w.st = mkod::momentum_step(w.r.p, w.r.d, w.r.opl, k, n_dot);
        }
    };
    // the reference sphere: final status in w.st
    const auto finish = [&](Way& w, double n_last, double mz) {
        if (w.st != MKO_STATUS_OK) return;
        const double rn = mkod::rev_rcp(n_last);
        w.r.d = V3<double>{rn * w.r.d.x, rn * w.r.d.y, rn * w.r.d.z};
        if (!(w.r.d.z > 0.0)) {
            w.st = MKO_STATUS_BACKWARD;
            return;
        }
        Soft soft{w.pen, w.first};
        uint8_t rb = 0;
        const uint8_t rst = mkod::reference_step<kSoft>(w.r, V3<double>{M.x, M.y, mz}, kappa,
                                                        P.ref_kind, n_last, soft, rb);
        if constexpr (kSoft) {
            w.pen = soft.penalty;
            w.first = soft.first;
        }
        w.st = !mkod::in_piston(rst) ? rst : kSoft ? soft.first : uint8_t(MKO_STATUS_OK);
    };
    // weight and weighted path of a finished ray
    const auto count = [&](const Way& w, double weight, double& sw, double& swo) {
        if (mkod::in_piston(w.st)) {
            sw += weight;
            swo += weight * w.r.opl;
        }
    };
    const auto penalty_row = [&](const Way& w, double rootw) {
        const double fp = w.st == MKO_STATUS_OK ? 0.0 : mkod::is_soft(w.st) ? w.pen : w.pen + 1.0;
        return t.pscale * rootw * fp;
    };

    double weight[kRpl], rootw[kRpl], base_r[kRpl], base_p[kRpl];
    Way way[kRpl];
    const auto start = [&](int i) {
        Way w{};
        const int k = tid + i * threads;
        w.st = MKO_STATUS_UNSUPPORTED;
        if (k < t.n) {
            const Sample s = sample_at(P, t, ST, k);
            w.r = source_ray(P, t, s, a, sin_t, cos_t, L[0].n);
            const double n0 = L[0].n;
            w.r.d = V3<double>{n0 * w.r.d.x, n0 * w.r.d.y, n0 * w.r.d.z};
            w.st = MKO_STATUS_OK;
            w.first = MKO_STATUS_OK;
            weight[i] = s.weight;
            rootw[i] = s.rootw;
        }
        return w;
    };
    // the point itself: r0
    {
        double sw = 0.0, swo = 0.0;
#pragma unroll
        for (int i = 0; i < kRpl; ++i) {
            weight[i] = rootw[i] = 0.0;
            Way w = start(i);
            for (int s = 1; s < P.S; ++s) advance(w, L[s], L[s - 1].n);
            finish(w, L[P.S - 1].n, M.z);
            count(w, weight[i], sw, swo);
            base_r[i] = mkod::in_piston(w.st) ? w.r.opl : __builtin_nan("");
            base_p[i] = kSoft ? penalty_row(w, rootw[i]) : 0.0;
        }
        sw = wave_sum(sw);
        swo = wave_sum(swo);
        if (lane == 0) {
            red[0][0][wave] = sw;
            red[0][1][wave] = swo;
        }
        __syncthreads();
        double W = red[0][0][0], O = red[0][1][0];
        for (int w = 1; w < waves; ++w) {
            W += red[0][0][w];
            O += red[0][1][w];
        }
        const double piston = W > 0.0 ? O / W : 0.0;
#pragma unroll
        for (int i = 0; i < kRpl; ++i) {
            const int k = tid + i * threads;
            const bool ok = W > 0.0 && !__builtin_isnan(base_r[i]);
            const double e = ok ? base_r[i] - piston : 0.0;
            base_r[i] = t.scale * rootw[i] * e;
            if (k < t.n && part == 0) {
                double* out = r0 + size_t(run) * jstride + t.offset + k;
                out[0] = base_r[i];
                if (kSoft) out[P.rays] = base_p[i];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < kRpl; ++i) way[i] = start(i);
    int q = 0, parity = 0;
    for (int s = 1; s <= P.S; ++s) {
        // `way` is on surface s - 1: the differences whose first step is s
        for (; q < Pn && ((plan.var[q] >> 16) & 0xff) == s; ++q) {
            if (q % plan.parts != part) continue;
            parity ^= 1;
            const int k = plan.var[q] & 0xffff;
            const bool glass = (plan.var[q] >> 24) != 0;
            const size_t ik = size_t(run) * Pn + k;
            double opl[2][kRpl], pen[2][kRpl], sw[2] = {0.0, 0.0}, swo[2] = {0.0, 0.0};
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const Step* mv = moved + (4 * q + 2 * side);
                const double n_last = glass && s == P.S - 1 ? mv[0].n : L[P.S - 1].n;
                const double mz = s == P.S ? mv[0].t : M.z;
#pragma unroll
                for (int i = 0; i < kRpl; ++i) {
                    Way w = way[i];
                    for (int j = s; j < P.S; ++j) {
                        const bool second = glass && j == s + 1;
                        const Step* kj = j == s ? mv : second ? mv + 1 : L + j;
                        advance(w, *kj, second ? mv[0].n : L[j - 1].n);
                    }
                    finish(w, n_last, mz);
                    count(w, weight[i], sw[side], swo[side]);
                    opl[side][i] = mkod::in_piston(w.st) ? w.r.opl : __builtin_nan("");
                    pen[side][i] = kSoft ? penalty_row(w, rootw[i]) : 0.0;
                }
                sw[side] = wave_sum(sw[side]);
                swo[side] = wave_sum(swo[side]);
            }
            if (lane == 0) {
#pragma unroll
                for (int side = 0; side < 2; ++side) {
                    red[parity][2 * side][wave] = sw[side];
                    red[parity][2 * side + 1][wave] = swo[side];
                }
            }
            __syncthreads(); // the other half of red is free: every wave has read it by now
            double W[2], piston[2];
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                double x = red[parity][2 * side][0], o = red[parity][2 * side + 1][0];
                for (int w = 1; w < waves; ++w) {
                    x += red[parity][2 * side][w];
                    o += red[parity][2 * side + 1][w];
                }
                W[side] = x;
                piston[side] = x > 0.0 ? o / x : 0.0;
            }
            const double da = step_plus[ik], db = step_minus[ik];
            const uint8_t sten = stencil[ik];
#pragma unroll
            for (int i = 0; i < kRpl; ++i) {
                const int kr = tid + i * threads;
                if (kr >= t.n) continue;
                double r[2];
#pragma unroll
                for (int side = 0; side < 2; ++side) {
                    const bool ok = W[side] > 0.0 && !__builtin_isnan(opl[side][i]);
                    const double e = ok ? opl[side][i] - piston[side] : 0.0;
                    r[side] = t.scale * rootw[i] * e;
                }
                double* col = J + ik * jstride + t.offset + kr;
                col[0] = fd_derivative(base_r[i], r[0], r[1], da, db, sten);
                if (kSoft)
                    col[P.rays] = fd_derivative(base_p[i], pen[0][i], pen[1][i], da, db, sten);
            }
        }
        if (s < P.S) {
#pragma unroll
            for (int i = 0; i < kRpl; ++i) advance(way[i], L[s], L[s - 1].n);
        }
    }
}

// ---- ADJOINT Jacobian -----------------------------------------------------------------------

// Writes one ray's parameter gradients into its J row: value * factor at column p.
struct RowSink {
    double* col0; // J of the variant
    int64_t rows; // R
    int64_t row;
    double factor;
    __device__ __forceinline__ void write(int p, double value) const {
        if (p >= 0) col0[int64_t(p) * rows + row] = factor * value;
    }
};

// backward_ray (adjoint_backward.hpp:496-580) over the record of a ray with a soft continuation.
// The thickness columns less the common part n (sweep_ray's kFine form).
template <class Sink>
__device__ __forceinline__ void backward_ray(const TraceParams& P, const Step* L,
                                             const ParamMap& map, const Record& rec,
                                             bool reached_image, V3<double> M, double kappa,
                                             double seed_opl, double seed_pen, const Sink& sink,
                                             int l) {
    const int S = P.S;
    const int count = rec.count;
    mkod::RayAdj<double> adj{{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
    uint8_t next_branch = 0;
    double n_carry = 0.0; // adjoint of index[j] from step j + 1 (or the reference sphere)
    // JacobianRowWriter::index: the glass variables of the medium after surface j
    const auto index_sink = [&](int j, double value) {
        if (!map.glass) return;
        const double w = map.omega[l];
        const double slope[3] = {1.0, w, w * w};
#pragma unroll
        for (int c = 0; c < 3; ++c) sink.write(map.glass_col[j][c], value * slope[c]);
    };
    for (int s = count - 1; s >= 0; --s) {
        const V3<double> p = rec.p[s];
        const double rn = mkod::rev_rcp(L[s].n);
        const V3<double> d{rn * rec.P[s].x, rn * rec.P[s].y, rn * rec.P[s].z};
        if (s == count - 1) {
            if (reached_image && count == S) {
                double nib = 0.0;
                const double mz = mkod::reference_step_backward<double>(
                    p, d, M, kappa, P.ref_kind, L[S - 1].n, rec.image_branch, seed_opl, seed_pen,
                    adj, nib);
                sink.write(map.thick_col[S - 1], mz);
                n_carry = nib;
            }
        } else {
            const int j = s + 1;
            double tb = 0.0, cb = 0.0, nbb = 0.0, nab = 0.0;
            mkod::refracting_step_backward<double>(p, d, L[j].t, L[j].c, L[s].n, L[j].n,
                                                   next_branch, seed_opl, seed_pen, adj, tb, cb,
                                                   nbb, nab);
            if ((P.sphere_mask >> j) & 1ull) sink.write(map.curv_col[j], cb);
            sink.write(map.thick_col[s], tb - seed_opl * L[s].n);
            index_sink(j, nab + n_carry);
            n_carry = nbb;
        }
        next_branch = rec.branch[s];
    }
}

// A soft ray's second trace, with its record, and the sweep over it.
template <class Sink>
__device__ __forceinline__ void soft_backward(const TraceParams& P, const Step* L,
                                           const ParamMap& map, const Ray& start, V3<double> M,
                                           double kappa, double seed_opl, double seed_pen,
                                           const Sink& sink, int l) {
    Record rec;
    rec.count = 0;
    rec.image_branch = 0;
    Ray r = start;
    Soft soft{0.0, MKO_STATUS_OK};
    const uint8_t st = trace_ray<true>(P, L, r, M, kappa, soft, rec);
    const bool reached = mkod::in_piston(st);
    backward_ray(P, L, map, rec, reached, M, kappa, reached ? seed_opl : 0.0, seed_pen, sink, l);
}

// The gradients of a regular ray (backward_ray, adjoint_backward.hpp:496-580, with seed 1 for the
// optical path) from its state (p, d) on the last surface, by mkod's reverse sweep. kGlass: the
// index gradients as well, into the glass variables' columns of each medium
// (dn/d(n0, nu1, nu2) = 1, w_l, w_l^2). kFine: a thickness gradient P_z + dP_z is given less its
// common part n, as dP_z - (P_x^2 + P_y^2) / (n + P_z): the projections that follow remove what
// the rays of a tuple have in common (1e4 to 1e5 times the variation for weak beams), and the
// variation then keeps its digits.
template <bool kGlass, bool kFine, class Sink>
__device__ __forceinline__ void sweep_ray(const TraceParams& P, const Step* L, const ParamMap& map,
                                          V3<double> p, V3<double> d, V3<double> M, double kappa,
                                          const Sink& sink, int l) {
    const int S = P.S;
    const double least = first_lane(mkod::sweep_least(L[0].n));
    double mz, length;
    mkod::SweepState w = mkod::sweep_reference(p, d, M, kappa, P.ref_kind, L[S - 1].n, L[S - 1].c,
                                               mz, length);
    sink.write(map.thick_col[S - 1], mz);
    if constexpr (kGlass) length -= mkod::rev_div(mkod::dot(w.P, w.dq), L[S - 1].n);
    for (int j = S - 1;; --j) {
        if constexpr (kGlass) {
            const double wl = map.omega[l];
            sink.write(map.glass_col[j][0], length);
            sink.write(map.glass_col[j][1], length * wl);
            sink.write(map.glass_col[j][2], length * (wl * wl));
        }
        const double cb = mkod::sweep_refract(w, L[j], least);
        if ((P.sphere_mask >> j) & 1ull) sink.write(map.curv_col[j], cb);
        if (kFine) {
            const double n = L[j - 1].n;
            const double t2 = w.P.x * w.P.x + w.P.y * w.P.y;
            sink.write(map.thick_col[j - 1], w.dP.z - mkod::rev_div(t2, n + w.P.z));
        } else {
            sink.write(map.thick_col[j - 1], w.P.z + w.dP.z);
        }
        if (j == 1) break;
        mkod::sweep_transfer<kGlass>(w, L[j], L[j - 1].c, L[j - 1].cna, L[j - 1].n, least,
                                     length);
    }
}

// Stored Jacobian: one workgroup of up to 4 waves per (variant = run, tuple), kRpl rays per lane.
// Each ray is traced and swept backwards at once (no record of its states in memory: only a ray
// with a soft continuation is traced again for its record), its raw gradients going straight into
// the column-major J (J[v][p][row]: a wave writes 512 contiguous bytes per column). After the
// tuple's piston sums the waves take the columns in turn, a column's rays in registers: weighted
// mean, then J(k,p) = s sqrt(W_k) (g_k - gbar_p) for rays in the piston, 0 otherwise
// (adjoint_jacobian.cpp:462-479), one read and one write of J and no barrier per column. Penalty
// rows (soft mode) get pscale sqrt(W_k) times the penalty gradient. r0 rows and the status are
// written as by RESIDUALS. What bounds it: the vector ALU (a trace and a sweep, about 4000
// instructions per ray at 25 surfaces) and 3 x 8 P bytes of J per ray: 0.36 ms for 64 runs x 17920
// rays x 48 variables (1.24 ms with a record of the states in private memory, a pass that cleared
// J and two passes and four barriers per column for the projection).
// wr: weight and s sqrt(W) of each ray of the tuple (0, 0 outside the piston).
template <bool kSoft, bool kGlass, int kRpl>
__global__ __launch_bounds__(kBlock) void adjoint_kernel(TraceParams P, ParamMap map, double* J,
                                                         double* r0, uint8_t* status) {
    extern __shared__ __align__(16) unsigned char adj_lds[];
    __shared__ SampleTable ST;
    __shared__ double red[2][kWaves];
    if (P.live && int(blockIdx.x) / P.T >= *P.live) return;
    const Tuple t = tuple_of(P, blockIdx.x);
    Step* steps = reinterpret_cast<Step*>(adj_lds);
    double2* wr = reinterpret_cast<double2*>(adj_lds + size_t(P.S + 1) * sizeof(Step));
    const Step* L = steps;
    stage_samples(P, t, ST);
    stage_steps(P, t.v, t.l, steps);
    __syncthreads();
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int threads = int(blockDim.x), waves = threads >> 6;
    const size_t vf = size_t(t.v) * P.F + t.f;
    const double a = P.pupil_radius[t.v];
    double sin_t, cos_t;
    sincos(P.field_angle[vf], &sin_t, &cos_t);
    const V3<double> M{0.0, P.field_target[vf], L[P.S].t};
    const double kappa = P.ref_kind != MKO_REF_LAST_SURFACE ? P.reference_curvature[vf] : 0.0;
    const int64_t R = P.stride;
    double* col0 = J + size_t(t.v) * map.P * R;

    double opl[kRpl];
    uint8_t st[kRpl];
    double pen[kRpl];
    double sw = 0.0, swo = 0.0;
#pragma unroll
    for (int i = 0; i < kRpl; ++i) {
        const int k = tid + i * threads;
        st[i] = MKO_STATUS_UNSUPPORTED;
        opl[i] = 0.0;
        pen[i] = 0.0;
        if (k >= t.n) continue;
        const int64_t row = t.offset + k;
        const Sample s = sample_at(P, t, ST, k);
        const Ray start = source_ray(P, t, s, a, sin_t, cos_t, L[0].n);
        Ray r = start;
        Soft soft{0.0, MKO_STATUS_OK};
        LastState last{};
        st[i] = trace_ray<kSoft>(P, L, r, M, kappa, soft, last);
        pen[i] = soft.penalty;
        const bool reached = mkod::in_piston(st[i]);
        if (reached) {
            opl[i] = r.opl;
            sw += s.weight;
            swo += s.weight * r.opl;
        }
        wr[k] = reached ? double2{s.weight, t.scale * s.rootw} : double2{0.0, 0.0};
        if (st[i] == MKO_STATUS_OK)
            sweep_ray<kGlass, true>(P, L, map, last.p, last.d, M, kappa,
                                    RowSink{col0, R, row, 1.0}, t.l);
        if constexpr (kSoft) {
            // penalty rows: zero but for a ray with a continuation, whose sweep may end early
            for (int p = 0; p < map.P; ++p) col0[int64_t(p) * R + P.rays + row] = 0.0;
            if (soft.first != MKO_STATUS_OK) {
                if (reached)
                    soft_backward(P, L, map, start, M, kappa, 1.0, 0.0,
                                  RowSink{col0, R, row, 1.0}, t.l);
                soft_backward(P, L, map, start, M, kappa, 0.0, 1.0,
                              RowSink{col0, R, P.rays + row, t.pscale * s.rootw}, t.l);
            }
        }
    }
    sw = wave_sum(sw);
    swo = wave_sum(swo);
    if (lane == 0) {
        red[0][wave] = sw;
        red[1][wave] = swo;
    }
    __syncthreads(); // also publishes the raw gradients to the workgroup's other waves
    double w_ok = red[0][0], sum = red[1][0];
    for (int w = 1; w < waves; ++w) {
        w_ok += red[0][w];
        sum += red[1][w];
    }
    const bool valid = w_ok > 0.0;
    const double piston = valid ? sum / w_ok : 0.0;
#pragma unroll
    for (int i = 0; i < kRpl; ++i) {
        const int k = tid + i * threads;
        if (k >= t.n) continue;
        const Sample s = sample_at(P, t, ST, k);
        const bool ok = valid && mkod::in_piston(st[i]);
        const double e = ok ? opl[i] - piston : 0.0;
        const int64_t row = t.offset + k;
        r0[size_t(t.v) * R + row] = t.scale * s.rootw * e;
        if (kSoft) {
            const double fp = st[i] == MKO_STATUS_OK ? 0.0
                              : mkod::is_soft(st[i]) ? pen[i]
                                                     : pen[i] + 1.0;
            r0[size_t(t.v) * R + P.rays + row] = t.pscale * s.rootw * fp;
        }
        if (status) status[size_t(t.v) * P.rays + row] = st[i];
    }
    // piston projection: a wave per column, 64 rays at a time in registers (sums in FP64, fixed
    // order); columns that no sweep writes (map.unswept) are zero
    constexpr int kSlots = 4 * kRpl; // 64 lanes, up to 256 kRpl rays
    for (int p = wave; p < map.P; p += waves) {
        double* col = col0 + int64_t(p) * R + t.offset;
        const bool swept = !((map.unswept[p >> 6] >> (p & 63)) & 1ull);
        double g[kSlots], part = 0.0;
#pragma unroll
        for (int i = 0; i < kSlots; ++i) {
            const int k = lane + 64 * i;
            g[i] = 0.0;
            if (k < t.n) {
                const double w = wr[k].x;
                if (swept && w != 0.0) g[i] = col[k];
                part += w * g[i];
            }
        }
        const double mean = valid ? wave_sum(part) / w_ok : 0.0;
#pragma unroll
        for (int i = 0; i < kSlots; ++i) {
            const int k = lane + 64 * i;
            if (k < t.n) col[k] = wr[k].y * (g[i] - mean);
        }
    }
}

// ---- vector-Jacobian product J^T v without J ---------------------------------------------
//
// J^T v of one (variant = run, tuple) per workgroup. The sweep is linear in its seeds
// (ray_gradient_rows, ray_jacobian.hpp:93), so each ray runs it once with
//   seed_opl = s (v_k sqrt(W_k) - W_k m),  m = sum_j v_j sqrt(W_j) / W_ok (rays in the piston),
//   seed_pen = pscale sqrt(W_k) u_k      (soft mode, rays with a failure),
// v and u being the cotangents of the ray's residual and penalty rows: sum_k v_k J(k, p) with
// J(k, p) = s sqrt(W_k) (g_kp - gbar_p) equals sum_k g_kp s (v_k sqrt(W_k) - W_k m), so neither
// J nor the piston-projected columns are formed. The seeds sum to zero, so the common part n of a
// thickness column drops out and is left away (kFine). part[tuple][p]: the tuple's share.

// Hard failure mode: up to 4 waves per tuple, kRpl rays per lane. A first pass traces the rays,
// for W_ok and the sum behind m, and keeps their last states in registers for the sweeps. A
// column's products are summed over groups of 4 lanes by one matrix instruction with a vector of
// ones (v_mfma_f64_4x4x4_4b: lane l holds the sum of the group l / 4 in all four lanes) and added
// to the wave's own 16 sums of the column: 128 bytes of LDS per column and wave, a quarter of a
// slot per lane, so 5 workgroups fit a CU at 48 variables (0.42 ms for 128 runs x 17920 rays; 1.99
// ms with two traces, a record in private memory and a slot per lane: 1.5 waves per SIMD). Every lane
// of a wave runs the sweep (the matrix instruction takes all lanes); those without a regular ray give
// zeros.
struct GroupSink {
    double* acc; // [P][16] of this wave
    int slot;    // lane / 4
    double beta;
    __device__ __forceinline__ void write(int p, double value) const {
        if (p < 0) return;
        const double x = beta != 0.0 ? beta * value : 0.0;
        const double sum = __builtin_amdgcn_mfma_f64_4x4x4f64(x, 1.0, 0.0, 0, 0, 0);
        acc[p * 16 + slot] += sum; // the group's four lanes write the same value
    }
};

template <bool kGlass, int kRpl>
__global__ __launch_bounds__(kBlock) void vjp_kernel(TraceParams P, ParamMap map,
                                                     const double* grad, int64_t gstride,
                                                     double* part) {
    extern __shared__ __align__(16) unsigned char vjp_lds[];
    __shared__ SampleTable ST;
    __shared__ double red[2][kWaves];
    const Tuple t = tuple_of(P, blockIdx.x);
    Step* steps = reinterpret_cast<Step*>(vjp_lds);
    const Step* L = steps;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int threads = int(blockDim.x), waves = threads >> 6;
    double* acc0 = reinterpret_cast<double*>(vjp_lds + size_t(P.S + 1) * sizeof(Step));
    double* acc = acc0 + size_t(wave) * map.P * 16;
    stage_samples(P, t, ST);
    stage_steps(P, t.v, t.l, steps);
    for (int e = lane; e < map.P * 16; e += 64) acc[e] = 0.0;
    __syncthreads();
    const size_t vf = size_t(t.v) * P.F + t.f;
    const double a = P.pupil_radius[t.v];
    double sin_t, cos_t;
    sincos(P.field_angle[vf], &sin_t, &cos_t);
    const V3<double> M{0.0, P.field_target[vf], L[P.S].t};
    const double kappa = P.ref_kind != MKO_REF_LAST_SURFACE ? P.reference_curvature[vf] : 0.0;
    const double* gv = grad + size_t(t.v) * size_t(gstride) + t.offset;
    V3<double> lp[kRpl], ld[kRpl];
    double vr[kRpl], wt[kRpl]; // v sqrt(W) and W of a regular ray, else 0
    double sw = 0.0, svw = 0.0;
#pragma unroll
    for (int i = 0; i < kRpl; ++i) {
        const int k = tid + i * threads;
        lp[i] = V3<double>{0.0, 0.0, 0.0};
        ld[i] = V3<double>{0.0, 0.0, 1.0};
        vr[i] = wt[i] = 0.0;
        if (k >= t.n) continue;
        const Sample smp = sample_at(P, t, ST, k);
        Ray r = source_ray(P, t, smp, a, sin_t, cos_t, L[0].n);
        Soft soft{0.0, MKO_STATUS_OK};
        LastState last{};
        if (trace_ray<false>(P, L, r, M, kappa, soft, last) == MKO_STATUS_OK) {
            lp[i] = last.p;
            ld[i] = last.d;
            wt[i] = smp.weight;
            vr[i] = gv[k] * smp.rootw;
            sw += wt[i];
            svw += vr[i];
        }
    }
    sw = wave_sum(sw);
    svw = wave_sum(svw);
    if (lane == 0) {
        red[0][wave] = sw;
        red[1][wave] = svw;
    }
    __syncthreads();
    double W = red[0][0], SV = red[1][0];
    for (int w = 1; w < waves; ++w) {
        W += red[0][w];
        SV += red[1][w];
    }
    const double m = W > 0.0 ? SV / W : 0.0;
#pragma unroll
    for (int i = 0; i < kRpl; ++i) {
        const double beta = wt[i] != 0.0 ? t.scale * (vr[i] - wt[i] * m) : 0.0;
        if (__ballot(beta != 0.0) == 0) continue; // uniform
        sweep_ray<kGlass, true>(P, L, map, lp[i], ld[i], M, kappa, GroupSink{acc, lane >> 2, beta},
                                t.l);
    }
    __syncthreads();
    for (int p = tid; p < map.P; p += threads) {
        double total = 0.0;
        for (int w = 0; w < waves; ++w)
            for (int i = 0; i < 16; ++i) total += acc0[(size_t(w) * map.P + p) * 16 + i];
        part[size_t(blockIdx.x) * map.P + p] = total;
    }
}

// Soft failure mode: one wave per tuple, the tuple's rays 64 at a time, each lane adding into its
// own slot of acc [P][64] (rays with soft continuations take their sweeps at different surfaces).
struct AccSink {
    double* acc;
    int lane;
    double factor;
    __device__ __forceinline__ void write(int p, double value) const {
        if (p >= 0) acc[p * 64 + lane] += factor * value;
    }
};

template <bool kGlass>
__global__ __launch_bounds__(64) void vjp_soft_kernel(TraceParams P, ParamMap map,
                                                      const double* grad, int64_t gstride,
                                                      double* part) {
    extern __shared__ __align__(16) unsigned char vjp_lds[];
    const Tuple t = tuple_of(P, blockIdx.x);
    Step* steps = reinterpret_cast<Step*>(vjp_lds);
    const Step* L = steps;
    double* acc = reinterpret_cast<double*>(vjp_lds + size_t(P.S + 1) * sizeof(Step)); // [P][64]
    const int lane = threadIdx.x;
    stage_steps(P, t.v, t.l, steps);
    for (int p = 0; p < map.P; ++p) acc[p * 64 + lane] = 0.0;
    __syncthreads();
    const size_t vf = size_t(t.v) * P.F + t.f;
    const double a = P.pupil_radius[t.v];
    double sin_t, cos_t;
    sincos(P.field_angle[vf], &sin_t, &cos_t);
    const V3<double> M{0.0, P.field_target[vf], L[P.S].t};
    const double kappa = P.ref_kind != MKO_REF_LAST_SURFACE ? P.reference_curvature[vf] : 0.0;
    const double* gv = grad + size_t(t.v) * size_t(gstride) + t.offset;
    double sw = 0.0, svw = 0.0;
    for (int k = lane; k < t.n; k += 64) {
        const Sample smp = sample_of(P, t, k);
        Ray r = source_ray(P, t, smp, a, sin_t, cos_t, L[0].n);
        Soft soft{0.0, MKO_STATUS_OK};
        NoRecord nr;
        if (mkod::in_piston(trace_ray<true>(P, L, r, M, kappa, soft, nr))) {
            sw += smp.weight;
            svw += gv[k] * smp.rootw;
        }
    }
    const double W = wave_sum(sw), SV = wave_sum(svw);
    const bool valid = W > 0.0;
    const double m = valid ? SV / W : 0.0;
    for (int k = lane; k < t.n; k += 64) {
        const Sample smp = sample_of(P, t, k);
        const Ray start = source_ray(P, t, smp, a, sin_t, cos_t, L[0].n);
        Ray r = start;
        Soft soft{0.0, MKO_STATUS_OK};
        LastState last{};
        const uint8_t st = trace_ray<true>(P, L, r, M, kappa, soft, last);
        const double beta = valid && mkod::in_piston(st)
                                ? t.scale * (gv[k] * smp.rootw - smp.weight * m)
                                : 0.0;
        if (st == MKO_STATUS_OK) {
            if (beta != 0.0)
                sweep_ray<kGlass, true>(P, L, map, last.p, last.d, M, kappa,
                                        AccSink{acc, lane, beta}, t.l);
            continue;
        }
        const double gamma =
            soft.first != MKO_STATUS_OK ? t.pscale * smp.rootw * gv[P.rays + k] : 0.0;
        if (beta != 0.0 || gamma != 0.0)
            soft_backward(P, L, map, start, M, kappa, beta, gamma, AccSink{acc, lane, 1.0}, t.l);
    }
    for (int p = 0; p < map.P; ++p) {
        const double total = wave_sum(acc[p * 64 + lane]);
        if (lane == 0) part[size_t(blockIdx.x) * map.P + p] = total;
    }
}

// out[v][p] = sum over the run's tuples of part, in (field, wavelength) order.
__global__ void vjp_finalize_kernel(int V, int T, int Pn, const double* part, double* out) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= int64_t(V) * Pn) return;
    const int64_t v = i / Pn, p = i - v * Pn;
    double x = 0.0;
    const double* at = part + v * T * Pn + p;
    int t = 0;
    for (; t + 8 <= T; t += 8) { // 8 loads in flight
        double y[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) y[q] = at[int64_t(t + q) * Pn];
#pragma unroll
        for (int q = 0; q < 8; ++q) x += y[q];
    }
    for (; t < T; ++t) x += at[int64_t(t) * Pn];
    out[i] = x;
}

// ---- ADJOINT fused with the normal equations (hard failure mode) ---------------------------

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
constexpr int kMaxVariablesFused = 96;

// Per-(run, tuple) partial of the normal equations. With a per-tuple shift c (near the tuple's
// weighted mean gradient), o (near its weighted mean OPL) and u_k = sqrt(W_k) (g_k - c) over the
// rays in the piston:
//   C  = sum_k u_k u_k^T                  (P x P, MFMA, float)
//   S  = sum_k W_k (g_k - c)              (P, double)
//   Tr = sum_k W_k (g_k - c) (OPL_k - o)  (P, double)
// the tuple adds s^2 (C - S S^T / W_ok) to J^T J and s^2 (Tr - (piston - o) S) to J^T r0, because
// J(k,p) = s sqrt(W_k) (g_kp - gbar_p), r_k = s sqrt(W_k) (OPL_k - piston) and
// sum_k W_k (OPL_k - piston) = 0 (adjoint_jacobian.cpp:462-479 for J, normal_equations.cpp for
// the products).
struct TupleNormal {
    double w_ok, piston, s2;
};

// Gradient block of one chunk of rays in LDS: P rows of 64 * kNW rays, 4 bytes per ray (a float
// during the sweep, then bf16 hi and lo). Rays sit in groups of 8 (32 bytes); the group's place in
// row p is XOR-swizzled by p, so that the MFMA operand loads (32 rows at one ray group, 16 bytes
// per lane) hit distinct banks. A group's floats and its bf16 values share the same 32 bytes (hi
// in one half, lo in the other, the order alternating with bit 3 of the swizzled slot for the
// same reason), so the 8 lanes of a group -- one wave -- convert in place without a barrier.
template <int kNW>
struct GradLayout {
    static constexpr int kRow = 64 * kNW;
    static constexpr int kRowBytes = 4 * kRow;
    static constexpr int kMask = kRow / 8 >= 16 ? 15 : kRow / 8 - 1;
    __device__ static __forceinline__ int slot(int group, int p) { return group ^ (p & kMask); }
    __device__ static __forceinline__ int float_off(int p, int k) {
        return p * kRowBytes + ((4 * k) ^ ((p & kMask) << 5));
    }
    __device__ static __forceinline__ int hi_off(int p, int s) {
        return p * kRowBytes + 32 * s + (((s >> 3) & 1) << 4);
    }
    __device__ static __forceinline__ int lo_off(int p, int s) {
        return p * kRowBytes + 32 * s + ((((s >> 3) & 1) ^ 1) << 4);
    }
};

// Gradient sink of the fused kernel. Every lane of the wave runs the sweep (those without a
// reached ray on a placeholder state), so column p is written by all lanes together: the value of
// the wave's first lane with a reached ray (pilot) is kept in lane p mod 64 of the wave's pilot
// registers and each lane stores its difference to it in float. The float then carries the
// variation of the gradient over the pupil, not its (often much larger) common part.
template <int kRows>
struct Pilots {
    int lo[kRows] = {}, hi[kRows] = {};
    __device__ __forceinline__ double value(int h) const { return __hiloint2double(hi[h], lo[h]); }
};
// v with lane `lane`'s value replaced by x (both wave-uniform)
__device__ int write_lane(int x, int lane, int v) __asm("llvm.amdgcn.writelane.i32");
template <int kNW, int kRows>
struct SwzSink {
    unsigned char* G; // gradient block
    Pilots<kRows>& pilots;
    int k;      // ray of the chunk (thread)
    int leader; // the wave's first lane with a reached ray (uniform)
    __device__ __forceinline__ void write(int p, double value) const {
        if (p < 0) return;
        const int lo = __builtin_amdgcn_readlane(__double2loint(value), leader);
        const int hi = __builtin_amdgcn_readlane(__double2hiint(value), leader);
        *reinterpret_cast<float*>(G + GradLayout<kNW>::float_off(p, k)) =
            float(value - __hiloint2double(hi, lo));
        if (kRows == 1 || p < 64) {
            pilots.lo[0] = write_lane(lo, p, pilots.lo[0]);
            pilots.hi[0] = write_lane(hi, p, pilots.hi[0]);
        } else {
            pilots.lo[kRows - 1] = write_lane(lo, p - 64, pilots.lo[kRows - 1]);
            pilots.hi[kRows - 1] = write_lane(hi, p - 64, pilots.hi[kRows - 1]);
        }
    }
};

// Orders a wave's LDS accesses across its lanes (they execute in order; this keeps the compiler
// from moving them).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Value of lane I of the caller's row of 16 lanes.
template <int I>
__device__ __forceinline__ double row_lane(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x150 + I, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x150 + I, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// Row sums of one wave's 64 rays in the gradient block: A[h] = sum_k W_k G[p][k] and
// B[h] = sum_k V_k G[p][k] for row p = lane + 64 h, G the stored floats of ray k of the wave, W_k and
// V_k lane k's values. 16 rows at a time: a row of 16 lanes takes the rays of its own 16 lanes
// (their W and V broadcast along the row once), 16-byte words of G; then the four rows of lanes
// are added. One lane per row with W and V by readlane took twice the instructions (16 of 64 lanes
// idle at 48 rows, four readlanes per ray).
template <int kNW, int kRows>
__device__ __forceinline__ void wave_row_sums(const unsigned char* G, int Pn, int wave, int lane,
                                              double wk, double vk, double (&A)[kRows],
                                              double (&B)[kRows]) {
    using Lay = GradLayout<kNW>;
    const int r = lane & 15, seg = lane >> 4;
    double w[16], v[16];
    const auto spread = [&](auto I) {
        constexpr int i = decltype(I)::value;
        w[i] = row_lane<i>(wk);
        v[i] = row_lane<i>(vk);
    };
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (spread(std::integral_constant<int, I>{}), ...);
    }(std::make_integer_sequence<int, 16>{});
#pragma unroll
    for (int h = 0; h < kRows; ++h) {
        A[h] = B[h] = 0.0;
#pragma unroll 1
        for (int q = 0; q < 4; ++q) {
            const int first = 64 * h + 16 * q;
            if (first >= Pn) break; // uniform
            const int p = min(first + r, Pn - 1); // rows >= P: the last one again, not used
            const unsigned char* row = G + size_t(p) * Lay::kRowBytes;
            double a = 0.0, b = 0.0;
#pragma unroll
            for (int g2 = 0; g2 < 2; ++g2) {
                const unsigned char* at = row + 32 * ((8 * wave + 2 * seg + g2) ^ (p & Lay::kMask));
                const float4 x = *reinterpret_cast<const float4*>(at);
                const float4 y = *reinterpret_cast<const float4*>(at + 16);
                const float gv[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const double g = double(gv[i]);
                    a = __fma_rn(w[8 * g2 + i], g, a);
                    b = __fma_rn(v[8 * g2 + i], g, b);
                }
            }
#pragma unroll
            for (int off = 16; off <= 32; off <<= 1) {
                a += __shfl_xor(a, off, 64);
                b += __shfl_xor(b, off, 64);
            }
            if (seg == q) {
                A[h] = a;
                B[h] = b;
            }
        }
    }
}

// C tile t of the upper triangle of a tg x tg grid of 32 x 32 tiles, row-major: (I, J), I <= J.
__device__ __forceinline__ void tile_of(int t, int tg, int& I, int& J) {
    I = 0;
    while (t >= tg - I) {
        t -= tg - I;
        ++I;
    }
    J = I + t;
}

// Dynamic LDS of adjoint_normal_kernel<kNW> for P variables and S surfaces: the step table, the
// gradient block (at least the 4 KB per wave that the waves' sums of a tile take at the end), then
// one double per variable and wave. The table is sized by the batch: at 25 surfaces and 48
// variables a workgroup of 4 waves takes 52.8 KB and three fit a CU, with a table for 64 surfaces
// two (2.69 instead of 2.26 ms per 512 runs).
template <int kNW>
constexpr size_t fused_block_bytes(int Pn) {
    const size_t block = size_t(Pn) * GradLayout<kNW>::kRowBytes, tiles = size_t(kNW) * 4096;
    return kNW > 1 && block < tiles ? tiles : block;
}
template <int kNW>
constexpr size_t fused_lds_bytes(int Pn, int S) {
    return size_t(S + 1) * sizeof(Step) + fused_block_bytes<kNW>(Pn) +
           size_t(kNW) * Pn * sizeof(double);
}

// One workgroup of kNW waves per (run, tuple); the tuple's rays in chunks of 64 kNW, one ray per
// thread. A wave keeps to its own 64 rays of a chunk, so that after the first chunk the waves run
// without barriers and one wave's sweep overlaps another's products. Per chunk: the forward trace
// in double (or, kStates, the last state and OPL of each ray from a MERIT trace of the same point,
// mko_internal::RayStates; the next chunk's are loaded while this one is worked on), the reverse
// sweep into the LDS gradient block (pilot-relative floats); S and Tr of the wave's rays in FP64
// from row sums, lane p holding variable p's (p + 64 in a second set); the wave's part of the
// block rewritten in place as bf16 hi / lo, 8 rays of a row per lane; C on MFMA
// (v_mfma_f32_32x32x16_bf16, 3 products, every upper tile of the 32 x 32 tile grid in each wave).
// At the end the waves' C, S and Tr are added in wave order through the LDS. The shift c is the
// weighted mean gradient of the first chunk that holds a reached ray, o its weighted mean OPL; its
// exchange between the waves is the chunk loop's only barriers. kNW 1: tuples of at most 64 rays,
// one chunk.
// What bounds it: FP64 issue on the vector ALU; 3 waves per SIMD (LDS: 192 bytes per ray at 48
// variables), 2 above 64 variables, whose 6 tiles take 96 registers. Measured against tiles spread
// over the waves, a barrier between every phase, a ray per lane in the conversion and S and Tr
// slots per wave in memory: 256 runs x 17920 rays x 48 variables on stored states 0.85 -> 0.81 ms,
// 512 runs with their own trace 2.21 -> 2.04, 301 runs of 20 tuples of 48 rays 0.058 -> 0.047; the
// sweep with its sink is 112 of the vector instructions per ray-surface.
template <int kNW, int kPMax, bool kStates, bool kGlass>
__global__ __launch_bounds__(64 * kNW) __attribute__((amdgpu_waves_per_eu(kPMax > 64 ? 2 : 3)))
void adjoint_normal_kernel(TraceParams P, ParamMap map, float* partC, double* partST,
                           TupleNormal* partT, mko_internal::RayStates states) {
    using Lay = GradLayout<kNW>;
    constexpr int kThreads = 64 * kNW;
    constexpr int kTileGrid = (kPMax + 31) / 32;
    constexpr int kTiles = kTileGrid * (kTileGrid + 1) / 2;
    constexpr int kRows = kPMax > 64 ? 2 : 1; // variables per lane
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ double wsum_l[kNW], osum_l[kNW];
    if (P.live && int(blockIdx.x) / P.T >= *P.live) return;
    const Tuple t = tuple_of(P, blockIdx.x);
    Step* L = reinterpret_cast<Step*>(lds);
    stage_steps(P, t.v, t.l, L);
    const int Pn = map.P;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = kNW == 1 ? 0 : tid >> 6;
    unsigned char* G = lds + size_t(P.S + 1) * sizeof(Step);
    double* xchg = reinterpret_cast<double*>(G + fused_block_bytes<kNW>(Pn)); // [kNW][P]
    // every column that a sweep reaches is written for every ray; the others stay zero
    {
        float4* z = reinterpret_cast<float4*>(G);
        const int words = Pn * (Lay::kRowBytes / 16);
        for (int e = tid; e < words; e += kThreads) z[e] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    __syncthreads();
    const size_t vf = size_t(t.v) * P.F + t.f;
    // block-uniform values in scalar registers (they stay live across the sweep)
    const double a = first_lane(P.pupil_radius[t.v]);
    double sin_t, cos_t;
    sincos(P.field_angle[vf], &sin_t, &cos_t);
    sin_t = first_lane(sin_t);
    cos_t = first_lane(cos_t);
    const V3<double> M{0.0, first_lane(P.field_target[vf]), first_lane(L[P.S].t)};
    const double kappa =
        first_lane(P.ref_kind != MKO_REF_LAST_SURFACE ? P.reference_curvature[vf] : 0.0);
    const int tg = (Pn + 31) / 32;
    const size_t tuple = size_t(blockIdx.x);
    f32x16 acc[kTiles];
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
    double S_p[kRows] = {}, T_p[kRows] = {}, shift[kRows] = {};
    double sw = 0.0, swo = 0.0, o_shift = 0.0;
    bool shift_ready = false;
    const int nchunks = kNW == 1 ? 1 : (t.n + kThreads - 1) / kThreads;
    // when the tuple's spoke count divides the chunk, a lane's spoke (k mod M) is the same in every
    // chunk: its angle is formed once here and a ray's sample needs only its ring (the same
    // functions as sample_of, hence the same bits)
    const bool fixed_spoke = !kStates && kThreads % t.M == 0;
    Sample spoke{};
    if (fixed_spoke) spoke_of(P, t, tid % t.M, spoke);
    double st[7];
    const auto load_states = [&](int k) {
        st[6] = __builtin_nan("");
        if (k < t.n) {
            const double* at = states.data + state_index(states, t.v, 0, t.offset + k);
            const int64_t stride = states.slots * states.rays;
#pragma unroll
            for (int c = 0; c < 7; ++c) st[c] = at[c * stride];
        }
    };
    if constexpr (kStates) load_states(tid);
    for (int ch = 0; ch < nchunks; ++ch) {
        const int k = ch * kThreads + tid;
        double wk = 0.0, opl = 0.0;
        bool ok = false;
        LastState last{V3<double>{0.0, 0.0, 0.0}, V3<double>{0.0, 0.0, 1.0}, 0};
        if (k < t.n) {
            Sample smp{};
            if constexpr (kStates) {
                ring_of(P, t, k / t.M, smp);
                opl = st[6];
                ok = !__builtin_isnan(opl);
                if (ok) {
                    last.p = V3<double>{st[0], st[1], st[2]};
                    last.d = V3<double>{st[3], st[4], st[5]};
                }
            } else {
                if (fixed_spoke) {
                    smp = spoke;
                    ring_of(P, t, k / t.M, smp);
                } else {
                    smp = sample_of(P, t, k);
                }
                Ray r = source_ray(P, t, smp, a, sin_t, cos_t, L[0].n);
                Soft soft{0.0, MKO_STATUS_OK};
                ok = trace_ray<false>(P, static_cast<const Step*>(L), r, M, kappa, soft, last) ==
                     MKO_STATUS_OK;
                opl = r.opl;
            }
            wk = ok ? smp.weight : 0.0;
        }
        Pilots<kRows> pilots;
        if (!ok) opl = 0.0;
        sw += wk;
        swo += wk * opl;
        const uint64_t okmask = __ballot(ok);
        if (okmask) { // uniform
            sweep_ray<kGlass, false>(P, L, map, last.p, last.d, M, kappa,
                                     SwzSink<kNW, kRows>{G, pilots, tid,
                                                         int(__builtin_ctzll(okmask))},
                                     t.l);
        }
        if (!ok)
            for (int p = 0; p < Pn; ++p)
                *reinterpret_cast<float*>(G + Lay::float_off(p, tid)) = 0.0f;
        if constexpr (kStates)
            if (ch + 1 < nchunks) load_states(k + kThreads);
        wave_sync();
        // this wave's weight sum W_w; the first chunk with a reached ray fixes o = sum W OPL / W
        const double ww = wave_sum(wk);
        double W = 0.0;
        if (!shift_ready) {
            const double wo = wave_sum(wk * opl);
            if (lane == 0) {
                wsum_l[wave] = ww;
                osum_l[wave] = wo;
            }
            __syncthreads();
            double WO = 0.0;
#pragma unroll
            for (int w = 0; w < kNW; ++w) {
                W += wsum_l[w];
                WO += osum_l[w];
            }
            if (!(W > 0.0)) { // no reached ray yet: nothing of this chunk counts
                __syncthreads();
                continue;
            }
            o_shift = WO / W;
        }
        // A_p = sum_k W_k G_pk and B_p = sum_k W_k (OPL_k - o) G_pk over the wave's rays, G the
        // stored floats relative to the wave's pilot: the parts of S and Tr that do not depend on
        // the shift c (S = A + (pilot - c) W_w, Tr = B + (pilot - c) V_w)
        const double vk = ok ? wk * (opl - o_shift) : 0.0;
        double A[kRows], B[kRows];
        wave_row_sums<kNW, kRows>(G, Pn, wave, lane, wk, vk, A, B);
        const double vw = wave_sum(vk);
        if (!shift_ready) {
            // c = sum_w (W_w pilot_w + A_w) / W, the chunk's weighted mean gradient
#pragma unroll
            for (int h = 0; h < kRows; ++h) {
                const int p = lane + 64 * h;
                if (p < Pn)
                    xchg[wave * Pn + p] = __fma_rn(ww, pilots.value(h), A[h]);
            }
            __syncthreads();
#pragma unroll
            for (int h = 0; h < kRows; ++h) {
                const int p = lane + 64 * h;
                if (p < Pn) {
                    double c = xchg[p];
#pragma unroll
                    for (int w = 1; w < kNW; ++w) c += xchg[w * Pn + p];
                    shift[h] = c / W;
                }
            }
            shift_ready = true;
        }
        // S and Tr of the wave's rays; delta = pilot - c for the bf16 conversion
        float delta[kRows];
#pragma unroll
        for (int h = 0; h < kRows; ++h) {
            const double d = pilots.value(h) - shift[h];
            S_p[h] += A[h] + d * ww;
            T_p[h] += B[h] + d * vw;
            delta[h] = float(d);
        }
        // u = sqrt(W) (g - c), split into bf16 hi + lo in place: a lane takes 8 rays (32 bytes) of
        // one row at a time
        {
            const float root = __builtin_sqrtf(float(wk));
            const int g8 = lane & 7, r8 = lane >> 3;
            float sq[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) sq[i] = __shfl(root, 8 * g8 + i, 64);
            const int rows8 = (Pn + 7) / 8;
#pragma unroll 2
            for (int it = 0; it < rows8; ++it) {
                const int p = r8 + 8 * it;
                float d = __shfl(delta[0], p & 63, 64);
                if (kRows == 2 && it >= 8) d = __shfl(delta[kRows - 1], p & 63, 64);
                if (p < Pn) {
                    const int slot = Lay::slot(8 * wave + g8, p);
                    unsigned char* at = G + size_t(p) * Lay::kRowBytes + 32 * slot;
                    const float4 x = *reinterpret_cast<const float4*>(at);
                    const float4 y = *reinterpret_cast<const float4*>(at + 16);
                    const float g[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
                    bf16x8 hi, lo;
#pragma unroll
                    for (int i = 0; i < 8; i += 2) {
                        const f32x2 u{sq[i] * (g[i] + d), sq[i + 1] * (g[i + 1] + d)};
                        const bf16x2 h2 = __builtin_convertvector(u, bf16x2);
                        const f32x2 rest{u.x - float(h2[0]), u.y - float(h2[1])};
                        const bf16x2 l2 = __builtin_convertvector(rest, bf16x2);
                        hi[i] = h2[0];
                        hi[i + 1] = h2[1];
                        lo[i] = l2[0];
                        lo[i + 1] = l2[1];
                    }
                    const int swap = ((slot >> 3) & 1) << 4;
                    *reinterpret_cast<bf16x8*>(at + swap) = hi;
                    *reinterpret_cast<bf16x8*>(at + (swap ^ 16)) = lo;
                }
            }
        }
        wave_sync();
        // C over the wave's 64 rays, 16 at a time: operand lane = (row lane % 32 of a 32-row block,
        // rays 8 (lane / 32) ...), hi*hi + hi*lo + lo*hi. Rows >= P take the last row's values:
        // their products are not stored.
        {
            const int m = lane & 31, kb = lane >> 5;
#pragma unroll
            for (int step = 0; step < 4; ++step) {
                const int grp = 8 * wave + 2 * step + kb;
                bf16x8 hi[kTileGrid], lo[kTileGrid];
#pragma unroll
                for (int I = 0; I < kTileGrid; ++I) {
                    const int p = min(I * 32 + m, Pn - 1);
                    const int slot = Lay::slot(grp, p);
                    hi[I] = *reinterpret_cast<const bf16x8*>(G + Lay::hi_off(p, slot));
                    lo[I] = *reinterpret_cast<const bf16x8*>(G + Lay::lo_off(p, slot));
                }
                int i = 0;
#pragma unroll
                for (int I = 0; I < kTileGrid; ++I)
#pragma unroll
                    for (int J = I; J < kTileGrid; ++J, ++i) {
                        if (J >= tg) continue; // uniform
                        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi[I], hi[J], acc[i], 0, 0, 0);
                        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi[I], lo[J], acc[i], 0, 0, 0);
                        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo[I], hi[J], acc[i], 0, 0, 0);
                    }
            }
        }
        wave_sync();
    }
    // the waves' sums added in wave order. A tile's lane holds column n = lane % 32 of rows
    // 8 (e / 4) + 4 (lane / 32) + e % 4.
    float* C = partC + tuple * size_t(Pn) * Pn;
    int i = 0;
#pragma unroll
    for (int I = 0; I < kTileGrid; ++I)
#pragma unroll
        for (int J = I; J < kTileGrid; ++J, ++i) {
            if (J >= tg) continue; // uniform
            const auto put = [&](int e, float value) {
                const int row = I * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                const int col = J * 32 + (lane & 31);
                if (row < Pn && col < Pn) C[size_t(row) * Pn + col] = value;
            };
            if constexpr (kNW == 1) {
#pragma unroll
                for (int e = 0; e < 16; ++e) put(e, acc[i][e]);
            } else {
                float* X = reinterpret_cast<float*>(G); // [kNW][16][64]
                __syncthreads();
#pragma unroll
                for (int e = 0; e < 16; ++e) X[(wave * 16 + e) * 64 + lane] = acc[i][e];
                __syncthreads();
#pragma unroll
                for (int q = 0; q < 16 / kNW; ++q) {
                    const int e = wave * (16 / kNW) + q;
                    float x = X[e * 64 + lane];
#pragma unroll
                    for (int w = 1; w < kNW; ++w) x += X[(w * 16 + e) * 64 + lane];
                    put(e, x);
                }
            }
        }
    sw = wave_sum(sw);
    swo = wave_sum(swo);
    double* X = reinterpret_cast<double*>(G); // [kNW][2 P]
    __syncthreads();
    if (lane == 0) {
        wsum_l[wave] = sw;
        osum_l[wave] = swo;
    }
#pragma unroll
    for (int h = 0; h < kRows; ++h) {
        const int p = lane + 64 * h;
        if (p < Pn) {
            X[wave * 2 * Pn + p] = S_p[h];
            X[wave * 2 * Pn + Pn + p] = T_p[h];
        }
    }
    __syncthreads();
    double* slot_st = partST + tuple * 2 * Pn;
    for (int e = tid; e < 2 * Pn; e += kThreads) {
        double x = X[e];
#pragma unroll
        for (int w = 1; w < kNW; ++w) x += X[w * 2 * Pn + e];
        slot_st[e] = x;
    }
    if (tid == 0) {
        double w_ok = wsum_l[0], sum = osum_l[0];
#pragma unroll
        for (int w = 1; w < kNW; ++w) {
            w_ok += wsum_l[w];
            sum += osum_l[w];
        }
        // piston - o, the OPL shift of Tr
        partT[tuple] = TupleNormal{w_ok, w_ok > 0.0 ? sum / w_ok - o_shift : 0.0,
                                   t.scale * t.scale};
    }
}

// a = sum_t s_t^2 (C_t - S_t S_t^T / W_t), g = sum_t s_t^2 (Tr_t - (piston_t - o_t) S_t), tuples
// in (field, wavelength) order; `parts` workgroups per run, each with 256 kE entries of the upper
// triangle (mirrored on output), kE per thread; the tuples' S, Tr and factors are staged through
// LDS 16 tuples at a time and the C of 4 tuples are loaded together (the sum over the tuples is
// one dependent chain per entry, their loads are not). What bounds it is latency up to some
// hundred runs, then the reading of C (4 P^2 bytes per tuple): one entry per thread and more
// workgroups, or five and fewer that stage S (finalize_entries). Runs of 35 tuples and 48
// variables, before (one workgroup per run, a tuple at a time) and now: 256 runs 98 -> 25 us, 512
// runs 95 -> 34 us. The contraction is spelled out, so both instantiations give the same bits.
constexpr int kFinalizeChunk = 16;

template <int kE>
__global__ __launch_bounds__(256) void adjoint_normal_finalize_kernel(
    int T, int Pn, int parts, const float* partC, const double* partST, const TupleNormal* partT,
    double* a, double* g, const int32_t* live) {
    extern __shared__ double S_l[]; // [kFinalizeChunk][2 P]
    __shared__ double f1[kFinalizeChunk], f2[kFinalizeChunk], pist[kFinalizeChunk];
    const int v = int(blockIdx.x) / parts, part = int(blockIdx.x) - v * parts;
    if (live && v >= *live) return;
    const int tid = threadIdx.x;
    const int nu = Pn * (Pn + 1) / 2;
    int eq[kE], ep[kE];
    double acc[kE];
#pragma unroll
    for (int i = 0; i < kE; ++i) {
        acc[i] = 0.0;
        // upper-triangle index u -> (q, p), q <= p, row-major over q: row q starts at
        // q (2 P + 1 - q) / 2; the root of that quadratic, corrected to the row
        const int u = min((part * kE + i) * 256 + tid, nu - 1);
        const float b = float(2 * Pn + 1);
        int q = int(0.5f * (b - __builtin_sqrtf(fmaxf(b * b - 8.0f * float(u), 0.0f))));
        while (q > 0 && q * (2 * Pn + 1 - q) / 2 > u) --q;
        while ((q + 1) * (2 * Pn - q) / 2 <= u) ++q;
        eq[i] = q;
        ep[i] = q + u - q * (2 * Pn + 1 - q) / 2;
    }
    double gacc = 0.0;
    const float* C0 = partC + size_t(v) * T * size_t(Pn) * Pn;
    for (int t0 = 0; t0 < T; t0 += kFinalizeChunk) {
        const int nt = min(kFinalizeChunk, T - t0);
        for (int e = tid; e < nt * 2 * Pn; e += 256)
            S_l[e] = partST[(size_t(v) * T + t0) * 2 * Pn + e];
        if (tid < nt) {
            const TupleNormal tn = partT[size_t(v) * T + t0 + tid];
            const bool valid = tn.w_ok > 0.0;
            f1[tid] = valid ? tn.s2 : 0.0;
            f2[tid] = valid ? tn.s2 / tn.w_ok : 0.0;
            pist[tid] = valid ? tn.piston : 0.0;
        }
        __syncthreads();
        for (int tt = 0; tt < nt; tt += 4) {
            float c[4][kE];
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int i = 0; i < kE; ++i) {
                    const size_t tu = size_t(t0 + min(tt + x, nt - 1));
                    c[x][i] = C0[(tu * Pn + eq[i]) * Pn + ep[i]];
                }
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                if (tt + x >= nt) break; // uniform
                const double* St = S_l + (tt + x) * 2 * Pn;
#pragma unroll
                for (int i = 0; i < kE; ++i)
                    acc[i] += __builtin_fma(f1[tt + x], double(c[x][i]),
                                            -(f2[tt + x] * (St[ep[i]] * St[eq[i]])));
                if (part == 0 && tid < Pn)
                    gacc = __builtin_fma(f1[tt + x],
                                         __builtin_fma(-pist[tt + x], St[tid], St[Pn + tid]), gacc);
            }
        }
        __syncthreads();
    }
    double* A = a + size_t(v) * Pn * Pn;
#pragma unroll
    for (int i = 0; i < kE; ++i) {
        if ((part * kE + i) * 256 + tid < nu) {
            A[size_t(eq[i]) * Pn + ep[i]] = acc[i];
            A[size_t(ep[i]) * Pn + eq[i]] = acc[i];
        }
    }
    if (part == 0 && tid < Pn) g[size_t(v) * Pn + tid] = gacc;
}

// ---- Gram: A = J^T J, g = J^T r0 per run ----------------------------------------------------

typedef __attribute__((ext_vector_type(4))) double f64x4;

// Each element is one FMA chain over the rows in ascending order starting from 0 (gram_dot,
// normal_equations.hpp:19), products of the stored J values: bitwise the host definition.
// v_mfma_f64_16x16x4_f64 adds its four products to the accumulator as that chain does (measured
// bit for bit on MI355X against the VALU chain over rows of mixed signs and 24 decades, subnormal
// numbers, zeros of either sign, infinities and NaN; the GPU tests hold it), so J^T J runs on it in
// 16 x 16 tiles; operand lane l: A(m = l % 16, k = l / 16), B(k = l / 16, n = l % 16), result lane l,
// element e: row 4 e + l / 16, column l % 16. g is a VALU chain per column beside the tiles: as a
// matrix column it would cost a row of tiles of its own (10 instead of 6 at 48 variables).
//
// One workgroup of 8 waves per (run, part): the units (a wave of 64 columns of g, or one upper
// tile) are cut into `parts` ranges, a wave takes kT of its range; the columns that the range
// needs are staged kC rows at a time, one wave load per 64 rows of a column, the next rows
// loaded into registers while the tiles run on the present ones. What bounds it: a tile's chain
// is rows / 4 dependent matrix instructions of 16 passes (17920 rows: 0.12 ms however many runs),
// so a few runs are spread over more workgroups, at most one tile per SIMD; with many runs the
// reading of J (7 MB per run at 48 variables). Measured at 48 variables and 17920 rows, against
// one 64 x 64 tile of 4 x 4 VALU chains per thread and workgroup: 1 run 0.31 (2.65) ms, 64 runs
// 0.34 (3.21) ms, 1024 runs 1.79 (5.03) ms (3.9 TB/s of J); 1024 runs of 96 variables and 1200
// rows 0.38 (1.16) ms.
template <int kT, int kC, int kV>
__global__ __launch_bounds__(512) void gram_kernel(const double* J, const double* r0, int P,
                                                   int64_t rows, int parts, int upp, double* a,
                                                   double* g, const int32_t* live) {
    constexpr int kLd = kC + 2; // doubles; 2 modulo 32: a tile's 16 columns x 2 rows hit all banks
    constexpr int kH = kC / 64; // wave loads per column and stage
    extern __shared__ __align__(16) double Xs[]; // [16 tg + 1][kLd], r0 last
    const int run = int(blockIdx.x) / parts, part = int(blockIdx.x) - run * parts;
    if (live && run >= *live) return;
    const int tg = (P + 15) / 16, gw = (P + 63) / 64;
    const int units = gw + tg * (tg + 1) / 2;
    const int first = part * upp, last = min(units, first + upp);
    if (first >= last) return; // no such part (gram_plan makes none)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, kk = lane >> 4;
    f64x4 acc[kT];
    double gacc[kT];
    int tI[kT], tJ[kT]; // unit: tile (I, J); (-2, w): columns 64 w ... of g; (-1, .): none
#pragma unroll
    for (int i = 0; i < kT; ++i) {
        acc[i] = f64x4{0.0, 0.0, 0.0, 0.0};
        gacc[i] = 0.0;
        tI[i] = tJ[i] = -1;
        const int u = first + wave + 8 * i;
        if (u < last) {
            if (u < gw) {
                tI[i] = -2;
                tJ[i] = u;
            } else {
                tile_of(u - gw, tg, tI[i], tJ[i]);
            }
        }
    }
    // the columns staged: from the first tile's row panel on (all with a g unit)
    int c0 = 0;
    if (first >= gw) {
        int J0;
        tile_of(first - gw, tg, c0, J0);
        c0 *= 16;
    }
    const bool with_r0 = first < gw;
    const int ncols = P - c0 + (with_r0 ? 1 : 0);
    const double* Jr = J + size_t(run) * P * rows;
    const double* rr = r0 + size_t(run) * rows;
    double* Xr = Xs + size_t(16 * tg) * kLd;
    for (int e = tid; e < (16 * tg - P) * kLd; e += 512) Xs[size_t(P) * kLd + e] = 0.0;
    double next[kV];
    auto load = [&](int64_t base) {
#pragma unroll
        for (int i = 0; i < kV; ++i) {
            const int x = wave + 8 * (i / kH); // staged column
            const int64_t row = base + 64 * (i % kH) + lane;
            const int c = c0 + x;
            next[i] = 0.0;
            if (x < ncols && row < rows) next[i] = c < P ? Jr[size_t(c) * rows + row] : rr[row];
        }
    };
    load(0);
    for (int64_t base = 0; base < rows; base += kC) {
        const int n = int(rows - base < kC ? rows - base : kC);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kV; ++i) {
            const int x = wave + 8 * (i / kH), c = c0 + x;
            if (x < ncols) (c < P ? Xs + size_t(c) * kLd : Xr)[64 * (i % kH) + lane] = next[i];
        }
        __syncthreads();
        if (base + kC < rows) load(base + kC);
#pragma unroll
        for (int i = 0; i < kT; ++i) {
            if (tI[i] >= 0) {
                const double* xa = Xs + size_t(tI[i] * 16 + m) * kLd + kk;
                const double* xb = Xs + size_t(tJ[i] * 16 + m) * kLd + kk;
                const int steps = n >> 2; // the last 1 ... 3 rows below
#pragma unroll 8
                for (int st = 0; st < steps; ++st)
                    acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(xa[4 * st], xb[4 * st], acc[i],
                                                                  0, 0, 0);
            } else if (tI[i] == -2) {
                const int p = tJ[i] * 64 + lane;
                const double* x = Xs + size_t(p < P ? p : 0) * kLd;
#pragma unroll 8
                for (int r = 0; r < n; ++r) gacc[i] = __fma_rn(x[r], Xr[r], gacc[i]);
            }
        }
    }
    // the rows beyond the last multiple of 4, still staged: the instruction's other rows are zeros
    // times -0, which leave every sum as it is, also -0
    const int rest = int(rows & 3), at = int((rows & ~int64_t(3)) % kC);
    if (rest) {
#pragma unroll
        for (int i = 0; i < kT; ++i)
            if (tI[i] >= 0) {
                const double* xa = Xs + size_t(tI[i] * 16 + m) * kLd + kk + at;
                const double* xb = Xs + size_t(tJ[i] * 16 + m) * kLd + kk + at;
                acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(*xa, kk < rest ? *xb : -0.0, acc[i],
                                                              0, 0, 0);
            }
    }
    double* A = a + size_t(run) * P * P;
#pragma unroll
    for (int i = 0; i < kT; ++i) {
        if (tI[i] >= 0) {
            const int col = tJ[i] * 16 + m;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = tI[i] * 16 + 4 * e + kk;
                if (row < P && col < P) {
                    A[size_t(row) * P + col] = acc[i][e];
                    A[size_t(col) * P + row] = acc[i][e];
                }
            }
        } else if (tI[i] == -2) {
            const int p = tJ[i] * 64 + lane;
            if (p < P) g[size_t(run) * P + p] = gacc[i];
        }
    }
}

// More than 127 variables (their columns do not fit the LDS stages above): 64 x 64 output tile per
// workgroup over the upper tiles of the (P+1) x (P+1) matrix, 256 threads each holding a 4 x 4 block
// of elements: 16 independent FMA chains per thread (the chains' latency is what bounds a Gram of
// long columns). Rows are staged through LDS 32 at a time, row-major
// [row][column], so a thread reads its 4 consecutive columns as two 16-byte words. Each element is
// one FMA chain over the rows in ascending order starting from 0 (gram_dot,
// normal_equations.hpp:19), products of the stored J values: bitwise the host definition.
__global__ __launch_bounds__(256) void gram_wide_kernel(const double* J, const double* r0, int runs, int P,
                                                   int64_t rows, double* a, double* g,
                                                   const int32_t* live) {
    constexpr int kT = 64, kC = 32, kLd = kT + 2; // row stride in doubles (16-byte aligned rows)
    __shared__ __align__(16) double As[kC][kLd];
    __shared__ __align__(16) double Bs[kC][kLd];
    const int T = (P + 1 + kT - 1) / kT;
    const int tiles = T * (T + 1) / 2;
    const int run = blockIdx.x / tiles;
    if (live && run >= *live) return;
    int tile = blockIdx.x - run * tiles;
    int tq = 0;
    while (tile >= T - tq) {
        tile -= T - tq;
        ++tq;
    }
    const int tp = tq + tile; // column tile >= row tile
    const bool diag = tp == tq;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const double* Jr = J + size_t(run) * P * rows;
    const double* rr = r0 + size_t(run) * rows;
    auto column = [&](int col, int64_t row) {
        return col < P ? Jr[size_t(col) * rows + row] : col == P ? rr[row] : 0.0;
    };
    double acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.0;
    const double(*Bsrc)[kLd] = diag ? As : Bs;
    for (int64_t base = 0; base < rows; base += kC) {
        const int n = int(rows - base < kC ? rows - base : kC);
        for (int e = threadIdx.x; e < kT * kC; e += 256) {
            const int c = e / kC, rw = e - c * kC;
            const int64_t row = base + rw;
            As[rw][c] = rw < n ? column(tq * kT + c, row) : 0.0;
            if (!diag) Bs[rw][c] = rw < n ? column(tp * kT + c, row) : 0.0;
        }
        __syncthreads();
        for (int rw = 0; rw < n; ++rw) {
            const double2 a01 = *reinterpret_cast<const double2*>(&As[rw][ty * 4]);
            const double2 a23 = *reinterpret_cast<const double2*>(&As[rw][ty * 4 + 2]);
            const double2 b01 = *reinterpret_cast<const double2*>(&Bsrc[rw][tx * 4]);
            const double2 b23 = *reinterpret_cast<const double2*>(&Bsrc[rw][tx * 4 + 2]);
            const double av[4] = {a01.x, a01.y, a23.x, a23.y};
            const double bv[4] = {b01.x, b01.y, b23.x, b23.y};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __fma_rn(av[i], bv[j], acc[i][j]);
        }
        __syncthreads();
    }
    double* A = a + size_t(run) * P * P;
    double* gr = g + size_t(run) * P;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int p = tq * kT + ty * 4 + i;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int q = tp * kT + tx * 4 + j;
            const double v = acc[i][j];
            if (p < P && q < P) {
                A[size_t(p) * P + q] = v;
                A[size_t(q) * P + p] = v;
            } else if (p < P && q == P) {
                gr[p] = v;
            } else if (p == P && q < P) {
                gr[q] = v;
            }
        }
    }
}

// ---- helpers ---------------------------------------------------------------------------------

void check_hip(hipError_t e, const char* what) {
    if (e != hipSuccess)
        throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// The raw device entry points trace ray rows only; constraint rows are the host layer's
// (mko_engine_*), which evaluates them next to the traces.
void no_rows(const mko_residual_settings& s) {
    if (s.extra && s.extra->count > 0)
        throw std::invalid_argument("constraint rows are evaluated by the mko_engine_* entry points");
}

TraceParams make_params(const mko_batch& b, const mko_residual_settings& s) {
    if (b.surfaces < 2 || b.surfaces > MKO_MAX_SURFACES)
        throw std::invalid_argument("surfaces outside [2, 64]");
    if (b.fields < 1 || b.fields > kMaxFields)
        throw std::invalid_argument("fields outside [1, 32]");
    if (b.wavelengths < 1 || b.wavelengths > kMaxWavelengths)
        throw std::invalid_argument("wavelengths outside [1, 32]");
    if (s.rings < 1 || s.rings > MKO_MAX_RINGS) throw std::invalid_argument("rings outside [1, 16]");
    if (s.spokes < 1) throw std::invalid_argument("spokes < 1");
    if (s.failure != MKO_FAILURE_SOFT && s.failure != MKO_FAILURE_HARD)
        throw std::invalid_argument("unknown failure mode");
    if (!(s.fail_weight >= 0.0) || !std::isfinite(s.fail_weight))
        throw std::invalid_argument("fail_weight must be finite and >= 0");
    if (s.precision != MKO_PRECISION_FP64 && s.precision != MKO_PRECISION_DF64)
        throw std::invalid_argument("trace precision must be MKO_PRECISION_FP64 or MKO_PRECISION_DF64");
    if (b.reference_sphere != MKO_REF_LAST_SURFACE && b.reference_curvature == nullptr)
        throw std::invalid_argument("image reference sphere needs reference_curvature");
    if (b.source == MKO_SOURCE_POINT && b.fields != 1)
        throw std::invalid_argument("point source needs exactly one field");
    TraceParams P{};
    P.curvature = b.curvature;
    P.thickness = b.thickness;
    P.index = b.index;
    P.pupil_radius = b.pupil_radius;
    P.field_angle = b.field_angle;
    P.field_target = b.field_target;
    P.reference_curvature = b.reference_curvature;
    P.V = b.variants;
    P.S = b.surfaces;
    P.L = b.wavelengths;
    P.F = b.fields;
    P.T = b.fields * b.wavelengths;
    P.source = b.source;
    P.ref_kind = b.reference_sphere;
    P.rings = s.rings;
    P.spokes = s.spokes;
    P.soft = s.failure == MKO_FAILURE_SOFT;
    P.precision = s.precision;
    P.fail_weight = s.fail_weight;
    P.lambda_ref_nm = b.reference_wavelength_nm;
    for (int i = 0; i < 3; ++i) P.src_pt[i] = b.source_point[i];
    P.src_na = b.source_na;
    P.sphere_mask = 0;
    for (int i = 0; i < b.surfaces; ++i) {
        if (b.type[i] > MKO_SURFACE_SPHERE)
            throw std::invalid_argument("unsupported surface type (ghost plates are not supported)");
        if (b.type[i] == MKO_SURFACE_SPHERE) P.sphere_mask |= 1ull << i;
    }
    int64_t rays = 0;
    int nmax = 0;
    for (int f = 0; f < b.fields; ++f) {
        if (b.pupil_mode[f] > MKO_PUPIL_AXIS) throw std::invalid_argument("unknown pupil mode");
        P.pupil_mode[f] = b.pupil_mode[f];
        P.field_weight[f] = b.field_weight[f];
        const int n = s.rings * (b.pupil_mode[f] == MKO_PUPIL_AXIS ? 1 : s.spokes);
        nmax = std::max(nmax, n);
        rays += int64_t(b.wavelengths) * n;
    }
    if (nmax > kBlock * kMaxRaysPerLane)
        throw std::invalid_argument("more than 2048 pupil samples per tuple");
    for (int l = 0; l < b.wavelengths; ++l) P.wavelength_weight[l] = b.wavelength_weight[l];
    const int off = s.rings * (s.rings - 1) / 2;
    for (int i = 0; i < s.rings; ++i) {
        P.gl_u[i] = mko_gl_u[off + i];
        P.gl_w[i] = mko_gl_w[off + i];
    }
    P.rays = rays;
    P.trace_rows = P.soft ? 2 * rays : rays;
    P.stride = P.trace_rows;
    return P;
}

// Launch shapes of the calling thread (set by the host layer for its calls; the device-layer
// entry points run with the defaults).
thread_local mko_internal::Tuning g_tuning{};

// Segment of a tuple pack for this launch (0: one tuple per workgroup): tuples of at most 128
// rays (FP64 traces without extrema) share a workgroup in segments of 32, 64 or 128 lanes, the
// smallest that holds the largest tuple, or the tuning's pack_rays where the tuples fit it
// (pack_rays 256 turns packing off).
int pack_segment(const TraceParams& P, bool packable) {
    if (!packable || P.precision != MKO_PRECISION_FP64) return 0;
    int nmax = 0;
    for (int f = 0; f < P.F; ++f)
        nmax = std::max(nmax, P.rings * (P.pupil_mode[f] == MKO_PUPIL_AXIS ? 1 : P.spokes));
    const int want = g_tuning.pack_rays;
    if (want >= kBlock || nmax > 128 || P.T < 2) return 0;
    int seg = nmax <= 32 ? 32 : nmax <= 64 ? 64 : 128;
    if (want == 32 || want == 64 || want == 128) seg = std::max(seg, want);
    return seg;
}

int largest_tuple(const TraceParams& P) {
    int nmax = 0;
    for (int f = 0; f < P.F; ++f)
        nmax = std::max(nmax, P.rings * (P.pupil_mode[f] == MKO_PUPIL_AXIS ? 1 : P.spokes));
    return nmax;
}

int rays_per_lane(const TraceParams& P) {
    const int r = (largest_tuple(P) + kBlock - 1) / kBlock;
    return r <= 1 ? 1 : r <= 2 ? 2 : r <= 4 ? 4 : 8;
}

template <int kMode, bool kSoft, class R, bool kStates, bool kExt>
void launch_trace_rpl(int rpl, const TraceParams& P, double* res, double* opd, uint8_t* st,
                      double* part, int* pf, int* ph, const mko_internal::RayStates& states,
                      double* ext, hipStream_t stream) {
    const dim3 grid(unsigned(P.V) * unsigned(P.T));
#define MKO_LAUNCH(RPL)                                                                          \
    hipLaunchKernelGGL((trace_kernel<kMode, kSoft, RPL, R, kStates, kExt>), grid, dim3(kBlock),   \
                       0, stream, P, res, opd, st, part, pf, ph, states, ext)
    switch (rpl) {
    case 1: MKO_LAUNCH(1); break;
    case 2: MKO_LAUNCH(2); break;
    case 4: MKO_LAUNCH(4); break;
    default: MKO_LAUNCH(8); break;
    }
#undef MKO_LAUNCH
}

template <int kMode, bool kSoft, class R>
void launch_trace_ext(int rpl, const TraceParams& P, double* res, double* opd, uint8_t* st,
                      double* part, int* pf, int* ph, double* ext, hipStream_t stream) {
    const mko_internal::RayStates none{};
    if (ext) launch_trace_rpl<kMode, kSoft, R, false, true>(rpl, P, res, opd, st, part, pf, ph, none, ext, stream);
    else launch_trace_rpl<kMode, kSoft, R, false, false>(rpl, P, res, opd, st, part, pf, ph, none, nullptr, stream);
}

template <class R>
void launch_trace_r(int mode, int rpl, const TraceParams& P, double* res, double* opd, uint8_t* st,
                    double* part, int* pf, int* ph, double* ext, hipStream_t stream) {
    if (mode == 0) {
        if (P.soft) launch_trace_ext<0, true, R>(rpl, P, res, opd, st, part, pf, ph, ext, stream);
        else launch_trace_ext<0, false, R>(rpl, P, res, opd, st, part, pf, ph, ext, stream);
    } else {
        if (P.soft) launch_trace_ext<1, true, R>(rpl, P, res, opd, st, part, pf, ph, ext, stream);
        else launch_trace_ext<1, false, R>(rpl, P, res, opd, st, part, pf, ph, ext, stream);
    }
}

// RESIDUALS (mode 0) or MERIT partials (mode 1); ext: extrema partials [V*T][S][2] or NULL;
// states: the LM MERIT's final ray states (mode 1, FP64 trace; stored for the rays that end
// with status Ok) or NULL.
void launch_trace(int mode, const TraceParams& P, double* res, double* opd, uint8_t* st,
                  double* part, int* pf, int* ph, double* ext, hipStream_t stream,
                  const mko_internal::RayStates* states = nullptr) {
    if (int64_t(P.V) * P.T > 0x7fffffffLL) throw std::invalid_argument("batch too large for one launch");
    const int rpl = rays_per_lane(P);
    const int seg = pack_segment(P, ext == nullptr);
    if (seg > 0) {
        if (states && (mode != 1 || P.precision != MKO_PRECISION_FP64))
            throw std::invalid_argument("ray states need the MERIT trace and FP64");
        const int tpb = kBlock / seg;
        const dim3 grid(unsigned(P.V) * unsigned((P.T + tpb - 1) / tpb));
        const size_t lds = size_t(tpb) * size_t(P.S + 1) * sizeof(Step);
        const mko_internal::RayStates none{};
        const mko_internal::RayStates& rs = states ? *states : none;
#define MKO_PACK(M, SOFT, ST)                                                                      \
    hipLaunchKernelGGL((trace_pack_kernel<M, SOFT, ST>), grid, dim3(kBlock), lds, stream, P, seg,   \
                       res, opd, st, part, pf, ph, rs)
        if (states) {
            if (P.soft) MKO_PACK(1, true, true);
            else MKO_PACK(1, false, true);
        } else if (mode == 0) {
            if (P.soft) MKO_PACK(0, true, false);
            else MKO_PACK(0, false, false);
        } else {
            if (P.soft) MKO_PACK(1, true, false);
            else MKO_PACK(1, false, false);
        }
#undef MKO_PACK
        check_hip(hipGetLastError(), "trace pack kernel launch");
        return;
    }
    if (states) {
        if (mode != 1 || P.precision != MKO_PRECISION_FP64)
            throw std::invalid_argument("ray states need the MERIT trace and FP64");
        if (P.soft) {
            if (ext) launch_trace_rpl<1, true, double, true, true>(rpl, P, res, opd, st, part, pf, ph, *states, ext, stream);
            else launch_trace_rpl<1, true, double, true, false>(rpl, P, res, opd, st, part, pf, ph, *states, nullptr, stream);
        } else if (ext) {
            launch_trace_rpl<1, false, double, true, true>(rpl, P, res, opd, st, part, pf, ph, *states, ext, stream);
        } else {
            launch_trace_rpl<1, false, double, true, false>(rpl, P, res, opd, st, part, pf, ph, *states, nullptr, stream);
        }
    } else if (P.precision == MKO_PRECISION_DF64) {
        launch_trace_r<mkod::df64>(mode, rpl, P, res, opd, st, part, pf, ph, ext, stream);
    } else {
        launch_trace_r<double>(mode, rpl, P, res, opd, st, part, pf, ph, ext, stream);
    }
    check_hip(hipGetLastError(), "trace kernel launch");
}

// buchdahl_omega (dispersion.hpp:18-89) of nm / 1000 on the host, contract off
double buchdahl_omega_host(double lambda_nm, bool& ok) {
#pragma clang fp contract(off)
    const double um = lambda_nm / 1000.0;
    const double den = 1.0 + 2.5 * (um - 0.546074);
    ok = ok && den > 0.0;
    return (um - 0.546074) / den;
}

OmegaTable omega_table(const mko_batch& b) {
    OmegaTable t{};
    t.valid = 0;
    if (!b.wavelength_nm || b.wavelengths > kMaxWavelengths) return t;
    bool ok = true;
    for (int l = 0; l < b.wavelengths; ++l) t.w[l] = buchdahl_omega_host(b.wavelength_nm[l], ok);
    t.w[b.wavelengths] = buchdahl_omega_host(b.reference_wavelength_nm, ok);
    t.valid = ok ? 1 : 0;
    return t;
}

// Column map of the variables (AdjointParameters, src/optim/adjoint_jacobian.cpp:79-127); glass
// variables need the batch's wavelengths (host) for their slopes, and `allow_glass`.
static_assert(sizeof(TraceParams) + sizeof(ParamMap) < 3584, "kernel arguments within 4 KB");
ParamMap make_map(const mko_variables& vars, const mko_batch& batch, bool allow_glass) {
    const int S = batch.surfaces;
    ParamMap m{};
    m.P = vars.count;
    if (vars.count < 1 || vars.count > 127) throw std::invalid_argument("1 ... 127 variables");
    for (int s = 0; s < MKO_MAX_SURFACES; ++s) {
        m.curv_col[s] = -1;
        m.thick_col[s] = -1;
        for (int c = 0; c < 3; ++c) m.glass_col[s][c] = -1;
    }
    for (int k = 0; k < vars.count; ++k) {
        const int s = vars.batch_surface[k];
        if (s < 0 || s >= S) throw std::invalid_argument("variable surface out of range");
        if (vars.type[k] < MKO_VAR_CURVATURE || vars.type[k] > MKO_VAR_GLASS)
            throw std::invalid_argument("unsupported variable type");
        if (vars.type[k] == MKO_VAR_GLASS) {
            if (!allow_glass)
                throw std::invalid_argument("glass variables need the FP64 adjoint (not the fused "
                                            "normal equations)");
            if (!vars.component || vars.component[k] < 0 || vars.component[k] > 2)
                throw std::invalid_argument("glass variables need components 0 ... 2");
            int32_t& slot = m.glass_col[s][vars.component[k]];
            if (slot >= 0) throw std::invalid_argument("parameter belongs to two variables");
            slot = k;
            m.glass = 1;
        } else {
            int32_t& slot = vars.type[k] == MKO_VAR_CURVATURE ? m.curv_col[s] : m.thick_col[s];
            if (slot >= 0) throw std::invalid_argument("parameter belongs to two variables");
            slot = k;
        }
    }
    for (int s = 0; s < S; ++s) {
        const auto unswept = [&](int col) {
            if (col >= 0) m.unswept[col >> 6] |= uint64_t(1) << (col & 63);
        };
        if (s == 0 || batch.type[s] != MKO_SURFACE_SPHERE) unswept(m.curv_col[s]);
        if (s == 0)
            for (int c = 0; c < 3; ++c) unswept(m.glass_col[s][c]);
    }
    if (m.glass) {
        const OmegaTable t = omega_table(batch);
        if (!t.valid)
            throw std::invalid_argument("glass variables need wavelength_nm with a defined Buchdahl "
                                        "coordinate (lambda > 146.074 nm)");
        for (int l = 0; l < batch.wavelengths; ++l) m.omega[l] = t.w[l];
    }
    return m;
}

// Lanes of a workgroup for tuples of at most nmax rays: as many waves as they fill, up to 4.
int tuple_lanes(int nmax) { return std::min(kBlock, 64 * ((nmax + 63) / 64)); }

template <bool kSoft, bool kGlass>
void launch_adjoint(const TraceParams& P, const ParamMap& m, double* J, double* r0, uint8_t* st,
                    hipStream_t stream) {
    const int nmax = largest_tuple(P);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(unsigned(P.V) * unsigned(P.T)), dim3(tuple_lanes(nmax)),
                           size_t(P.S + 1) * sizeof(Step) + size_t(nmax) * sizeof(double2), stream,
                           P, m, J, r0, st);
    };
    switch (rays_per_lane(P)) {
    case 1: launch(adjoint_kernel<kSoft, kGlass, 1>); break;
    case 2: launch(adjoint_kernel<kSoft, kGlass, 2>); break;
    case 4: launch(adjoint_kernel<kSoft, kGlass, 4>); break;
    default: launch(adjoint_kernel<kSoft, kGlass, 8>); break;
    }
}

template <bool kGlass>
void launch_vjp(const TraceParams& P, const ParamMap& m, const double* grad, int64_t gstride,
                double* part, hipStream_t stream) {
    const int nmax = largest_tuple(P), lanes = tuple_lanes(nmax);
    const dim3 grid(unsigned(P.V) * unsigned(P.T));
    const size_t table = size_t(P.S + 1) * sizeof(Step);
    if (P.soft) {
        hipLaunchKernelGGL(vjp_soft_kernel<kGlass>, grid, dim3(64),
                           table + size_t(m.P) * 64 * sizeof(double), stream, P, m, grad, gstride,
                           part);
        return;
    }
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(lanes),
                           table + size_t(lanes / 64) * m.P * 16 * sizeof(double), stream, P, m,
                           grad, gstride, part);
    };
    switch (rays_per_lane(P)) {
    case 1: launch(vjp_kernel<kGlass, 1>); break;
    case 2: launch(vjp_kernel<kGlass, 2>); break;
    case 4: launch(vjp_kernel<kGlass, 4>); break;
    default: launch(vjp_kernel<kGlass, 8>); break;
    }
}

#define MKO_TRY(...)                                                                               \
    try {                                                                                          \
        __VA_ARGS__;                                                                               \
        return 0;                                                                                  \
    } catch (const std::invalid_argument& e) {                                                     \
        mko_detail::last_error = e.what();                                                                        \
        return MKO_ERR_INVALID;                                                                    \
    } catch (const std::exception& e) {                                                            \
        mko_detail::last_error = e.what();                                                                        \
        return MKO_ERR_DEVICE;                                                                     \
    }

// Check kernel of the df64 arithmetic (df64_check_kernel, src/cuda/df64_check.cu:17): one
// operation per element, for the bitwise comparison with the host restatement.
__global__ void df64_ops_kernel(int op, int64_t n, const float* a, const float* b, float* out) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    using mkod::df64;
    const df64 x{a[2 * i], a[2 * i + 1]};
    const df64 y = op == 5 ? df64{0.0f, 0.0f} : df64{b[2 * i], b[2 * i + 1]};
    df64 z;
    switch (op) {
    case 0: z = x + y; break;
    case 1: z = x - y; break;
    case 2: z = x * y; break;
    case 3: z = mkod::mul_fp(x, y.hi); break;
    case 4: z = x / y; break;
    default: z = mkod::sqrt(x); break;
    }
    out[2 * i] = z.hi;
    out[2 * i + 1] = z.lo;
}

} // namespace

namespace mko_internal {

int point_batch(const mko_batch* templ, const int32_t* template_index, int template_per_run,
                int runs, int per_run, const mko_variables* vars_device, const double* x0,
                const double* plus, const double* minus, double* curvature, double* thickness,
                double* index, double* pupil_radius, double* field_angle, double* field_target,
                double* reference_curvature, double* paraxial_index, double* buchdahl,
                void* stream, const int32_t* live) {
    MKO_TRY({
        if (runs <= 0) return 0;
        const ConstBatchPtrs src{templ->curvature, templ->thickness, templ->index,
                                 templ->pupil_radius, templ->field_angle, templ->field_target,
                                 templ->reference_curvature, templ->paraxial_index,
                                 templ->buchdahl};
        const BatchPtrs dst{curvature, thickness, index, pupil_radius, field_angle, field_target,
                            reference_curvature, paraxial_index, buchdahl};
        const OmegaTable om = omega_table(*templ);
        hipLaunchKernelGGL(point_batch_kernel, dim3(unsigned(runs) * unsigned(per_run)), dim3(64),
                           0, static_cast<hipStream_t>(stream), src, dst, runs, per_run,
                           template_index, template_per_run, templ->surfaces, templ->wavelengths,
                           templ->fields, vars_device->count, vars_device->type,
                           vars_device->batch_surface, vars_device->component, x0, plus, minus,
                           live, om);
        check_hip(hipGetLastError(), "point batch launch");
    })
}

template <int kNW, int kPMax, bool kStates, bool kGlass>
void launch_fused(const TraceParams& P, const ParamMap& m, float* partC, double* partST,
                  TupleNormal* partT, const RayStates& states, hipStream_t s) {
    const size_t tuples = size_t(P.V) * P.T;
    hipLaunchKernelGGL((adjoint_normal_kernel<kNW, kPMax, kStates, kGlass>), dim3(unsigned(tuples)),
                       dim3(64 * kNW), fused_lds_bytes<kNW>(m.P, P.S), s, P, m, partC, partST, partT,
                       states);
}

template <bool kStates, bool kGlass>
void launch_fused_waves(int waves, const TraceParams& P, const ParamMap& m, float* partC,
                        double* partST, TupleNormal* partT, const RayStates& states,
                        hipStream_t s) {
    const bool wide = m.P > 64;
#define MKO_FUSED(NW, PM) launch_fused<NW, PM, kStates, kGlass>(P, m, partC, partST, partT, states, s)
    switch (waves) {
    case 1: wide ? MKO_FUSED(1, 96) : MKO_FUSED(1, 64); break;
    case 2: wide ? MKO_FUSED(2, 96) : MKO_FUSED(2, 64); break;
    default: wide ? MKO_FUSED(4, 96) : MKO_FUSED(4, 64); break;
    }
#undef MKO_FUSED
}

// Waves per workgroup of the fused kernel: 1 for tuples of at most 64 rays (one chunk, tiles
// formed one after another), 2 up to 128, else 4 (chunks of 256 rays); `requested` (1, 2, 4)
// overrides where it fits (1 needs tuples of at most 64 rays).
int fused_waves(const TraceParams& P, int requested) {
    int nmax = 0;
    for (int f = 0; f < P.F; ++f)
        nmax = std::max(nmax, P.rings * (P.pupil_mode[f] == MKO_PUPIL_AXIS ? 1 : P.spokes));
    if (requested == 2 || requested == 4) return requested;
    if (requested == 1 && nmax <= 64) return 1;
    return nmax <= 64 ? 1 : nmax <= 128 ? 2 : 4;
}

int adjoint_normal_states(const mko_batch* batch, const mko_residual_settings* settings,
                          const mko_variables* vars, double* a, double* g, void* workspace,
                          size_t workspace_bytes, const RayStates& states, void* stream,
                          const int32_t* live, int waves) {
    MKO_TRY({
        TraceParams P = make_params(*batch, *settings);
        P.live = live;
        // glass variables (index adjoints in the reverse sweep) on the LM path's stored states
        const ParamMap m = make_map(*vars, *batch, states.data != nullptr);
        if (P.soft) throw std::invalid_argument("fused adjoint normal equations need hard failure mode");
        if (m.P > kMaxVariablesFused)
            throw std::invalid_argument("fused adjoint normal equations: at most 96 variables");
        if (P.V == 0) return 0;
        if (int64_t(P.V) * P.T > 0x7fffffffLL) throw std::invalid_argument("batch too large");
        const size_t need = mko_adjoint_normal_workspace(P.V, P.F, P.L, m.P);
        if (workspace_bytes < need) throw std::invalid_argument("workspace too small");
        const size_t tuples = size_t(P.V) * P.T;
        auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
        char* w = static_cast<char*>(workspace);
        float* partC = reinterpret_cast<float*>(w);
        double* partST = reinterpret_cast<double*>(w + up(tuples * m.P * m.P * sizeof(float)));
        TupleNormal* partT = reinterpret_cast<TupleNormal*>(
            w + up(tuples * m.P * m.P * sizeof(float)) +
            up(tuples * 2 * m.P * sizeof(double)));
        const hipStream_t s = static_cast<hipStream_t>(stream);
        const int nw = fused_waves(P, waves ? waves : g_tuning.fused_waves);
        if (states.data) {
            if (P.precision != MKO_PRECISION_FP64)
                throw std::invalid_argument("stored ray states need the FP64 trace");
            if (states.rays != P.rays) throw std::invalid_argument("ray states of another layout");
            if (m.glass) launch_fused_waves<true, true>(nw, P, m, partC, partST, partT, states, s);
            else launch_fused_waves<true, false>(nw, P, m, partC, partST, partT, states, s);
        } else {
            launch_fused_waves<false, false>(nw, P, m, partC, partST, partT, states, s);
        }
        check_hip(hipGetLastError(), "adjoint normal launch");
        const int nu = m.P * (m.P + 1) / 2;
        const size_t lds = size_t(kFinalizeChunk) * 2 * m.P * sizeof(double);
        const auto finalize = [&](auto kernel, int entries) {
            const int parts = (nu + 256 * entries - 1) / (256 * entries);
            hipLaunchKernelGGL(kernel, dim3(unsigned(P.V) * unsigned(parts)), dim3(256), lds, s,
                               P.T, m.P, parts, partC, partST, partT, a, g, live);
        };
        if (finalize_entries(m.P, P.V) == 1) finalize(adjoint_normal_finalize_kernel<1>, 1);
        else finalize(adjoint_normal_finalize_kernel<5>, 5);
        check_hip(hipGetLastError(), "adjoint normal finalize launch");
    })
}

int merit_states(const mko_batch* batch, const mko_residual_settings* settings, double* merit,
                 int64_t* failed, int64_t* hard_failed, double* partial, int* partial_counts,
                 const RayStates& states, void* stream, const int32_t* live) {
    MKO_TRY({
        TraceParams P = make_params(*batch, *settings);
        P.live = live;
        if (P.precision != MKO_PRECISION_FP64)
            throw std::invalid_argument("ray states need the FP64 trace");
        if (states.rays != P.rays) throw std::invalid_argument("ray states of another layout");
        if (P.V == 0) return 0;
        const hipStream_t s = static_cast<hipStream_t>(stream);
        int* pf = partial_counts;
        int* ph = partial_counts + size_t(P.V) * P.T;
        launch_trace(1, P, nullptr, nullptr, nullptr, partial, pf, ph, nullptr, s, &states);
        hipLaunchKernelGGL(merit_finalize_kernel, dim3((P.V + 3) / 4), dim3(256), 0, s, P.V,
                           P.T, partial, pf, ph, nullptr, nullptr, merit, failed, hard_failed, live);
        check_hip(hipGetLastError(), "merit finalize launch");
    })
}

int trace_extrema(const mko_batch* batch, const mko_residual_settings* settings, int mode,
                  double* residuals, int64_t stride, double* opd, uint8_t* status,
                  double* partial, int* partial_counts, const RayStates* states,
                  double* ext_partial, double* extrema, uint64_t surfaces, void* stream) {
    MKO_TRY({
        TraceParams P = make_params(*batch, *settings);
        P.ext_mask = surfaces;
        if (mode == 0) {
            if (stride < P.trace_rows) throw std::invalid_argument("stride smaller than trace rows");
            P.stride = stride;
        }
        if (states && states->rays != P.rays) throw std::invalid_argument("ray states of another layout");
        if (P.V == 0) return 0;
        const hipStream_t s = static_cast<hipStream_t>(stream);
        int* pf = mode == 1 ? partial_counts : nullptr;
        int* ph = mode == 1 ? partial_counts + size_t(P.V) * P.T : nullptr;
        launch_trace(mode, P, residuals, opd, status, partial, pf, ph, ext_partial, s, states);
        if (ext_partial) {
            const int64_t n = int64_t(P.V) * P.S;
            hipLaunchKernelGGL(extrema_finalize_kernel, dim3(unsigned((n + 255) / 256)), dim3(256),
                               0, s, P.V, P.T, P.S, ext_partial, extrema);
            check_hip(hipGetLastError(), "extrema finalize launch");
        }
    })
}

int candidate_extrema(const mko_batch* base, const mko_batch* fd,
                      const mko_residual_settings* settings, int per_run, uint64_t hmask,
                      uint64_t cmask, double delta, const double* ex0, uint8_t* flags,
                      int* tcount, int* others, int* tstart, int* list, int cap, int* overflow,
                      double* ext, void* stream) {
    MKO_TRY({
        TraceParams Pb = make_params(*base, *settings);
        TraceParams Pf = make_params(*fd, *settings);
        if (settings->precision != MKO_PRECISION_FP64)
            throw std::invalid_argument("candidate rays trace in FP64");
        if (Pf.V != Pb.V * per_run || Pf.T != Pb.T || Pf.rays != Pb.rays)
            throw std::invalid_argument("candidate rays: batch shapes differ");
        if (Pb.V == 0) return 0;
        Pb.ext_mask = Pf.ext_mask = hmask | cmask;
        const hipStream_t s = static_cast<hipStream_t>(stream);
        check_hip(hipMemsetAsync(others, 0, size_t(Pb.V) * sizeof(int), s), "memset");
        const dim3 gb(unsigned(Pb.V) * unsigned(Pb.T));
        if (Pb.soft)
            hipLaunchKernelGGL(ray_candidates_kernel<true>, gb, dim3(kBlock), 0, s, Pb, hmask,
                               cmask, delta, ex0, flags, tcount, others);
        else
            hipLaunchKernelGGL(ray_candidates_kernel<false>, gb, dim3(kBlock), 0, s, Pb, hmask,
                               cmask, delta, ex0, flags, tcount, others);
        check_hip(hipGetLastError(), "ray candidates launch");
        hipLaunchKernelGGL(candidate_list_kernel, dim3(unsigned(Pb.V)), dim3(1024), 0, s, Pb.T,
                           Pb.rays, cap, flags, tcount, tstart, list, overflow);
        check_hip(hipGetLastError(), "candidate list launch");
        if (Pf.soft)
            hipLaunchKernelGGL(candidate_extrema_kernel<true>, dim3(unsigned(Pf.V)), dim3(64), 0,
                               s, Pf, per_run, cap, tstart, list, ext);
        else
            hipLaunchKernelGGL(candidate_extrema_kernel<false>, dim3(unsigned(Pf.V)), dim3(64), 0,
                               s, Pf, per_run, cap, tstart, list, ext);
        check_hip(hipGetLastError(), "candidate extrema launch");
    })
}

int extrema_check(int runs, int per_run, int S, uint64_t hmask, uint64_t cmask, double delta,
                  const double* ex, const double* ex0, const int* others, const int* overflow,
                  double K, int* flag, void* stream) {
    MKO_TRY({
        if (runs <= 0) return 0;
        hipLaunchKernelGGL(extrema_check_kernel, dim3((runs + 127) / 128), dim3(128), 0,
                           static_cast<hipStream_t>(stream), runs, per_run, S, hmask, cmask,
                           delta, ex, ex0, others, overflow, K, flag);
        check_hip(hipGetLastError(), "extrema check launch");
    })
}

int prefilter_stats(const mko_batch* batch, const mko_residual_settings* settings, double boundary,
                    void* workspace, double* merit, double* optical, int64_t* failed,
                    int64_t* uncertain_ok, int64_t* uncertain_failed, void* stream) {
    MKO_TRY({
        TraceParams P = make_params(*batch, *settings);
        if (!(boundary >= 0.0) || !std::isfinite(boundary))
            throw std::invalid_argument("prefilter boundary margin must be finite and >= 0");
        if (P.V == 0) return 0;
        if (int64_t(P.V) * P.T > 0x7fffffffLL) throw std::invalid_argument("batch too large");
        const size_t tuples = size_t(P.V) * P.T;
        char* w = static_cast<char*>(workspace);
        double* pm = reinterpret_cast<double*>(w);
        float* pl = reinterpret_cast<float*>(w + tuples * 8);
        int* pc = reinterpret_cast<int*>(w + tuples * 12);
        const hipStream_t s = static_cast<hipStream_t>(stream);
        const float eta = float(boundary);
        const PrefilterPlan p = prefilter_plan(P.V, P.T, P.S, P.rings, largest_tuple(P));
        const auto kernel = p.q == kBlock ? prefilter_kernel<true> : prefilter_kernel<false>;
        hipLaunchKernelGGL(kernel, dim3(unsigned(p.groups) * unsigned(P.T)), dim3(kBlock), p.lds, s,
                           P, p.Q, p.q, eta, pm, pl, pc);
        check_hip(hipGetLastError(), "prefilter launch");
        hipLaunchKernelGGL(prefilter_finalize_kernel, dim3((P.V + 255) / 256), dim3(256), 0, s,
                           P.V, P.T, pm, pl, pc, merit, optical, failed, uncertain_ok,
                           uncertain_failed);
        check_hip(hipGetLastError(), "prefilter finalize launch");
    })
}

void set_thread_tuning(const Tuning& t) { g_tuning = t; }
Tuning thread_tuning() { return g_tuning; }

int merit_finalize(int V, int T, const double* partial, const int* partial_counts,
                   const double* extra, const double* traced, double* merit, int64_t* failed,
                   int64_t* hard_failed, void* stream) {
    MKO_TRY({
        if (V <= 0) return 0;
        hipLaunchKernelGGL(merit_finalize_kernel, dim3((V + 3) / 4), dim3(256), 0,
                           static_cast<hipStream_t>(stream), V, T, partial, partial_counts,
                           partial_counts + size_t(V) * T, extra, traced, merit, failed,
                           hard_failed, nullptr);
        check_hip(hipGetLastError(), "merit finalize launch");
    })
}

int constraint_rows(const mko_batch* batch, const mko_constraint* items, int count,
                    int need_paraxial, const double* extrema, double* rows, int64_t stride,
                    int64_t offset, void* stream, const double* glass_hull) {
    MKO_TRY({
        if (batch->variants <= 0 || count <= 0) return 0;
        if (glass_hull && !batch->buchdahl)
            throw std::invalid_argument("glass-hull rows need the batch's Buchdahl coefficients");
        uint64_t mask = 0;
        for (int i = 0; i < batch->surfaces; ++i)
            if (batch->type[i] == MKO_SURFACE_SPHERE) mask |= 1ull << i;
        if (need_paraxial && !batch->paraxial_index)
            throw std::invalid_argument("paraxial constraint rows need the batch's paraxial_index");
        hipLaunchKernelGGL(constraint_rows_kernel, dim3((batch->variants + 127) / 128), dim3(128),
                           0, static_cast<hipStream_t>(stream), batch->variants, batch->surfaces,
                           batch->fields, batch->curvature, batch->thickness,
                           batch->paraxial_index, batch->pupil_radius, batch->field_angle,
                           batch->field_target, mask, items, count, need_paraxial, extrema, rows,
                           stride, offset, batch->buchdahl, glass_hull);
        check_hip(hipGetLastError(), "constraint rows launch");
    })
}

int extra_normal(int runs, int P, int E, const double* Je, const double* re, double* a, double* g,
                 void* stream) {
    MKO_TRY({
        if (runs <= 0 || E <= 0) return 0;
        hipLaunchKernelGGL(extra_normal_kernel, dim3(unsigned(runs)), dim3(256), 0,
                           static_cast<hipStream_t>(stream), P, E, Je, re, a, g);
        check_hip(hipGetLastError(), "extra normal launch");
    })
}

int rows_merit(int V, const double* rows, int64_t stride, int64_t offset, int E, int Et,
               const double* extra, double* e_sum, double* t_sum, void* stream) {
    MKO_TRY({
        if (V <= 0) return 0;
        hipLaunchKernelGGL(rows_merit_kernel, dim3((V + 255) / 256), dim3(256), 0,
                           static_cast<hipStream_t>(stream), V, rows, stride, offset, E, Et,
                           extra, e_sum, t_sum);
        check_hip(hipGetLastError(), "rows merit launch");
    })
}

} // namespace mko_internal

namespace {

// Tuple partials of mko_merit_device_noalloc: [kScratchTuples] doubles (merit partials), then
// 2 x [kScratchTuples] ints (failed / hard-failed counts), 8 MiB in all. A static device array
// of the library: each GPU the library runs on holds its own copy until the process ends, and
// every call on that GPU shares it.
constexpr size_t kScratchTuples = size_t(1) << 19;
constexpr size_t kScratchBytes = kScratchTuples * (sizeof(double) + 2 * sizeof(int));
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Device address of `scratch` on the current device. In host code `scratch` names a host-side
// stand-in, never the device memory: the address comes from hipGetSymbolAddress, once per
// device with that device current, and is kept per device (each GPU's copy has its own).
unsigned char* scratch_address() {
    constexpr int kMaxDevices = 64;
    static std::mutex mutex;
    static unsigned char* address[kMaxDevices] = {};
    int device = 0;
    check_hip(hipGetDevice(&device), "hipGetDevice");
    if (device < 0 || device >= kMaxDevices) throw std::runtime_error("device ordinal out of range");
    std::lock_guard<std::mutex> lock(mutex);
    if (!address[device]) {
        void* ptr = nullptr;
        check_hip(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
        if (!ptr) throw std::runtime_error("hipGetSymbolAddress(scratch) returned no address");
        address[device] = static_cast<unsigned char*>(ptr);
    }
    return address[device];
}

} // namespace

extern "C" {

const char* mko_last_error(void) { return mko_detail::last_error.c_str(); }

int mko_residuals_device(const mko_batch* batch, const mko_residual_settings* settings,
                         double* residuals, int64_t stride, double* opd, uint8_t* status,
                         void* stream) {
    MKO_TRY({
        no_rows(*settings);
        TraceParams P = make_params(*batch, *settings);
        if (stride < P.trace_rows) throw std::invalid_argument("stride smaller than trace rows");
        P.stride = stride;
        if (P.V == 0) return 0;
        launch_trace(0, P, residuals, opd, status, nullptr, nullptr, nullptr, nullptr,
                     static_cast<hipStream_t>(stream));
    })
}

int mko_merit_device(const mko_batch* batch, const mko_residual_settings* settings,
                     const double* extra_merit, double* merit, int64_t* failed,
                     int64_t* hard_failed, double* partial, int* partial_counts, void* stream) {
    MKO_TRY({
        no_rows(*settings);
        const TraceParams P = make_params(*batch, *settings);
        if (P.V == 0) return 0;
        const hipStream_t s = static_cast<hipStream_t>(stream);
        int* pf = partial_counts;
        int* ph = partial_counts + size_t(P.V) * P.T;
        launch_trace(1, P, nullptr, nullptr, nullptr, partial, pf, ph, nullptr, s);
        hipLaunchKernelGGL(merit_finalize_kernel, dim3((P.V + 3) / 4), dim3(256), 0, s, P.V,
                           P.T, partial, pf, ph, extra_merit, nullptr, merit, failed, hard_failed,
                           nullptr);
        check_hip(hipGetLastError(), "merit finalize launch");
    })
}

int mko_merit_device_noalloc(const mko_batch* batch, const mko_residual_settings* settings,
                             const double* extra_merit, double* merit, int64_t* failed,
                             int64_t* hard_failed, void* stream) {
    MKO_TRY({
        no_rows(*settings);
        const TraceParams P = make_params(*batch, *settings);
        if (P.V == 0) return 0;
        const size_t tuples = size_t(P.V) * size_t(P.T);
        if (tuples > kScratchTuples)
            throw std::invalid_argument(
                "mko_merit_device_noalloc: " + std::to_string(tuples) +
                " (variant, field, wavelength) tuples, at most " + std::to_string(kScratchTuples) +
                " per call (split the batch, or use mko_merit_device with a workspace)");
        unsigned char* base = scratch_address();
        double* partial = reinterpret_cast<double*>(base);
        int* counts = reinterpret_cast<int*>(base + kScratchTuples * sizeof(double));
        const hipStream_t s = static_cast<hipStream_t>(stream);
        int* pf = counts;
        int* ph = counts + tuples;
        // every tuple's partial and counts are written by its trace block before the finalize
        // reads them, so the previous call's contents need no clearing
        launch_trace(1, P, nullptr, nullptr, nullptr, partial, pf, ph, nullptr, s);
        hipLaunchKernelGGL(merit_finalize_kernel, dim3((P.V + 3) / 4), dim3(256), 0, s, P.V,
                           P.T, partial, pf, ph, extra_merit, nullptr, merit, failed, hard_failed,
                           nullptr);
        check_hip(hipGetLastError(), "merit finalize launch");
    })
}

int mko_point_batch_device(const mko_batch* templ, int template_per_run, int runs, int per_run,
                           const mko_variables* vars_device, const double* x0,
                           const double* plus, const double* minus, double* curvature,
                           double* thickness, double* index, double* pupil_radius,
                           double* field_angle, double* field_target,
                           double* reference_curvature, double* paraxial_index, void* stream) {
    return mko_internal::point_batch(templ, nullptr, template_per_run, runs, per_run, vars_device,
                                     x0, plus, minus, curvature, thickness, index, pupil_radius,
                                     field_angle, field_target, reference_curvature,
                                     paraxial_index, nullptr, stream);
}

int mko_fd_difference_device(const double* fd_residuals, int64_t stride,
                             const uint8_t* fd_status, int64_t rays, int runs, int variables,
                             int64_t rows, const double* step_plus, const double* step_minus,
                             const uint8_t* stencil, double* jacobian, double* r0,
                             int64_t* status_changes, void* stream) {
    MKO_TRY({
        if (runs <= 0) return 0;
        hipLaunchKernelGGL(fd_difference_kernel, dim3(unsigned(runs) * unsigned(variables + 1)),
                           dim3(kBlock), 0, static_cast<hipStream_t>(stream), fd_residuals,
                           stride, fd_status, rays, runs, variables, rows, step_plus, step_minus,
                           stencil, jacobian, r0, status_changes, rows, int64_t(0));
        check_hip(hipGetLastError(), "fd difference launch");
    })
}

int mko_adjoint_jacobian_device(const mko_batch* batch, const mko_residual_settings* settings,
                                const mko_variables* vars, int precision, double* jacobian,
                                double* r0, uint8_t* status, void* stream) {
    MKO_TRY({
        no_rows(*settings);
        if (precision != MKO_PRECISION_FP64 && precision != MKO_PRECISION_MIXED)
            throw std::invalid_argument("unknown precision");
        return mko_internal::adjoint_jacobian(batch, settings, vars, jacobian, r0, status, 0,
                                              stream);
    })
}

} // extern "C"

namespace mko_internal {

int adjoint_jacobian(const mko_batch* batch, const mko_residual_settings* settings,
                     const mko_variables* vars, double* jacobian, double* r0, uint8_t* status,
                     int64_t stride, void* stream, const int32_t* live) {
    MKO_TRY({
        TraceParams P = make_params(*batch, *settings);
        P.live = live;
        if (stride > 0) {
            if (stride < P.trace_rows) throw std::invalid_argument("stride smaller than trace rows");
            P.stride = stride;
        }
        const int precision = MKO_PRECISION_FP64;
        const ParamMap m = make_map(*vars, *batch, true);
        if (P.V == 0) return 0;
        if (int64_t(P.V) * P.T > 0x7fffffffLL) throw std::invalid_argument("batch too large");
        const hipStream_t s = static_cast<hipStream_t>(stream);
        // MKO_PRECISION_MIXED computes the stored Jacobian in FP64 as well: on this hardware
        // the reduced-precision stage is the MFMA normal equations of the fused LM path.
        if (precision != MKO_PRECISION_FP64 && precision != MKO_PRECISION_MIXED)
            throw std::invalid_argument("unknown precision");
        double* Jd = static_cast<double*>(jacobian);
        if (P.soft) m.glass ? launch_adjoint<true, true>(P, m, Jd, r0, status, s)
                            : launch_adjoint<true, false>(P, m, Jd, r0, status, s);
        else m.glass ? launch_adjoint<false, true>(P, m, Jd, r0, status, s)
                     : launch_adjoint<false, false>(P, m, Jd, r0, status, s);
        check_hip(hipGetLastError(), "adjoint launch");
    })
}

int gram_chain(const double* jacobian, const double* r0, int runs, int variables, int64_t rows,
               double* a, double* g, void* stream, const int32_t* live) {
    MKO_TRY({
        if (runs <= 0 || variables == 0) return 0;
        if (variables < 0) throw std::invalid_argument("negative variable count");
        const hipStream_t s = static_cast<hipStream_t>(stream);
        if (variables > 127) {
            const int T = (variables + 1 + 63) / 64;
            hipLaunchKernelGGL(gram_wide_kernel, dim3(unsigned(runs) * unsigned(T * (T + 1) / 2)),
                               dim3(256), 0, s, jacobian, r0, runs, variables, rows, a, g, live);
            check_hip(hipGetLastError(), "gram launch");
            return 0;
        }
        const GramPlan plan = gram_plan(variables, runs);
        const int parts = plan.parts, upp = plan.upp;
        const auto launch = [&](auto kernel, int stage) {
            hipLaunchKernelGGL(kernel, dim3(unsigned(runs) * unsigned(parts)), dim3(512),
                               size_t(16 * plan.tg + 1) * size_t(stage + 2) * sizeof(double), s,
                               jacobian, r0, variables, rows, parts, upp, a, g, live);
        };
        // staged values per thread: (variables + 1) columns / 8 waves x (rows of a stage) / 64;
        // above 64 variables 64 rows at a time, so that the columns fit the LDS of two workgroups
        if (variables < 56) {
            if (upp <= 8) launch(gram_kernel<1, 128, 14>, 128);
            else launch(gram_kernel<2, 128, 14>, 128);
        } else if (variables <= 64) {
            if (upp <= 8) launch(gram_kernel<1, 128, 18>, 128);
            else launch(gram_kernel<2, 128, 18>, 128);
        } else {
            if (upp <= 8) launch(gram_kernel<1, 64, 16>, 64);
            else if (upp <= 24) launch(gram_kernel<3, 64, 16>, 64);
            else launch(gram_kernel<5, 64, 16>, 64);
        }
        check_hip(hipGetLastError(), "gram launch");
    })
}

// Dynamic LDS of fd_jacobian_kernel: the point's steps and two per difference.
static size_t fd_lds_bytes(int S, int P) { return size_t(S + 1 + 4 * P) * sizeof(Step); }

bool fd_direct(const mko_batch& batch, const mko_residual_settings& s, const mko_variables& vars) {
    if (s.precision != MKO_PRECISION_FP64 || vars.count > kFdMaxVariables ||
        fd_lds_bytes(batch.surfaces, vars.count) > size_t(96) << 10)
        return false;
    for (int k = 0; k < vars.count; ++k)
        if (vars.type[k] == MKO_VAR_GLASS && vars.batch_surface[k] == 0) return false;
    return true;
}

int fd_jacobian(const mko_batch* fd_batch, const mko_residual_settings* settings,
                const mko_variables* vars, int runs, const double* step_plus,
                const double* step_minus, const uint8_t* stencil, double* jacobian, double* r0,
                int64_t jstride, void* stream) {
    MKO_TRY({
        TraceParams P = make_params(*fd_batch, *settings);
        if (runs <= 0) return 0;
        const int S = P.S;
        FdPlan plan{};
        plan.P = vars->count;
        int at = 0;
        for (int first = 1; first <= S; ++first)
            for (int k = 0; k < vars->count; ++k) {
                const int s = vars->batch_surface[k];
                if (s < 0 || s >= S) throw std::invalid_argument("variable surface out of range");
                const bool glass = vars->type[k] == MKO_VAR_GLASS;
                const bool curv = vars->type[k] == MKO_VAR_CURVATURE;
                // the curvature of the first surface (the stop) changes nothing: its differences
                // run through the reference sphere only
                const int f = curv && s == 0 ? S : glass || curv ? s : s + 1;
                if (f == first) plan.var[at++] = k | (f << 16) | (int(glass) << 24);
            }
        if (runs > fd_direct_runs(plan.P, P.T)) throw std::invalid_argument("batch too large");
        const int lanes = tuple_lanes(largest_tuple(P));
        plan.parts = fd_parts(plan.P, int64_t(runs) * P.T, lanes / 64);
        const hipStream_t st = static_cast<hipStream_t>(stream);
        const auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(unsigned(runs) * unsigned(P.T * plan.parts)),
                               dim3(lanes), fd_lds_bytes(S, vars->count),
                               st, P, plan, step_plus, step_minus, stencil, jacobian, r0, jstride);
        };
        const int rpl = rays_per_lane(P);
        if (P.soft)
            rpl == 1   ? launch(fd_jacobian_kernel<true, 1>)
            : rpl == 2 ? launch(fd_jacobian_kernel<true, 2>)
            : rpl == 4 ? launch(fd_jacobian_kernel<true, 4>)
                       : launch(fd_jacobian_kernel<true, 8>);
        else
            rpl == 1   ? launch(fd_jacobian_kernel<false, 1>)
            : rpl == 2 ? launch(fd_jacobian_kernel<false, 2>)
            : rpl == 4 ? launch(fd_jacobian_kernel<false, 4>)
                       : launch(fd_jacobian_kernel<false, 8>);
        check_hip(hipGetLastError(), "fd jacobian launch");
    })
}

int fd_difference(const double* rows, int64_t stride, const uint8_t* status, int64_t rays,
                  int runs, int variables, int64_t count, const double* step_plus,
                  const double* step_minus, const uint8_t* stencil, double* jacobian, double* r0,
                  int64_t* status_changes, int64_t jstride, int64_t joffset, void* stream) {
    MKO_TRY({
        if (runs <= 0 || count <= 0) return 0;
        hipLaunchKernelGGL(fd_difference_kernel, dim3(unsigned(runs) * unsigned(variables + 1)),
                           dim3(kBlock), 0, static_cast<hipStream_t>(stream), rows, stride,
                           status, rays, runs, variables, count, step_plus, step_minus, stencil,
                           jacobian, r0, status_changes, jstride, joffset);
        check_hip(hipGetLastError(), "fd difference launch");
    })
}

} // namespace mko_internal

extern "C" {

size_t mko_adjoint_normal_workspace(int variants, int fields, int wavelengths, int variables) {
    const size_t tuples = size_t(variants) * size_t(fields) * size_t(wavelengths);
    const size_t P = size_t(variables);
    auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    return up(tuples * P * P * sizeof(float)) + up(tuples * 2 * P * sizeof(double)) +
           up(tuples * sizeof(TupleNormal));
}

int mko_adjoint_normal_device(const mko_batch* batch, const mko_residual_settings* settings,
                              const mko_variables* vars, double* a, double* g, void* workspace,
                              size_t workspace_bytes, void* stream) {
    if (settings && settings->extra && settings->extra->count > 0) {
        mko_detail::last_error = "constraint rows are evaluated by the mko_engine_* entry points";
        return MKO_ERR_INVALID;
    }
    return mko_internal::adjoint_normal_states(batch, settings, vars, a, g, workspace,
                                               workspace_bytes, mko_internal::RayStates{}, stream);
}

int mko_df64_ops_device(int op, int64_t n, const float* a, const float* b, float* out,
                        void* stream) {
    MKO_TRY({
        if (op < 0 || op > 5) throw std::invalid_argument("df64 op outside [0, 5]");
        if (n < 0) throw std::invalid_argument("negative count");
        if (n == 0) return 0;
        hipLaunchKernelGGL(df64_ops_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0,
                           static_cast<hipStream_t>(stream), op, n, a, b, out);
        check_hip(hipGetLastError(), "df64 ops launch");
    })
}

int mko_gram_mfma_device(const double* jacobian, const double* r0, int runs, int variables,
                         int64_t rows, double* a, double* g, void* stream) {
    if (variables < 1 || variables > 127 || rows < 0) {
        mko_detail::last_error = rows < 0 ? "negative row count" : "1 ... 127 variables";
        return MKO_ERR_INVALID;
    }
    return mko_internal::gram_chain(jacobian, r0, runs, variables, rows, a, g, stream, nullptr);
}

size_t mko_vjp_workspace(int variants, int fields, int wavelengths, int variables) {
    return ((size_t(variants) * size_t(fields) * size_t(wavelengths) * size_t(variables) *
             sizeof(double)) + 255) & ~size_t(255);
}

int mko_vjp_device(const mko_batch* batch, const mko_residual_settings* settings,
                   const mko_variables* vars, const double* grad, int64_t grad_stride,
                   double* out, void* workspace, size_t workspace_bytes, void* stream) {
    MKO_TRY({
        no_rows(*settings);
        if (settings->precision != MKO_PRECISION_FP64)
            throw std::invalid_argument("the VJP traces in FP64 (precision MKO_PRECISION_FP64)");
        const TraceParams P = make_params(*batch, *settings);
        const ParamMap m = make_map(*vars, *batch, true);
        if (grad_stride < P.trace_rows) throw std::invalid_argument("grad_stride smaller than trace rows");
        if (P.V == 0) return 0;
        if (int64_t(P.V) * P.T > 0x7fffffffLL) throw std::invalid_argument("batch too large");
        if (workspace_bytes < mko_vjp_workspace(P.V, P.F, P.L, m.P))
            throw std::invalid_argument("workspace too small");
        const hipStream_t s = static_cast<hipStream_t>(stream);
        double* part = static_cast<double*>(workspace);
        if (m.glass) launch_vjp<true>(P, m, grad, grad_stride, part, s);
        else launch_vjp<false>(P, m, grad, grad_stride, part, s);
        check_hip(hipGetLastError(), "vjp launch");
        const int64_t n = int64_t(P.V) * m.P;
        hipLaunchKernelGGL(vjp_finalize_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s,
                           P.V, P.T, m.P, part, out);
        check_hip(hipGetLastError(), "vjp finalize launch");
    })
}

int mko_gram_device(const double* jacobian, const double* r0, int runs, int variables,
                    int64_t rows, double* a, double* g, void* stream) {
    return mko_internal::gram_chain(jacobian, r0, runs, variables, rows, a, g, stream, nullptr);
}

} // extern "C"
