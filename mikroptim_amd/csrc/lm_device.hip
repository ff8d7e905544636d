// Device side of the batched Levenberg-Marquardt control (levenberg_marquardt,
// src/optim/levenberg_marquardt.cpp:332-572): the per-run step solve, acceptance and convergence
// tests of one LM cycle run on the GPU, one wavefront (64 lanes) per run, so a cycle needs no
// host round trip of the normal equations or the trial points.
//
// Every floating-point operation is the one the host control performs, in the same order:
// products and sums without contraction (fp contract off below), correctly rounded division and
// square root (__ddiv_rn, __dsqrt_rn), std::max / std::min as (a < b) ? b : a / (b < a) ? b : a.
// Given the same normal equations and merits, device and host control take bit-identical
// trajectories. Sums keep the host order (that of the reference's cholesky / cholesky_solve,
// src/optim/levenberg_marquardt.cpp:70-112): the Cholesky factor and the forward substitution run
// lane-parallel over rows, each entry receiving its subtractions in the host's order; the back
// substitution and the step model (lin, quad) form their products on the lanes and add them in
// ascending order; maxima (order-independent) are wave reductions.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include "lm_device.hpp"

#pragma clang fp contract(off)

namespace mko_lmdev {
namespace {

constexpr int kLanes = 64;
constexpr int kMaxP = 128;            // two slots per lane
constexpr int kSlots = kMaxP / kLanes; // 2: the selects below assume it
constexpr double kModelDamping = 1e-12;
constexpr double kFdStepFactor = 6.0554544523933395e-06; // 2^(-52/3)

// Lane k's value of v, in every lane (k uniform).
__device__ __forceinline__ double lane_value(double v, int k) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), k);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), k);
    return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double dmax(double a, double b) { return (a < b) ? b : a; }
__device__ __forceinline__ double dmin(double a, double b) { return (b < a) ? b : a; }
__device__ __forceinline__ double scale_of(double x, double typical) { return dmax(fabs(x), typical); }

__device__ __forceinline__ bool blocks(const State& S, int k, double x, double dir) {
    if (S.lower[k] == S.upper[k]) return true;
    return (x <= S.lower[k] && dir < 0.0) || (x >= S.upper[k] && dir > 0.0);
}

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = dmax(v, __shfl_xor(v, off, 64));
    return v;
}

// Orders the wave's LDS accesses across its lanes (one wavefront per workgroup: they execute in
// order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The solve's LDS: the packed lower triangle of the free variables' matrix with the right-hand side
// as one more row (columns of P + 1, P, ... 2 entries), a step per variable and the free
// variables' indices; sized by P, so that more runs' workgroups fit a CU.
__host__ __device__ __forceinline__ size_t solve_entries(int P) { return size_t(P + 1) * (P + 2) / 2; }
struct SolveLds {
    double* m;
    double* delta;
    int* idx;
};
__device__ __forceinline__ SolveLds solve_lds(double* lds, int P) {
    double* delta = lds + solve_entries(P);
    return SolveLds{lds, delta, reinterpret_cast<int*>(delta + P)};
}

// solve_step: (A_FF + mu D_FF) delta_F = -g_F on the free variables with the active set; writes
// trial, step_norm, predicted and solved of the run (trial, step_norm and predicted only when
// the factorisation succeeds, like the host).
// a, g: the run's normal equations (a symmetric). Variable k, and row i of the free variables'
// matrix, belong to lane k % 64, slot k / 64 (two slots: up to 127 variables and the right-hand
// side's row).
//
// One wave works through dependent chains, so what bounds it is their latency, not the arithmetic
// (0.04 MFLOP at 48 variables): the matrix is loaded 8 columns at a time, the Cholesky is
// left-looking as the host's (a column's products are loaded 8 at a time ahead of the chain of
// subtractions, no index tables, no barriers), the right-hand side rides along as its last row
// (the forward substitution's operations in the same order), and the sums of the step's model are
// chains over values from other lanes' registers. 256 runs of 48 variables: 150 -> 120 us (a CU
// holds one wave then; half of it issue, half latency).
__device__ void solve_step(const State& S, int run, const double* a, const double* g, double mu,
                           const SolveLds& L) {
    const int n = S.P;
    const int lane = threadIdx.x;
    double* __restrict__ m = L.m;
    double x[kSlots], delta[kSlots];
    bool fixed[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        const int k = lane + s * kLanes;
        x[s] = delta[s] = 0.0;
        fixed[s] = true;
        if (k < n) {
            x[s] = S.x[size_t(run) * n + k];
            fixed[s] = blocks(S, k, x[s], -g[k]);
        }
    }
    const uint64_t below = (uint64_t(1) << lane) - 1;
    for (int round = 0; round <= n; ++round) {
        const uint64_t free0 = __ballot(!fixed[0]), free1 = __ballot(!fixed[1]);
        const int f0 = __popcll(free0), f = f0 + __popcll(free1);
        if (!fixed[0]) L.idx[__popcll(free0 & below)] = lane;
        if (!fixed[1]) L.idx[f0 + __popcll(free1 & below)] = lane + kLanes;
#pragma unroll
        for (int s = 0; s < kSlots; ++s) delta[s] = 0.0;
        if (f == 0) break;
        wave_sync();
        const int F = f + 1;
        const bool two = F > kLanes; // uniform
        // column j of the packed matrix at m + c(j), rows j ... f at their own index
        const auto c = [&](int j) { return j * F - (j * (j - 1)) / 2 - j; };
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            const int i = lane + s * kLanes;
            if (s == 1 && !two) break;
            const int var = i < f ? L.idx[i] : 0;
            const double d = i < f ? S.d[size_t(run) * n + var] : 0.0;
            for (int j0 = 0; j0 < f; j0 += 8) {
                double v[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int j = j0 + q;
                    v[q] = 0.0;
                    if (j < f && i >= j && i <= f) {
                        const int vj = L.idx[j];
                        v[q] = i < f ? a[size_t(vj) * n + var] : -g[vj];
                    }
                }
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int j = j0 + q;
                    if (j < f && i >= j && i <= f) m[c(j) + i] = i == j ? v[q] + mu * d : v[q];
                }
            }
        }
        wave_sync();
        // Cholesky, left-looking: entry (i, j) receives the subtractions of l(i, k) l(j, k), k < j,
        // in ascending order, as in the host's loop; the row f of the right-hand side receives
        // those of the forward substitution, y_j = (b_j - sum_k l(j, k) y_k) / l(j, j)
        int row[kSlots];
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            const int i = lane + s * kLanes;
            row[s] = i < f ? i : f; // lanes beyond the last row read it again
        }
        for (int j = 0; j < f; ++j) {
            const int cj = c(j);
            double acc[kSlots];
            acc[0] = m[cj + (row[0] < j ? j : row[0])];
            acc[1] = two ? m[cj + (row[1] < j ? j : row[1])] : 0.0;
            int ck = 0; // c(k)
            int k = 0;
            for (; k + 8 <= j; k += 8) {
                double u[8], w0[8], w1[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    u[q] = m[ck + j];
                    w0[q] = m[ck + row[0]];
                    w1[q] = two ? m[ck + row[1]] : 0.0;
                    ck += F - (k + q) - 1;
                }
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    acc[0] -= w0[q] * u[q];
                    if (two) acc[1] -= w1[q] * u[q];
                }
            }
            for (; k < j; ++k) {
                const double u = m[ck + j];
                acc[0] -= m[ck + row[0]] * u;
                if (two) acc[1] -= m[ck + row[1]] * u;
                ck += F - k - 1;
            }
            const double diag = lane_value(j < kLanes ? acc[0] : acc[1], j % kLanes);
            if (!(diag > 0.0) || !isfinite(diag)) {
                if (lane == 0) S.solved[run] = 0;
                return;
            }
            const double l = __dsqrt_rn(diag);
#pragma unroll
            for (int s = 0; s < kSlots; ++s) {
                const int i = lane + s * kLanes;
                if (s == 1 && !two) break;
                const double v = __ddiv_rn(acc[s], l);
                if (i >= j && i <= f) m[cj + i] = i == j ? l : v;
            }
            wave_sync();
        }
        // back substitution, x_i = (y_i - sum_{k > i} l(k, i) x_k) / l(i, i) for i = f-1 ... 0:
        // the lane of row k keeps y_k, then x_k, in a register and forms the product l(k, i) x_k;
        // every lane subtracts the products from y_i in ascending k, as the host does, and
        // divides, so x_i is the same in all lanes and the lane of row i keeps it
        double xk[kSlots];
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            const int k = lane + s * kLanes;
            xk[s] = k < f ? m[c(k) + f] : 0.0;
        }
        for (int i = f - 1; i >= 0; --i) {
            const int ci = c(i);
            double p[kSlots];
#pragma unroll
            for (int s = 0; s < kSlots; ++s) {
                const int k = lane + s * kLanes;
                p[s] = (k > i && k < f) ? m[ci + k] * xk[s] : 0.0;
            }
            const double lii = m[ci + i];
            double acc = lane_value(i < kLanes ? xk[0] : xk[1], i % kLanes);
            const int end0 = f < kLanes ? f : kLanes;
            int k = i + 1;
            for (; k + 8 <= end0; k += 8) {
                double t[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) t[q] = lane_value(p[0], k + q);
#pragma unroll
                for (int q = 0; q < 8; ++q) acc -= t[q];
            }
            for (; k < end0; ++k) acc -= lane_value(p[0], k);
            for (; k < f; ++k) acc -= lane_value(p[1], k - kLanes);
            const double xi = __ddiv_rn(acc, lii);
#pragma unroll
            for (int s = 0; s < kSlots; ++s)
                if (lane + s * kLanes == i) xk[s] = xi;
        }
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            const int i = lane + s * kLanes;
            if (i < f) L.delta[L.idx[i]] = xk[s];
        }
        wave_sync();
        bool newly_fixed = false;
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            const int k = lane + s * kLanes;
            if (!fixed[s]) {
                delta[s] = L.delta[k];
                if (blocks(S, k, x[s], delta[s])) {
                    fixed[s] = true;
                    newly_fixed = true;
                }
            }
        }
        wave_sync();
        if (!__any(newly_fixed)) break;
    }
    double step[kSlots], lin_p[kSlots], quad_p[kSlots];
    // dmax(0, .) per variable first: a NaN ratio drops out as in the host's sequential std::max,
    // so the butterfly only sees ordered values and every lane ends with the same maximum
    double r = 0.0;
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        const int k = lane + s * kLanes;
        step[s] = 0.0;
        if (k < n) {
            const double t = dmin(dmax(x[s] + delta[s], S.lower[k]), S.upper[k]);
            S.trial[size_t(run) * n + k] = t;
            step[s] = t - x[s];
            const double ratio = __ddiv_rn(fabs(step[s]), scale_of(x[s], S.typical[k]));
            r = dmax(r, dmax(0.0, ratio));
        }
    }
    const double nrm = wave_max(r);
    // a q of the step model: row q of a is its column q
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        const int q = lane + s * kLanes;
        const int qc = q < n ? q : n - 1;
        double aq = 0.0;
        for (int p0 = 0; p0 < n; p0 += 8) {
            double v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = p0 + e < n ? a[size_t(p0 + e) * n + qc] : 0.0;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int p = p0 + e;
                if (p < n)
                    aq += v[e] * lane_value(p < kLanes ? step[0] : step[1], p % kLanes);
            }
        }
        lin_p[s] = q < n ? step[s] * g[q] : 0.0;
        quad_p[s] = step[s] * aq;
        if (s == 0 && n <= kLanes) {
            lin_p[1] = quad_p[1] = 0.0;
            break;
        }
    }
    double lin = 0.0, quad = 0.0;
    for (int q = 0; q < n; ++q) {
        lin += lane_value(q < kLanes ? lin_p[0] : lin_p[1], q % kLanes);
        quad += lane_value(q < kLanes ? quad_p[0] : quad_p[1], q % kLanes);
    }
    if (lane == 0) {
        S.step_norm[run] = nrm;
        S.predicted[run] = -(2.0 * lin + quad);
        S.solved[run] = 1;
    }
    __syncthreads();
}

// prepare_step: scaling diagonal D (Marquardt with floor) and the scaled gradient norm. The
// per-variable terms are formed lane-parallel; the two maxima are order-independent (finite
// values), so they equal the host's sequential maxima.
__device__ void prepare_step(const State& S, const Options& o, int run, const double* a,
                             const double* g) {
    const int n = S.P;
    const int lane = threadIdx.x;
    const double* x = S.x + size_t(run) * n;
    double smax_l = 0.0;
    for (int k = lane; k < n; k += kLanes) {
        const double sk = scale_of(x[k], S.typical[k]);
        smax_l = dmax(smax_l, dmax(0.0, a[size_t(k) * n + k] * sk * sk));
    }
    const double smax = wave_max(smax_l);
    const double merit = S.merit[run];
    double gmax_l = 0.0;
    for (int k = lane; k < n; k += kLanes) {
        const double sk = scale_of(x[k], S.typical[k]);
        const double akk = a[size_t(k) * n + k];
        const double floor = smax > 0.0 ? __ddiv_rn(o.diag_floor * smax, sk * sk)
                                        : __ddiv_rn(1.0, sk * sk);
        S.d[size_t(run) * n + k] = dmax(akk, floor);
        double ratio = 0.0;
        if (!blocks(S, k, x[k], -g[k])) {
            const double den = __dsqrt_rn(akk * merit);
            if (den > 0.0) ratio = __ddiv_rn(fabs(g[k]), den);
        }
        gmax_l = dmax(gmax_l, dmax(0.0, ratio));
    }
    const double gmax = wave_max(gmax_l);
    if (lane == 0) S.gradient_norm[run] = gmax;
}

// One wavefront per run (also in update_kernel): its variables on the lanes. 256 runs of 48
// variables: 38 -> 4 us here, 22 -> 5 us in update_kernel (a thread per run walked its variables
// one load at a time).
__global__ __launch_bounds__(kLanes) void init_kernel(State S, Options o) {
    const int run = blockIdx.x;
    const int n = S.P;
    for (int k = threadIdx.x; k < n; k += kLanes) {
        S.trial[size_t(run) * n + k] = S.x[size_t(run) * n + k];
        S.g[size_t(run) * n + k] = 0.0;
        S.d[size_t(run) * n + k] = 0.0;
    }
    if (threadIdx.x != 0) return;
    S.mu[run] = o.initial_damping;
    S.nu[run] = 2.0;
    S.step_norm[run] = 0.0;
    S.predicted[run] = 0.0;
    S.gradient_norm[run] = 0.0;
    S.model_decrease[run] = __builtin_nan("");
    S.failed[run] = 0;
    S.hard[run] = 0;
    S.status[run] = MKO_LM_RUNNING;
    S.iterations[run] = 0;
    S.accepted[run] = 0;
    S.jacobians[run] = 0;
    S.history_len[run] = 0;
    S.need_jacobian[run] = 1;
    S.rejected[run] = 0;
    S.solved[run] = 0;
    S.evaluate[run] = 0;
}

__device__ __forceinline__ void push_history(const State& S, int run, double merit) {
    const int c = S.history_len[run];
    S.history[size_t(run) * S.H + (c % S.H)] = merit;
    S.history_len[run] = c + 1;
}

__global__ __launch_bounds__(256) void start_kernel(State S, const double* merit,
                                                    const int64_t* failed, const int64_t* hard) {
    const int run = blockIdx.x * blockDim.x + threadIdx.x;
    if (run >= S.n) return;
    const double m = merit[run];
    S.merit[run] = m;
    S.failed[run] = failed[run];
    S.hard[run] = hard[run];
    push_history(S, run, m);
    if (!isfinite(m)) S.status[run] = MKO_LM_NUMERICAL_ERROR;
    else if (m == 0.0) S.status[run] = MKO_LM_CONVERGED_MERIT;
}

// Ordered compaction in one workgroup of 1024 threads (chunks of 1024 runs, block scan).
__global__ __launch_bounds__(1024) void select_kernel(State S, int kind, int max_iterations,
                                                      const int32_t* in, const int32_t* in_count,
                                                      int32_t* list, int32_t* count, int32_t* pos) {
    __shared__ int32_t wave_total[16];
    __shared__ int32_t base_s;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int total = kind == kListEvaluate ? *in_count : S.n;
    if (tid == 0) base_s = 0;
    __syncthreads();
    for (int start = 0; start < total; start += 1024) {
        const int e = start + tid;
        bool pick = false;
        int run = -1;
        if (e < total) {
            run = kind == kListEvaluate ? in[e] : e;
            const int st = S.status[run];
            if (kind == kListJacobian) {
                pick = st == MKO_LM_RUNNING && S.need_jacobian[run] &&
                       S.iterations[run] < max_iterations;
            } else if (kind == kListCycle) {
                if (st == MKO_LM_RUNNING) {
                    if (S.iterations[run] >= max_iterations) S.status[run] = MKO_LM_MAX_ITERATIONS;
                    else pick = true;
                }
            } else {
                pick = S.evaluate[run] != 0;
            }
        }
        const uint64_t mask = __ballot(pick);
        const int before = __popcll(mask & ((uint64_t(1) << lane) - 1));
        if (lane == 0) wave_total[wave] = __popcll(mask);
        __syncthreads();
        int offset = base_s;
        for (int w = 0; w < wave; ++w) offset += wave_total[w];
        if (pick) list[offset + before] = run;
        if (pos && run >= 0) pos[run] = pick ? offset + before : -1;
        __syncthreads();
        if (tid == 0) {
            int sum = 0;
            for (int w = 0; w < 16; ++w) sum += wave_total[w];
            base_s += sum;
        }
        __syncthreads();
    }
    if (tid == 0) *count = base_s;
}

// Stable split of the Jacobian list `in` (*in_count runs) in one workgroup of 1024 threads: the
// runs whose point has no failed ray into `clean` (in order, count *clean_count), the others
// into `other` (in order, count *other_count).
__global__ __launch_bounds__(1024) void split_kernel(State S, const int32_t* in,
                                                     const int32_t* in_count, int32_t* clean,
                                                     int32_t* clean_count, int32_t* other,
                                                     int32_t* other_count) {
    __shared__ int32_t wave_clean[16], wave_other[16];
    __shared__ int32_t base_c, base_o;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int total = *in_count;
    if (tid == 0) base_c = base_o = 0;
    __syncthreads();
    for (int start = 0; start < total; start += 1024) {
        const int e = start + tid;
        const int run = e < total ? in[e] : -1;
        const bool c = run >= 0 && S.failed[run] == 0;
        const bool o = run >= 0 && !c;
        const uint64_t mc = __ballot(c), mo = __ballot(o);
        const uint64_t below = (uint64_t(1) << lane) - 1;
        if (lane == 0) {
            wave_clean[wave] = __popcll(mc);
            wave_other[wave] = __popcll(mo);
        }
        __syncthreads();
        int oc = base_c, oo = base_o;
        for (int w = 0; w < wave; ++w) {
            oc += wave_clean[w];
            oo += wave_other[w];
        }
        if (c) clean[oc + __popcll(mc & below)] = run;
        if (o) other[oo + __popcll(mo & below)] = run;
        __syncthreads();
        if (tid == 0) {
            for (int w = 0; w < 16; ++w) {
                base_c += wave_clean[w];
                base_o += wave_other[w];
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        *clean_count = base_c;
        *other_count = base_o;
    }
}

// Number of runs the next Jacobian list holds (kListJacobian's test) whose point has failed rays.
__global__ __launch_bounds__(1024) void count_failing_kernel(State S, int max_iterations,
                                                             int32_t* count) {
    __shared__ int32_t wave_total[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int n = 0;
    for (int run = tid; run < S.n; run += 1024)
        n += S.status[run] == MKO_LM_RUNNING && S.need_jacobian[run] &&
             S.iterations[run] < max_iterations && S.failed[run] > 0;
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off);
    if (lane == 0) wave_total[wave] = n;
    __syncthreads();
    if (tid == 0) {
        int sum = 0;
        for (int w = 0; w < 16; ++w) sum += wave_total[w];
        *count = sum;
    }
}

__global__ __launch_bounds__(64) void gather_kernel(State S, const int32_t* list, int count,
                                                    const int32_t* dcount, int trial,
                                                    const int32_t* round_index, double* xs,
                                                    int32_t* tidx) {
    const int j = blockIdx.x;
    if (j >= count || (dcount && j >= *dcount)) return;
    const int run = list[j];
    const double* src = (trial ? S.trial : S.x) + size_t(run) * S.P;
    for (int k = threadIdx.x; k < S.P; k += 64) xs[size_t(j) * S.P + k] = src[k];
    if (threadIdx.x == 0 && tidx) tidx[j] = round_index ? round_index[run] : run;
}

// One wavefront per listed run (round_cycle, the runs that received new normal equations).
__global__ __launch_bounds__(kLanes) void prepare_kernel(State S, Options o, const int32_t* list,
                                                         int count, const int32_t* dcount,
                                                         const double* a_c,
                                                         const double* g_c) {
    extern __shared__ double m_tri[];
    const SolveLds L = solve_lds(m_tri, S.P);
    const int j = blockIdx.x;
    if (j >= count || (dcount && j >= *dcount)) return;
    const int run = list[j];
    const int n = S.P, lane = threadIdx.x;
    bool finite = true;
    for (int e0 = lane; e0 < n * n; e0 += 8 * kLanes) {
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int e = e0 + q * kLanes;
            v[q] = e < n * n ? a_c[size_t(j) * n * n + e] : 0.0;
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int e = e0 + q * kLanes;
            if (e < n * n) S.a[size_t(run) * n * n + e] = v[q];
            finite = finite && isfinite(v[q]);
        }
    }
    for (int k = lane; k < n; k += kLanes) {
        const double v = g_c[size_t(j) * n + k];
        S.g[size_t(run) * n + k] = v;
        finite = finite && isfinite(v);
    }
    const bool all_finite = __all(finite);
    if (lane == 0) {
        S.need_jacobian[run] = 0;
        S.jacobians[run] += 1;
        if (!all_finite) S.status[run] = MKO_LM_NUMERICAL_ERROR;
    }
    if (!all_finite) return;
    // the compact inputs are read-only in this kernel; the state copies serve later kernels
    const double* a = a_c + size_t(j) * n * n;
    const double* g = g_c + size_t(j) * n;
    prepare_step(S, o, run, a, g);
    __syncthreads();
    solve_step(S, run, a, g, kModelDamping, L);
    if (lane == 0) {
        const bool solved = S.solved[run] != 0;
        const double merit = S.merit[run];
        const double predicted = S.predicted[run];
        S.model_decrease[run] = solved ? __ddiv_rn(predicted, merit) : __builtin_nan("");
        if (S.gradient_norm[run] <= o.gtol) S.status[run] = MKO_LM_CONVERGED_GRADIENT;
        else if (solved && predicted >= 0.0 && predicted <= o.ftol * merit)
            S.status[run] = MKO_LM_CONVERGED_MERIT;
        else if (solved && S.step_norm[run] <= o.xtol) S.status[run] = MKO_LM_CONVERGED_STEP;
    }
}

__global__ __launch_bounds__(kLanes) void step_kernel(State S, Options o, const int32_t* list,
                                                      int count, const int32_t* dcount) {
    extern __shared__ double m_tri[];
    const SolveLds L = solve_lds(m_tri, S.P);
    const int j = blockIdx.x;
    if (j >= count || (dcount && j >= *dcount)) return;
    const int run = list[j];
    solve_step(S, run, S.a + size_t(run) * S.P * S.P, S.g + size_t(run) * S.P, S.mu[run], L);
    if (threadIdx.x == 0) {
        const bool solved = S.solved[run] != 0;
        S.evaluate[run] = 0;
        if (solved && S.rejected[run] && S.step_norm[run] <= o.xtol)
            S.status[run] = MKO_LM_CONVERGED_STEP;
        else if (solved)
            S.evaluate[run] = 1;
    }
}

__global__ __launch_bounds__(kLanes) void update_kernel(State S, Options o, const int32_t* list,
                                                        int count, const int32_t* dcount,
                                                        const int32_t* pos, const double* f,
                                                        const int64_t* failed,
                                                        const int64_t* hard) {
    const int j = blockIdx.x;
    if (j >= count || (dcount && j >= *dcount)) return;
    const int run = list[j];
    int status = S.status[run];
    if (status == MKO_LM_CONVERGED_STEP) return;
    bool accept = false;
    const double merit = S.merit[run];
    double now = merit, rho = 0.0;
    int64_t failed_new = 0, hard_new = 0;
    if (S.solved[run]) {
        const int e = pos[run];
        const double f_new = f[e];
        failed_new = failed[e];
        hard_new = hard[e];
        const double predicted = S.predicted[run];
        rho = __ddiv_rn(merit - f_new, predicted);
        accept = isfinite(f_new) && predicted > 0.0 && f_new < merit &&
                 !(o.reject_new_failures && hard_new > S.hard[run]);
        if (accept) now = f_new;
    }
    if (accept) {
        const int n = S.P;
        for (int k = threadIdx.x; k < n; k += kLanes)
            S.x[size_t(run) * n + k] = S.trial[size_t(run) * n + k];
    }
    if (threadIdx.x != 0) return;
    S.iterations[run] += 1;
    if (accept) {
        S.merit[run] = now;
        S.failed[run] = failed_new;
        S.hard[run] = hard_new;
        const double t = 2.0 * rho - 1.0;
        S.mu[run] = S.mu[run] * dmax(1.0 / 3.0, 1.0 - t * t * t);
        S.nu[run] = 2.0;
        S.need_jacobian[run] = 1;
        S.rejected[run] = 0;
        S.accepted[run] += 1;
        if (now == 0.0) status = MKO_LM_CONVERGED_MERIT;
    } else {
        const double mu = S.mu[run] * S.nu[run];
        S.mu[run] = mu;
        S.nu[run] = S.nu[run] * 2.0;
        S.rejected[run] = 1;
        if (mu > o.max_damping) status = MKO_LM_DAMPING_LIMIT;
    }
    push_history(S, run, now);
    if (o.stall_window > 0 && status == MKO_LM_RUNNING) {
        const int w = o.stall_window;
        const int size = S.history_len[run];
        if (size > w) {
            const double old = S.history[size_t(run) * S.H + ((size - 1 - w) % S.H)];
            if (old - now <= o.stall_tolerance * old) status = MKO_LM_CONVERGED_STALL;
        }
    }
    S.status[run] = status;
}

__global__ __launch_bounds__(64) void fd_pattern_kernel(int count, int P, const double* xs,
                                                        const double* lower, const double* upper,
                                                        const double* typical, double* plus,
                                                        double* minus, double* step_plus,
                                                        double* step_minus, uint8_t* stencil) {
    const int j = blockIdx.x;
    if (j >= count) return;
    for (int k = threadIdx.x; k < P; k += 64) {
        const size_t at = size_t(j) * P + k;
        const double x = xs[at];
        const double lo = lower[k], hi = upper[k];
        const double h = kFdStepFactor * dmax(fabs(x), typical[k]);
        const double up = x + h, down = x - h;
        double xa, xb;
        uint8_t sten = MKO_STENCIL_CENTRAL;
        if (up <= hi && down >= lo) {
            xa = up;
            xb = down;
        } else {
            const bool towards_upper = hi - x >= x - lo;
            const double far = towards_upper ? x + 2.0 * h : x - 2.0 * h;
            if (towards_upper ? far <= hi : far >= lo) {
                sten = MKO_STENCIL_ONE_SIDED;
                xa = towards_upper ? up : down;
                xb = far;
            } else {
                sten = MKO_STENCIL_TRUNCATED;
                xa = up <= hi ? up : hi;
                xb = down >= lo ? down : lo;
            }
        }
        plus[at] = xa;
        minus[at] = xb;
        step_plus[at] = xa - x;
        step_minus[at] = xb - x;
        stencil[at] = sten;
    }
}

inline hipStream_t st(void* s) { return static_cast<hipStream_t>(s); }
inline size_t solve_bytes(int P) {
    return (solve_entries(P) + size_t(P)) * sizeof(double) + size_t(P) * sizeof(int);
}
inline unsigned blocks_of(int n, int per) { return unsigned((n + per - 1) / per); }

} // namespace

void launch_init(const State& s, const Options& o, void* stream) {
    if (s.n > 0) hipLaunchKernelGGL(init_kernel, dim3(unsigned(s.n)), dim3(kLanes), 0, st(stream), s, o);
}

void launch_start(const State& s, const double* merit, const int64_t* failed, const int64_t* hard,
                  void* stream) {
    if (s.n > 0)
        hipLaunchKernelGGL(start_kernel, dim3(blocks_of(s.n, 256)), dim3(256), 0, st(stream), s,
                           merit, failed, hard);
}

void launch_select(const State& s, int kind, int max_iterations, const int32_t* in,
                   const int32_t* in_count, int32_t* list, int32_t* count, int32_t* pos,
                   void* stream) {
    hipLaunchKernelGGL(select_kernel, dim3(1), dim3(1024), 0, st(stream), s, kind, max_iterations,
                       in, in_count, list, count, pos);
}

void launch_split(const State& s, const int32_t* in, const int32_t* in_count, int32_t* clean,
                  int32_t* clean_count, int32_t* other, int32_t* other_count, void* stream) {
    hipLaunchKernelGGL(split_kernel, dim3(1), dim3(1024), 0, st(stream), s, in, in_count, clean,
                       clean_count, other, other_count);
}

void launch_count_failing(const State& s, int max_iterations, int32_t* count, void* stream) {
    hipLaunchKernelGGL(count_failing_kernel, dim3(1), dim3(1024), 0, st(stream), s,
                       max_iterations, count);
}

void launch_gather(const State& s, const int32_t* list, int count, bool trial,
                   const int32_t* round_index, double* xs, int32_t* tidx, void* stream,
                   const int32_t* dcount) {
    if (count > 0)
        hipLaunchKernelGGL(gather_kernel, dim3(unsigned(count)), dim3(64), 0, st(stream), s, list,
                           count, dcount, trial ? 1 : 0, round_index, xs, tidx);
}

void launch_prepare(const State& s, const Options& o, const int32_t* list, int count,
                    const double* a_c, const double* g_c, void* stream, const int32_t* dcount) {
    if (count > 0)
        hipLaunchKernelGGL(prepare_kernel, dim3(unsigned(count)), dim3(kLanes), solve_bytes(s.P),
                           st(stream), s, o, list, count, dcount, a_c, g_c);
}

void launch_step(const State& s, const Options& o, const int32_t* list, int count, void* stream,
                 const int32_t* dcount) {
    if (count > 0)
        hipLaunchKernelGGL(step_kernel, dim3(unsigned(count)), dim3(kLanes), solve_bytes(s.P),
                           st(stream), s, o, list, count, dcount);
}

void launch_update(const State& s, const Options& o, const int32_t* list, int count,
                   const int32_t* pos, const double* f, const int64_t* failed,
                   const int64_t* hard, void* stream, const int32_t* dcount) {
    if (count > 0)
        hipLaunchKernelGGL(update_kernel, dim3(unsigned(count)), dim3(kLanes), 0, st(stream), s,
                           o, list, count, dcount, pos, f, failed, hard);
}

void launch_fd_pattern(int count, int P, const double* xs, const double* lower,
                       const double* upper, const double* typical, double* plus, double* minus,
                       double* step_plus, double* step_minus, uint8_t* stencil, void* stream) {
    if (count > 0)
        hipLaunchKernelGGL(fd_pattern_kernel, dim3(unsigned(count)), dim3(64), 0, st(stream), count,
                           P, xs, lower, upper, typical, plus, minus, step_plus, step_minus,
                           stencil);
}

} // namespace mko_lmdev
