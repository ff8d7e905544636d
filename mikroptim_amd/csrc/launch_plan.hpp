// Launch shapes that follow from the sizes alone: plain host code, shared by the launches and the
// host layer.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace mko_internal {

// Most runs of one fd_jacobian launch: the kernel counts the tuples of every variant, 2 P + 1
// variants a run, in 32 bits, and a launch holds fewer than 2^32 threads (up to 256 a tuple; a
// tuple's variables go to several workgroups only where there are fewer than 6144 tuples).
inline int64_t fd_direct_runs(int variables, int64_t tuples) {
    const int64_t per_run = (2 * int64_t(variables) + 1) * tuples;
    return std::min(int64_t(0x7fffffff) / per_run, int64_t(0xffffffff) / (256 * tuples));
}

// Workgroups (of 1 ... 4 waves) that share a tuple's variables in fd_jacobian_kernel. Each traces the
// point itself, 2 of its about 2 + P / parts passes, so parts pay where the tuples alone leave
// places on the chip empty: some 4 waves per SIMD are resident, and at most about 9 workgroups of
// small tuples per CU (LDS). us in 1 / 2 / 4 parts, 25 surfaces, 512 rays (4 waves) and 72 rays (2
// waves) a tuple, or 22 surfaces and 48 rays (1 wave):
//   48 variables, 512 rays   140 tuples 712 /  518 /  398,   840 1658 / 1430 / 1502,
//                           1120 2028 / 1788 / 1910,        1680 2754 / 2841 / 2941
//   24 variables, 72 rays    560 tuples 286 /  203 /  193,  1015  365 /  265 /  290,
//                           2240  555 /  519 /  591,        3500  757 /  766 /  887
//   47 variables, 48 rays    600 tuples 446 /  323 /  235,  1020  442 /  336 /  393,
//                           4080 1310 / 1236 / 1242
//   4 variables, 72 rays     144 tuples  18 /   16 /   13,   576   22 /   20 /   24,
//                           1800   31 /   39 /   54
inline int fd_parts(int variables, int64_t tuples, int waves) {
    const int64_t load = tuples * std::max(waves, 2);
    if (variables < 8) return load < 2560 ? 2 : 1;
    return load < 1792 ? 4 : tuples * waves < 6144 ? 2 : 1;
}

// Entries of the upper triangle per thread of adjoint_normal_finalize_kernel: five read the tuples'
// S once for all of them, which pays where many runs fill the chip and a workgroup's 1280 entries
// are nearly all there. us with 1 / 5: 48 variables of 35 tuples, 256 runs 21 / 23, 400 runs 35 / 28,
// 1024 runs 78 / 74; 96 variables of 20 tuples, 1024 runs 182 / 155; but 5 variables, 512 runs 10 /
// 20 and 2048 runs 20 / 70; 36 variables, 1024 runs 21 / 26; 56 variables (two workgroups, 62 % of
// their entries), 1024 runs 46 / 57.
inline int finalize_entries(int variables, int runs) {
    const int nu = variables * (variables + 1) / 2, places = 1280 * ((nu + 1279) / 1280);
    return runs >= 400 && 8 * nu >= 7 * places ? 5 : 1;
}

// gram_kernel's split of a run's units (gw waves of 64 columns of g, then the upper 16 x 16 tiles of
// a tg x tg grid) over `parts` workgroups of up to `upp` units, 1 ... 127 variables.
struct GramPlan {
    int tg, gw, units, parts, upp;
};
// At least 4 units (one tile per SIMD) each, and only while the runs leave CUs idle (up to 512
// workgroups): beyond that a second workgroup only reads most of the run's J again. Every part
// has a unit.
inline GramPlan gram_plan(int variables, int runs) {
    GramPlan p{};
    p.tg = (variables + 15) / 16;
    p.gw = (variables + 63) / 64;
    p.units = p.gw + p.tg * (p.tg + 1) / 2;
    p.parts = std::max(1, std::min((p.units + 3) / 4, 512 / runs));
    p.upp = (p.units + p.parts - 1) / p.parts;
    p.parts = (p.units + p.upp - 1) / p.upp; // rounding upp up may leave fewer
    return p;
}

// LDS slots of a tuple's n rays: a multiple of the q lanes by an odd number, so that the tuples
// side by side fall on different banks.
constexpr int prefilter_slots(int n, int q) { return q * (((n + q - 1) / q) | 1); }

// Lanes of prefilter_kernel that sum a tuple, by the largest tuple: the most of 8 ... 64 that idle on
// at most 1/8 of the rays' slots (72 rays: 16 lanes of 5 rays; 8 lanes if none does), a whole
// workgroup above 256 rays.
inline int prefilter_lanes(int n) {
    if (n > 256) return 256;
    for (int q = 64; q > 8; q /= 2)
        if (8 * n >= 7 * q * ((n + q - 1) / q)) return q;
    return 8;
}

constexpr size_t kPrefilterStepBytes = 16;

// prefilter_kernel's lanes per tuple (q sum it, Q trace it), workgroups per tuple index and dynamic
// LDS for `variants` of `tuples` tuples of up to n rays on `rings` rings.
struct PrefilterPlan {
    int q, Q, groups;
    size_t lds;
};
// Q is q, doubled (up to one ray per lane) while the launch has less than 4 workgroups per CU. One
// variant of 35 tuples of 72 rays and 25 surfaces, the whole call: 211 us with 16 lanes, 176 with
// 128; 2000 variants of 9 tuples of 72 rays and more keep the lanes of the sums (512 variants of 35
// tuples: 550 -> 418 us).
inline PrefilterPlan prefilter_plan(int variants, int tuples, int surfaces, int rings, int n) {
    PrefilterPlan p{};
    p.q = p.Q = prefilter_lanes(n);
    const auto groups = [&] { return (variants + 256 / p.Q - 1) / (256 / p.Q); };
    while (p.Q < 256 && p.Q < n && int64_t(groups()) * tuples < 1024) p.Q *= 2;
    p.groups = groups();
    const size_t G = size_t(256 / p.Q);
    p.lds = G * size_t(surfaces | 1) * kPrefilterStepBytes +
            size_t(n / rings) * 2 * sizeof(float) + // the most spokes of a field
            G * size_t(prefilter_slots(n, p.q)) * (sizeof(float) + 1);
    return p;
}

} // namespace mko_internal
