// Launch shapes that follow from the sizes alone: plain host code, shared by the launches and the
// host layer.
#pragma once

#include <algorithm>
#include <cstdint>

namespace mko_internal {

// Most runs of one fd_jacobian launch: the kernel counts the tuples of every variant, 2 P + 1
// variants a run, in 32 bits, and a launch holds fewer than 2^32 threads (up to 256 a tuple; a
// tuple's variables go to several workgroups only where there are fewer than 4096 tuples).
inline int64_t fd_direct_runs(int variables, int64_t tuples) {
    const int64_t per_run = (2 * int64_t(variables) + 1) * tuples;
    return std::min(int64_t(0x7fffffff) / per_run, int64_t(0xffffffff) / (256 * tuples));
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

} // namespace mko_internal
