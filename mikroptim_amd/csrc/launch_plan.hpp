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

} // namespace mko_internal
