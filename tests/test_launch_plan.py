"""Launch shapes at the sizes where 32-bit indices and grids end, on the CPU: a program built against
the internal headers asks the shared rules (launch_plan.hpp) and the library's entry points, which
refuse a call that is too large before they touch a device."""

import os
import subprocess

from mikroptim_amd import engine

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run_program(tmp_path, text):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(text)
    libdir = os.path.dirname(engine.LIB_PATH)
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "mikroptim_amd", "csrc"), str(src), "-o", str(exe),
                    "-L", libdir, "-l:" + os.path.basename(engine.LIB_PATH), "-Wl,-rpath," + libdir,
                    "-Wl,-rpath-link,/opt/rocm/lib"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr


FD_RUNS = r"""
#include "internal.hpp"
#include "launch_plan.hpp"
#include "mikroptim_hip.h"
#include <cstdio>
#include <vector>
using namespace mko_internal;

// the entry point on `runs` runs of a batch of F fields, L wavelengths and P thicknesses of one
// surface: device arrays are never read, since a refused call launches nothing
int call(int F, int L, int P, int64_t runs) {
    std::vector<uint8_t> type{0, 2, 2}, mode(F, MKO_PUPIL_FULL);
    std::vector<double> one(64, 1.0);
    std::vector<int32_t> kind(P, MKO_VAR_THICKNESS), surface(P, 1);
    mko_batch b{};
    b.variants = int32_t(runs * (2 * P + 1));
    b.surfaces = 3;
    b.wavelengths = L;
    b.fields = F;
    b.reference_wavelength_nm = 550.0;
    b.type = type.data();
    b.pupil_mode = mode.data();
    b.wavelength_weight = b.field_weight = one.data();
    mko_residual_settings s{};
    s.rings = s.spokes = 1;
    s.failure = MKO_FAILURE_HARD;
    mko_variables v{};
    v.count = P;
    v.type = kind.data();
    v.batch_surface = surface.data();
    return fd_jacobian(&b, &s, &v, int(runs), nullptr, nullptr, nullptr, nullptr, nullptr, 1,
                       nullptr);
}

int main() {
    int fails = 0;
    for (int F : {1, 5, 32})
        for (int L : {1, 7, 32})
            for (int P = 1; P <= 320; ++P) {
                const int64_t T = F * L, per = (2 * P + 1) * T, n = fd_direct_runs(P, T);
                // the last tuple's index, the variants and the threads of the launch fit
                const bool fits = n >= 1 && n * per - 1 < (int64_t(1) << 31) &&
                                  n * T * 256 < (int64_t(1) << 32);
                const bool most = (n + 1) * per > 0x7fffffff ||
                                  (n + 1) * T * 256 > int64_t(0xffffffff);
                if (!fits || !most) {
                    std::printf("F %d L %d P %d: %ld runs\n", F, L, P, long(n));
                    ++fails;
                }
                if (P != 16 && P != 127) continue;
                // the first refused number of runs, and one with a 32-bit product that wraps
                for (int64_t runs : {n + 1, (int64_t(1) << 31) / (2 * P + 1) - 1}) {
                    if (runs <= n) continue;
                    const int rc = call(F, L, P, runs);
                    if (rc != MKO_ERR_INVALID) {
                        std::printf("F %d L %d P %d runs %ld: %d\n", F, L, P, long(runs), rc);
                        ++fails;
                    }
                }
            }
    return fails != 0;
}
"""


def test_fd_jacobian_refuses_more_tuples_than_it_can_count(tmp_path):
    run_program(tmp_path, FD_RUNS)


GRAM_PARTS = r"""
#include "launch_plan.hpp"
#include <cstdio>
using namespace mko_internal;

int main() {
    int fails = 0;
    for (int P = 1; P <= 127; ++P)
        for (int runs = 1; runs <= 600; ++runs) {
            const GramPlan p = gram_plan(P, runs);
            // every unit belongs to a part and every part has one; a wave's units fit the
            // accumulators of the kernels launched (2 of 8 waves up to 64 variables, else 5)
            if (p.parts < 1 || p.upp < 1 || (p.parts - 1) * p.upp >= p.units ||
                p.parts * p.upp < p.units || p.upp > 8 * (P <= 64 ? 2 : 5)) {
                if (++fails <= 10)
                    std::printf("P %d runs %d: %d units, %d parts of %d\n", P, runs, p.units,
                                p.parts, p.upp);
            }
        }
    return fails != 0;
}
"""


def test_gram_parts_cover_the_units_and_none_is_empty(tmp_path):
    run_program(tmp_path, GRAM_PARTS)


def test_gram_without_variables_has_nothing_to_do():
    lib = engine.library()
    assert lib.mko_gram_device(None, None, 3, 0, 40, None, None, None) == 0
    assert lib.mko_gram_device(None, None, 3, -1, 40, None, None, None) != 0


PREFILTER_LDS = r"""
#include "launch_plan.hpp"
#include <cstdio>
using namespace mko_internal;

int main() {
    int fails = 0;
    for (int V : {1, 3, 100, 2001, 20000})
        for (int T : {1, 9, 35, 1024})
            for (int S : {2, 3, 25, 64})
                for (int rings = 1; rings <= 16; ++rings)
                    for (int M = 1; rings * M <= 2048; ++M) {
                        const PrefilterPlan p = prefilter_plan(V, T, S, rings, rings * M);
                        // beside it 1 KB of static LDS; 64 KB always fit a workgroup
                        const bool fits = p.lds + 1024 <= 65536 &&
                            p.lds >= size_t(256 / p.Q) * (S * kPrefilterStepBytes +
                                                          size_t(rings) * M * 5) + size_t(M) * 8;
                        const bool lanes = p.q >= 8 && p.q <= p.Q && p.Q <= 256 &&
                            int64_t(p.groups) * (256 / p.Q) >= V &&
                            int64_t(p.groups - 1) * (256 / p.Q) < V;
                        if ((!fits || !lanes) && ++fails <= 10)
                            std::printf("V %d T %d S %d rings %d spokes %d: q %d Q %d lds %zu\n", V,
                                        T, S, rings, M, p.q, p.Q, p.lds);
                    }
    return fails != 0;
}
"""


def test_prefilter_lds_holds_the_samples_of_the_largest_tuple(tmp_path):
    run_program(tmp_path, PREFILTER_LDS)
