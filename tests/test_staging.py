"""The transfers through pinned slots (staging.hpp) against a stand-in for the HIP calls they use, on
the CPU: device memory is host memory, and a copy or an event takes place only when its event or
the stream is waited for, as late as an asynchronous one may. What was handed in must then still be
what was handed in."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
using hipError_t = int;
using hipStream_t = void*;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum { hipEventDisableTiming = 2, hipHostMallocDefault = 0 };
struct Event { size_t at = 0; };
using hipEvent_t = Event*;
inline std::deque<std::function<void()>> queue;
inline size_t issued = 0, passed = 0;
inline void pass(size_t upto) {
    for (; passed < upto; ++passed) { queue.front()(); queue.pop_front(); }
}
inline const char* hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
    queue.push_back([=] { std::memcpy(d, s, n); });
    ++issued;
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { pass(issued); return hipSuccess; }
inline hipError_t hipDeviceSynchronize() { pass(issued); return hipSuccess; }
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, int) {
    pass(issued);
    std::memcpy(d, s, n);
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { *e = new Event; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { e->at = issued; return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t e) { pass(e->at); return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) { *p = std::malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
"""

PROGRAM = r"""
#include "staging.hpp"
#include <cstdint>
#include <cstdio>
using mko_host::Staging;

std::vector<uint8_t> pattern(size_t n, int seed) {
    std::vector<uint8_t> v(n);
    for (size_t i = 0; i < n; ++i) v[i] = uint8_t((i * 2654435761u) >> 13) ^ uint8_t(seed * 37);
    return v;
}

int main() {
    int fails = 0;
    Staging io;
    // arrays around the slots' size, one after another; each source is overwritten at once
    const size_t M = size_t(1) << 20;
    int seed = 0;
    for (size_t n : {size_t(1), size_t(8), M - 8, M, M + 1, 2 * M - 1, 2 * M, 2 * M + 3, 5 * M + 1,
                     size_t(16), 11 * M}) {
        const std::vector<uint8_t> want = pattern(n, ++seed);
        std::vector<uint8_t> source = want, dev(n), back(n);
        io.in(dev.data(), source.data(), n);
        std::fill(source.begin(), source.end(), uint8_t(0));
        io.out({{back.data(), dev.data(), n}});
        if (back != want) {
            std::printf("%zu bytes: not what was handed in\n", n);
            ++fails;
        }
    }
    return fails != 0;
}
"""


def test_in_takes_the_source_as_it_is_at_the_call(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    src, exe = tmp_path / "staging.cpp", tmp_path / "staging"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-I",
                    str(tmp_path), "-I", os.path.join(ROOT, "mikroptim_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
