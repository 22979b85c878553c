"""A context's growable buffers (csrc/sq8_buffers.h) on the CPU, against a stand-in for the runtime that records what is
allocated and freed: memory that a captured graph uses stays until the context goes."""
import os
import subprocess

from conftest import ROOT

CSRC = os.path.join(ROOT, "siliconed_amd", "csrc")
PROBE = r"""
#include "sq8_buffers.h"
#include <assert.h>
#include <set>
#include <stdio.h>
#include <stdlib.h>
static std::set<void *> live;
static bool captured = false, no_memory = false;
static int waits = 0;
extern "C" {
hipError_t hipMalloc(void **p, size_t bytes) {
    if (no_memory || captured) return hipErrorOutOfMemory;
    live.insert(*p = malloc(bytes));
    return hipSuccess;
}
hipError_t hipFree(void *p) { assert(live.erase(p) == 1); free(p); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { ++waits; return captured ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = captured ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
}
int main() {
    sq8::Buffer b{};
    sq8::SetAside *aside = nullptr;
    auto reserve = [&](size_t n) { return sq8::reserve(b, n, nullptr, aside); };
    assert(reserve(100) == hipSuccess && b.bytes == 100 && waits == 0);
    void *first = b.at;
    assert(reserve(50) == hipSuccess && b.at == first);                      // never shrinks
    assert(reserve(200) == hipSuccess && live.size() == 1 && waits == 1);    // grown: the old memory given back
    captured = true;
    assert(reserve(300) != hipSuccess && b.bytes == 200);                    // refused under capture, nothing lost
    assert(reserve(200) == hipSuccess);
    void *graphs = b.at;
    captured = false;
    assert(reserve(200) == hipSuccess && b.at == graphs);
    assert(reserve(400) == hipSuccess && b.at != graphs && live.count(graphs) == 1);  // grown: the graph's memory stays
    void *eager = b.at;
    assert(reserve(800) == hipSuccess && live.count(eager) == 0 && live.count(graphs) == 1);
    no_memory = true;
    assert(reserve(900) != hipSuccess && !b.at && b.bytes == 0);
    no_memory = false;
    captured = true;
    assert(reserve(0) == hipSuccess);
    captured = false;
    assert(reserve(10) == hipSuccess);
    sq8::release(b);
    sq8::release(aside);
    assert(live.empty() && !aside);
    puts("ok");
}
"""


def test_a_graphs_memory_outlives_growth(tmp_path):
    src, exe = str(tmp_path / "probe.cpp"), str(tmp_path / "probe")
    with open(src, "w") as f:
        f.write(PROBE)
    r = subprocess.run(["g++", "-std=c++17", "-g", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", CSRC, src, "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr
