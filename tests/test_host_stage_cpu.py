"""The pinned ring of large copies (host_stage.hpp) on the CPU, against a stand-in
for the runtime whose transfers arrive later: a batch may be made by a thread
that may use every CPU and copied by one bound to a single CPU."""
import subprocess
from pathlib import Path

import pytest

HEADER = Path(__file__).resolve().parent.parent / "swe-ppm_amd" / "csrc" / "host_stage.hpp"

# transfers take place when an event after them is queried for the third time,
# or when the stream is synchronised
RUNTIME = r"""
#pragma once
#include <cstdlib>
#include <cstring>
#include <functional>
#include <deque>
enum hipError_t { hipSuccess = 0, hipErrorNotReady = 1, hipErrorInvalidValue = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
struct hipPointerAttribute_t { hipMemoryType type; };
struct Stream { std::deque<std::function<void()>> work; size_t done = 0; };
struct Event { Stream* stream = nullptr; size_t at = 0; int asked = 0; };
using hipStream_t = Stream*;
using hipEvent_t = Event*;
inline void drain(Stream* s, size_t upTo) { for (; s->done < upTo; ++s->done) s->work[s->done](); }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new Event; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    st->work.push_back([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) { *e = Event{st, st->work.size(), 0}; return hipSuccess; }
inline hipError_t hipEventQuery(hipEvent_t e) {
    if (++e->asked < 3) return hipErrorNotReady;
    drain(e->stream, e->at);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t st) { drain(st, st->work.size()); return hipSuccess; }
"""

PROGRAM = r"""
#include "%s"
#include <cstdio>
#include <vector>
int main(int, char** argv) {
    const int cpus = std::atoi(argv[1]);
    const bool toDevice = std::atoi(argv[2]) != 0;
    const size_t bytes = (toDevice ? swe::HostStage::kLeastToDevice : swe::HostStage::kLeastToHost) + 4099;
    swe::HostStage stage;
    stage.create(bytes);
    cpu_set_t all, few;
    sched_getaffinity(0, sizeof(all), &all);
    CPU_ZERO(&few);
    for (int c = 0, n = 0; c < CPU_SETSIZE && n < cpus; ++c)
        if (CPU_ISSET(c, &all)) CPU_SET(c, &few), ++n;
    sched_setaffinity(0, sizeof(few), &few);
    std::vector<char> from(bytes), to(bytes, 1);
    for (size_t i = 0; i < bytes; ++i) from[i] = (char)(i * 7 + (i >> 11));
    const size_t cut = bytes / 3;
    char *host = toDevice ? from.data() : to.data(), *dev = toDevice ? to.data() : from.data();
    const swe::HostCopy copies[2] = {{host, dev, cut}, {host + cut, dev + cut, bytes - cut}};
    Stream stream;
    const hipError_t e = toDevice ? stage.to_device(copies, 2, &stream) : stage.to_host(copies, 2, &stream);
    hipStreamSynchronize(&stream);
    stage.destroy();
    return e != hipSuccess ? 2 : std::memcmp(from.data(), to.data(), bytes) ? 3 : 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_stage")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (d / "main.cpp").write_text(PROGRAM % HEADER)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", f"-I{d}", "-o", str(d / "main"), str(d / "main.cpp")],
                   check=True)
    return d / "main"


@pytest.mark.parametrize("to_device", [0, 1])
@pytest.mark.parametrize("cpus", [1, 2, 64])
def test_copy_ends_whatever_the_calling_thread_may_use(program, cpus, to_device):
    assert subprocess.run([str(program), str(cpus), str(to_device)], timeout=30).returncode == 0
