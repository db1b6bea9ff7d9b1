"""Transfers of states through pinned memory (csrc/ts_hostmem.cpp), built against a stand-in for the HIP
runtime whose device memory is the host's: every size arrives whole, with and without pinned memory and with
many CPUs or few.  Without pinned memory the transfers still work and leave no error behind for the next
call, and a process with few CPUs uses the runtime's own copy, which overlaps what one thread cannot."""
import os
import subprocess
import textwrap

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "turbostructred_amd", "csrc")

HIP = """
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>
typedef int hipError_t;
typedef struct stand_in_stream* hipStream_t;
typedef struct stand_in_event* hipEvent_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2, hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
inline thread_local int last_error = 0;
inline bool no_pinned = false, no_events = false;
inline std::atomic<int> copies{0}, pinned{0}, waits{0};
inline hipError_t done(int e) { if (e) last_error = e; return e; }
inline hipError_t hipGetLastError() { int e = last_error; last_error = 0; return e; }
inline hipError_t hipSetDevice(int) { return 0; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (no_pinned) return done(hipErrorOutOfMemory);
    *p = std::malloc(n); pinned++; return 0;
}
inline hipError_t hipHostFree(void* p) { std::free(p); pinned--; return 0; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (no_events) return done(hipErrorOutOfMemory);
    *e = (hipEvent_t)std::malloc(1); return 0;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return 0; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return 0; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return 0; }
inline hipError_t hipStreamSynchronize(hipStream_t) { waits++; return 0; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
    copies++; std::memcpy(d, s, n); return 0;
}
"""

MAIN = """
#include "ts_hostmem.hpp"
#include <cstdio>
#include <cstdint>
static int cpus;
extern "C" int get_nprocs() { return cpus; }   // what hardware_concurrency asks
#define REQUIRE(x) if (!(x)) { std::printf("line %d: %s\\n", __LINE__, #x); return 1; }
int main(int, char** argv) {
    cpus = std::atoi(argv[1]);
    no_pinned = std::atoi(argv[2]) == 1;
    no_events = std::atoi(argv[2]) == 2;
    REQUIRE(int(std::thread::hardware_concurrency()) == cpus);
    const size_t MB = size_t(1) << 20;
    for (size_t n : {size_t(8), 24 * MB - 8, 24 * MB, 64 * MB - 8, 64 * MB, 64 * MB + 4104, 97 * MB + 8}) {
        tsr::Staging st;
        std::vector<uint64_t> a(n / 8), b(n / 8), c(n / 8);
        for (size_t i = 0; i < a.size(); i++) a[i] = i * 0x9E3779B97F4A7C15u;
        copies = waits = 0;
        REQUIRE(st.to_device(b.data(), a.data(), n, 0, nullptr) == hipSuccess);
        const int up = copies.exchange(0);
        REQUIRE(up > 1 || waits == 0);   // the caller waits, once, for what follows the copy
        REQUIRE(st.to_host(c.data(), b.data(), n, 0, nullptr) == hipSuccess);
        const int down = copies.exchange(0);
        REQUIRE(a == b && a == c);
        REQUIRE(hipGetLastError() == hipSuccess);
        const bool threads = cpus >= 8 && !no_pinned && !no_events;
        REQUIRE((up > 1) == (threads && n >= 64 * MB));
        REQUIRE((down > 1) == (threads && n >= 24 * MB));
        st.release();
    }
    tsr::Staging st;
    for (int k = 0; k < 9; k++) {
        hipError_t e;
        char* p = st.take(4 * MB - 100, nullptr, &e);
        REQUIRE(p && e == hipSuccess);
        std::memset(p, k, 4 * MB - 100);
    }
    REQUIRE(hipGetLastError() == hipSuccess);
    st.release();
    REQUIRE(pinned == 0);
    std::printf("ok\\n");
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("hostmem")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "main.cpp").write_text(textwrap.dedent(MAIN))
    out = d / "hostmem"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-I", str(d), "-I", CSRC, "-o", str(out),
                           str(d / "main.cpp"), os.path.join(CSRC, "ts_hostmem.cpp")])
    return str(out)


@pytest.mark.parametrize("lacking", ["nothing", "pinned memory", "events"])
@pytest.mark.parametrize("cpus", [1, 4, 8, 64])
def test_transfers(program, cpus, lacking):
    which = {"nothing": 0, "pinned memory": 1, "events": 2}[lacking]
    r = subprocess.run([program, str(cpus), str(which)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
