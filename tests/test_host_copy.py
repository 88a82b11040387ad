"""The downloads' ring (tlbm_amd/csrc/host_copy.cpp) on the host, against a
stand-in for the HIP runtime that copies at once, knows which device an event,
a stream and a thread belong to, and fails on demand."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400, hipErrorUnknown = 999 };
enum { hipHostMallocPortable = 1, hipEventDisableTiming = 2, hipMemcpyDeviceToHost = 2 };
struct FakeEvent { int device; };
struct FakeStream { int device; };
typedef FakeEvent *hipEvent_t;
typedef FakeStream *hipStream_t;
inline thread_local int t_device = 0;
inline std::atomic<int> pinned{0}, events{0}, made{0}, copies{0}, fail_copy{-1}, fail_sync{-1}, syncs{0};
inline std::atomic<bool> no_pinned{false};
inline hipError_t hipGetDevice(int *d) { *d = t_device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { t_device = d; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (no_pinned) return hipErrorOutOfMemory;
    *p = std::malloc(n); ++pinned; ++made; return hipSuccess;
}
inline hipError_t hipHostFree(void *p) { std::free(p); --pinned; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new FakeEvent{t_device}; ++events; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; --events; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return e->device == s->device ? hipSuccess : hipErrorInvalidHandle; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return syncs++ == fail_sync ? hipErrorUnknown : hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) {
    if (copies++ == fail_copy) return hipErrorUnknown;
    std::memcpy(d, s, n);
    return hipSuccess;
}
"""

PROBE = r"""
#include <cstdio>
#include <vector>
#include "host_copy.h"
using namespace tlbm;
template <class T>
static hipError_t run(size_t n0, size_t n1, int device, bool &same) {
    FakeStream stream{device};
    std::vector<T> dev(n0 + n1);
    for (size_t i = 0; i < dev.size(); ++i) dev[i] = T(i % 9973) * T(0.25);
    std::vector<double> a(n0, -1.0), b(n1, -1.0);
    const char *p = reinterpret_cast<const char *>(dev.data());
    const CopyPart parts[2] = {{p, a.data(), n0}, {p + n0 * sizeof(T), b.data(), n1}};
    const hipError_t e = copy_to_host(parts, 2, sizeof(T) == 4, &stream, device);
    same = true;
    for (size_t i = 0; i < n0; ++i) same = same && a[i] == double(dev[i]);
    for (size_t i = 0; i < n1; ++i) same = same && b[i] == double(dev[n0 + i]);
    return e;
}
#define EXPECT(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); ++bad; } } while (0)
int main() {
    int bad = 0;
    bool same;
    const size_t n = 1500007;  // ragged: a last chunk of its own in either part
    host_copy_retain();
    // a lattice of another device than the calling thread's; its ring is kept
    for (int k = 0; k < 3; ++k) {
        EXPECT(run<float>(n, n / 3, 1, same) == hipSuccess && same && t_device == 0);
        EXPECT(run<double>(3 * n, n, 1, same) == hipSuccess && same && t_device == 0);
    }
    EXPECT(made == 1 && copies > 100);
    EXPECT(run<float>(n, n / 3, 0, same) == hipSuccess && same);
    EXPECT(made == 2);
    // short copies take no ring
    EXPECT(run<float>(1000, 17, 2, same) == hipSuccess && same && made == 2);
    // no pinned memory left: copied directly
    no_pinned = true;
    EXPECT(run<float>(n, n / 3, 3, same) == hipSuccess && same);
    EXPECT(run<double>(3 * n, n, 3, same) == hipSuccess && same);
    no_pinned = false;
    // a copy or a wait that fails, early, late and past the first round of
    // slots: its error comes back, and the ring serves the next call
    for (int at : {0, 3, 16, 20}) {
        copies = 0, fail_copy = at;
        EXPECT(run<double>(3 * n, n, 1, same) == hipErrorUnknown);
        fail_copy = -1;
        syncs = 0, fail_sync = at;
        EXPECT(run<double>(3 * n, n, 1, same) == hipErrorUnknown);
        fail_sync = -1;
        EXPECT(run<double>(3 * n, n, 1, same) == hipSuccess && same);
    }
    EXPECT(made == 2 && pinned == 2);
    host_copy_release();
    EXPECT(pinned == 0 && events == 0);
    std::printf("bad %d\n", bad);
}
"""


def test_ring_copies_fails_and_falls_back():
    with tempfile.TemporaryDirectory() as tmp:
        os.mkdir(os.path.join(tmp, "hip"))
        for name, text in (("hip/hip_runtime.h", RUNTIME), ("probe.cpp", PROBE)):
            with open(os.path.join(tmp, name), "w") as fh:
                fh.write(text)
        src = os.path.join(ROOT, "tlbm_amd", "csrc")
        exe = os.path.join(tmp, "probe")
        subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", tmp, "-I", src, os.path.join(tmp, "probe.cpp"),
                        os.path.join(src, "host_copy.cpp"), "-o", exe], check=True)
        out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=60).stdout
    assert out == "bad 0\n", out
