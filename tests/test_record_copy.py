"""RecordCopy (ds2d_amd/csrc/record_copy.hpp) on the host, over a stand-in for
the HIP calls that it makes: copies happen when their event is waited for, and
the first wait takes half a second, as behind a time loop that is still
running.  The records arrive whole, and nothing spins meanwhile."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r'''
#pragma once
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>
typedef int hipError_t;
typedef void* hipStream_t;
struct Event { size_t upto = 0; };
typedef Event* hipEvent_t;
enum { hipMemoryTypeUnregistered = 0, hipMemoryTypeDevice = 2 };
struct hipPointerAttribute_t { int type; };
enum { hipSuccess = 0, hipEventDisableTiming = 2, hipHostMallocDefault = 0, hipMemcpyDeviceToHost = 2 };
struct Copy { void* d; const void* s; size_t n; };
inline std::vector<Copy> queue_;
inline const void* device_ = nullptr;
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    a->type = p == device_ ? hipMemoryTypeDevice : hipMemoryTypeUnregistered;
    return hipSuccess;
}
inline size_t done_ = 0;
inline double busy_s = 0;
inline hipError_t reach(size_t upto) {
    if (busy_s > 0) std::this_thread::sleep_for(std::chrono::duration<double>(busy_s));
    busy_s = 0;
    for (; done_ < upto; ++done_) memcpy(queue_[done_].d, queue_[done_].s, queue_[done_].n);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new Event; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
    queue_.push_back({d, s, n});
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { e->upto = queue_.size(); return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t e) { return reach(e->upto); }
inline hipError_t hipStreamSynchronize(hipStream_t) { return reach(queue_.size()); }
'''

SHIM = r'''
#include <ctime>
#include "record_copy.hpp"
// copies straight to the caller's memory, of records whose z lies on the device
extern "C" int direct(size_t n, float* z, const float* dz, float* x, const float* dx) {
    queue_.clear();
    done_ = 0;
    device_ = z;
    ds2d::RecordCopy rc;
    const int e = rc.fetch(nullptr, n, z, dz, x, dx);
    device_ = nullptr;
    int k = 0;
    for (const Copy& c : queue_) k += c.n == 4 * n && (c.d == z || c.d == x);
    return e == hipSuccess && k == (int)queue_.size() ? k : -1;
}
// seconds of processor time of all threads
extern "C" double fetch(size_t n, float* z, const float* dz, float* x, const float* dx, double busy) {
    busy_s = busy;
    ds2d::RecordCopy rc;
    const clock_t t = clock();
    if (rc.fetch(nullptr, n, z, dz, x, dx) != hipSuccess) return -1;
    return (double)(clock() - t) / CLOCKS_PER_SEC;
}
'''


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("copy")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "shim.cpp").write_text(SHIM)
    so = d / "libcopy.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-pthread", "-I", str(d), "-I",
                    os.path.join(ROOT, "ds2d_amd", "csrc"), str(d / "shim.cpp"), "-o", str(so)], check=True)
    return C.CDLL(str(so))


@pytest.fixture(scope="module")
def fetch(lib):
    lib.fetch.restype = C.c_double
    fp = C.POINTER(C.c_float)
    lib.fetch.argtypes = [C.c_size_t, fp, fp, fp, fp, C.c_double]

    def run(n, both, busy):
        src = np.arange(2 * n, dtype=np.float32).reshape(2, n)
        dst = np.zeros((2, n), np.float32)
        p = lambda a: a.ctypes.data_as(fp)
        cpu = lib.fetch(n, p(dst[0]), p(src[0]), p(dst[1]) if both else None, p(src[1]), busy)
        assert np.array_equal(dst[0], src[0]) and np.array_equal(dst[1], src[1] if both else 0 * src[1])
        return cpu
    return run


# one piece, two and many of 4 MB with a rest, and less than is staged
@pytest.mark.parametrize("n,both", [(1000, True), (1 << 20, True), (2100001, False), (5 << 20, True), (3000017, True)])
def test_records_arrive_whole(fetch, n, both):
    assert fetch(n, both, 0.0) >= 0


def test_nothing_spins_while_the_device_computes(fetch):
    """16 MB take some 20 ms of processor time to copy into fresh pages; three threads that spin for half a
    second would take 1.5 s."""
    cpu = fetch(2 << 20, True, 0.5)
    print(f"{cpu:.3f} s of processor time")
    assert cpu < 0.25


def test_memory_that_hip_knows_is_left_to_it(lib):
    """No thread writes to a destination on the device: one copy for each component, whole."""
    n = 3 << 20
    src = np.arange(2 * n, dtype=np.float32).reshape(2, n)
    dst = np.zeros((2, n), np.float32)
    p = lambda a: a.ctypes.data_as(C.POINTER(C.c_float))
    assert lib.direct(C.c_size_t(n), p(dst[0]), p(src[0]), p(dst[1]), p(src[1])) == 2
    assert np.array_equal(dst, src)
