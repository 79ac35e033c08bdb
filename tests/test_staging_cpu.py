"""Downloads (brownian_amd/csrc/staging.h) when an allocation or a thread cannot
be had: the copies are whole or the call says that they are not, and the process
goes on.  The HIP calls are stood in for by host memory."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HARNESS = r"""
#include <dlfcn.h>
#include <pthread.h>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include "staging.h"

// the n-th allocation or thread start from when they are set fails
static std::atomic<long> fail_alloc{0}, fail_thread{0};
static void *take(std::size_t n) {
    if (fail_alloc.load() > 0 && fail_alloc.fetch_sub(1) == 1) return nullptr;
    return std::malloc(n ? n : 1);
}
void *operator new(std::size_t n) {
    void *p = take(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    if (fail_thread.load() > 0 && fail_thread.fetch_sub(1) == 1) return 11;  // EAGAIN
    static auto real = (decltype(&pthread_create))dlsym(RTLD_NEXT, "pthread_create");
    return real(t, a, f, arg);
}
extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = take(n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)take(1); return *e ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
}
namespace bw {
void launch_pack(const PackSegs &s, int *dst, hipStream_t) {
    for (int q = 0; q < s.n; q++) std::memcpy(dst + s.off[q], s.src[q], 4 * (size_t)(s.off[q + 1] - s.off[q]));
}
}
int main(int, char **argv) {
    const size_t n = (size_t)std::atol(argv[3]);
    std::vector<int> a(n), b(n, -1), c(n / 3), d(n / 3, -1);
    for (size_t i = 0; i < n; i++) a[i] = (int)(i * 2654435761u);
    for (size_t i = 0; i < c.size(); i++) c[i] = (int)(i * 40503u + 1);
    bool whole = true;
    bw::Staging st;
    for (int pass = 0; pass < 2; pass++) {  // the second without failures
        fail_alloc = pass ? 0 : std::atol(argv[1]);
        fail_thread = pass ? 0 : std::atol(argv[2]);
        std::fill(b.begin(), b.end(), -1);
        std::fill(d.begin(), d.end(), -1);
        const bw::StageSeg seg[] = {{b.data(), a.data(), 4 * n}, {nullptr, a.data(), 4 * n}, {d.data(), c.data(), 4 * c.size()}};
        const hipError_t e = st.download(seg, 3, nullptr);
        if (e != hipSuccess) return pass ? 2 : 3;
        whole = whole && a == b && c == d;
    }
    std::puts(whole ? "whole" : "not whole");
    return whole ? 0 : 1;
}
"""


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    d = tmp_path_factory.mktemp("staging")
    src, exe = d / "h.cpp", d / "h"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "brownian_amd", "csrc"), str(src), "-o", str(exe), "-pthread", "-ldl"], check=True)
    return str(exe)


@pytest.mark.parametrize("ints", [1000, 3_000_000, 12_000_001])
def test_downloads_without_failures(harness, ints):
    assert subprocess.run([harness, "0", "0", str(ints)], timeout=60).returncode == 0


@pytest.mark.parametrize("ints", [1000, 3_000_000, 12_000_001])
def test_downloads_when_memory_runs_out(harness, ints):
    for n in range(1, 40):
        assert subprocess.run([harness, str(n), "0", str(ints)], timeout=60).returncode == 0, n


def test_downloads_when_threads_cannot_be_started(harness):
    for n in range(1, 9):
        assert subprocess.run([harness, "0", str(n), "12000001"], timeout=60).returncode == 0, n
