"""The chunked copies of dnsmc_amd/csrc/transfer.h on the CPU: the header compiled
by g++ against a few lines that stand for the HIP runtime.  Rows and jobs around
the 1 MiB chunks and the 4 MiB from which threads are used arrive byte for byte,
nothing outside them is touched, a failed copy is reported, and an allocation
that fails anywhere in a copy neither throws nor ends the process (the caller is
a C function)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r'''
#pragma once
#include <stdlib.h>
#include <string.h>
#include <atomic>
typedef int hipError_t;
typedef void* hipStream_t;
typedef void* hipEvent_t;
enum { hipSuccess = 0, hipErrorUnknown = 999, hipMemcpyDeviceToHost = 2, hipMemcpyHostToDevice = 1, hipHostMallocDefault = 0,
       hipEventDisableTiming = 2, hipMemoryTypeUnregistered = 0 };
struct hipPointerAttribute_t { int type; };
inline std::atomic<long> fail_copy{-1};
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) { a->type = hipMemoryTypeUnregistered; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) { *p = malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { *e = nullptr; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t)
{
    if (fail_copy >= 0 && fail_copy-- == 0) return hipErrorUnknown;
    memcpy(d, s, n);
    return hipSuccess;
}
'''

MAIN = r'''
#include <new>
#include <cstdio>
#include <vector>
#include "transfer.h"
static std::atomic<long> fail_new{-1};
void* operator new(size_t n)
{
    if (fail_new >= 0 && fail_new-- == 0) throw std::bad_alloc();
    void* p = malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
using namespace dn;
static int bad(const char* what, size_t n) { printf("%s %zu\n", what, n); return 1; }
static int blocks(std::vector<size_t> sizes)
{
    HostPipe pipe;
    size_t total = 0;
    for (size_t s : sizes) total += s;
    std::vector<char> dev(total + 1), host(total + 2 * sizes.size() + 1, 77);
    for (size_t i = 0; i < total; ++i) dev[i] = (char)(i * 2654435761u >> 13);
    HostRows jobs[4];
    size_t d = 0, h = 1;
    for (size_t k = 0; k < sizes.size(); ++k) {
        jobs[k] = host_block(dev.data() + d, host.data() + h, sizes[k]);
        d += sizes[k];
        h += sizes[k] + 1;
    }
    for (int pass = 0; pass < 2; ++pass) {
        if (pipe.run(0, nullptr, jobs, (int)sizes.size()) != hipSuccess) return bad("run", total);
        for (size_t k = 0; k < sizes.size(); ++k) {
            if (memcmp(jobs[k].host, jobs[k].dev, sizes[k])) return bad("bytes", total);
            if (jobs[k].host[-1] != 77 || jobs[k].host[sizes[k]] != 77) return bad("outside", total);
        }
    }
    return 0;
}
static int rows(int n0, int n1, int n2)   // two arrays with ghost layers, as the Fortran results
{
    HostPipe pipe;
    const size_t ne = (size_t)n0 * n1 * n2, g = (size_t)(n0 + 2) * (n1 + 2) * (n2 + 2);
    std::vector<float> dev(2 * ne), host(2 * g, -7.f);
    for (size_t i = 0; i < 2 * ne; ++i) dev[i] = (float)i;
    HostRows j = host_block(dev.data(), host.data() + 1 + (n0 + 2) + (size_t)(n0 + 2) * (n1 + 2), 2 * ne * 4);
    j.row = (size_t)n0 * 4;
    j.n1 = n1;
    j.n2 = n2;
    j.p1 = (n0 + 2) * 4;
    j.p2 = j.p1 * (n1 + 2);
    j.p3 = g * 4;
    if (pipe.run(0, nullptr, &j, 1) != hipSuccess) return bad("run rows", ne);
    size_t inside = 0;
    for (int a = 0; a < 2; ++a)
        for (int z = 0; z < n2 + 2; ++z)
            for (int y = 0; y < n1 + 2; ++y)
                for (int x = 0; x < n0 + 2; ++x) {
                    const bool in = x > 0 && x <= n0 && y > 0 && y <= n1 && z > 0 && z <= n2;
                    const float want = in ? (float)inside++ : -7.f;
                    if (host[a * g + ((size_t)z * (n1 + 2) + y) * (n0 + 2) + x] != want) return bad("rows", ne);
                }
    return 0;
}
int main()
{
    const size_t C = HostPipe::kChunk, P = HostPipe::kParallel;
    for (size_t n : {(size_t)0, (size_t)1, C - 1, C, C + 1, 2 * C, 2 * C + 1, 3 * C + 5, P - 1, P, P + 1, 9 * C + 3})
        if (blocks({n})) return 1;
    if (blocks({C, 0, C + 1, 3}) || blocks({P, 1, 0, P - 1}) || blocks({5, 7, 11, 13}) || blocks({0, 0})) return 1;
    if (rows(1, 1, 1) || rows(45, 61, 37) || rows(513, 257, 4) || rows(512, 256, 4) || rows(384, 64, 32)) return 1;
    // the k-th copy fails: reported, and the next call works
    for (long k = 0; k < 24; ++k) {
        std::vector<char> dev(9 * C), host(9 * C);
        HostPipe pipe;
        const HostRows j = host_block(dev.data(), host.data(), 9 * C);
        fail_copy = k;
        const hipError_t e = pipe.run(0, nullptr, &j, 1);
        fail_copy = -1;
        if ((e != hipSuccess) != (k < 9)) return bad("failed copy", k);
        if (pipe.run(0, nullptr, &j, 1) != hipSuccess) return bad("after a failed copy", k);
    }
    // the k-th allocation fails: the copy is made all the same
    for (long k = 0; k < 16; ++k) {
        std::vector<char> dev(9 * C, 3), host(9 * C, 0);
        HostPipe pipe;
        const HostRows j = host_block(dev.data(), host.data(), 9 * C);
        fail_new = k;
        const hipError_t e = pipe.run(0, nullptr, &j, 1);
        fail_new = -1;
        if (e != hipSuccess || memcmp(dev.data(), host.data(), 9 * C)) return bad("failed allocation", k);
    }
    printf("ok\n");
    return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_transfer_on_the_host(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "transfer")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-I", str(tmp_path), "-I", os.path.join(ROOT, "dnsmc_amd", "csrc"),
                    str(tmp_path / "main.cpp"), "-o", exe, "-pthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout, r.stderr)
