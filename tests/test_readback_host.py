"""mm_readback.h built for the host with stand-ins for the HIP calls: its pieces,
its pool and what it does when the pool or its threads cannot be had.  The GPU side
is in test_gpu_readback.py and test_gpu_readback_shared.py."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "micromagnum_amd", "csrc")

HIP = r"""
#pragma once
#include <cstdlib>
#include <cstring>
#include <stdexcept>
typedef int hipStream_t;
typedef int *hipEvent_t;
enum { hipSuccess, hipHostMallocDefault, hipEventDisableTiming, hipMemcpyDeviceToHost };
extern int live, fail_alloc_at, fail_copy, allocs, device;
inline int hipGetDevice(int *d) { *d = device; return 0; }
inline int hipGetLastError() { return 0; }
inline int hipHostMalloc(void **p, size_t n, int)
{
    if (++allocs == fail_alloc_at) return 2;
    *p = malloc(n);
    ++live;
    return 0;
}
inline int hipHostFree(void *p) { free(p); --live; return 0; }
inline int hipEventCreateWithFlags(hipEvent_t *e, int) { *e = new int; ++live; return 0; }
inline int hipEventDestroy(hipEvent_t e) { delete e; --live; return 0; }
inline int hipEventRecord(hipEvent_t, hipStream_t) { return 0; }
inline int hipEventSynchronize(hipEvent_t) { return 0; }
inline int hipStreamSynchronize(hipStream_t) { return 0; }
inline int hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t)
{
    if (fail_copy) return 1;
    memcpy(d, s, n);
    return 0;
}
#define MM_HIP(x) do { if ((x) != 0) throw std::runtime_error(#x); } while (0)
"""

MAIN = r"""
#include <hip/hip_runtime.h>
#include "mm_readback.h"
#include <cstdio>
int live, fail_alloc_at, fail_copy, allocs, device;
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
template <typename T> static bool same(const std::vector<double> &d, const std::vector<T> &s)
{
    for (size_t i = 0; i < s.size(); ++i)
        if (d[i] != (double)s[i]) return false;
    return true;
}
template <typename T> static int whole(size_t n)
{
    std::vector<T> src(n);
    for (size_t i = 0; i < n; ++i) src[i] = (T)(i % 1000003) * (T)0.5;
    {   // two owners, two threads each, at the same time
        StateReader a, b;
        std::vector<std::vector<double>> dst(4, std::vector<double>(n));
        std::vector<int> ok(4);
        std::vector<std::thread> t;
        for (int c = 0; c < 4; ++c)
            t.emplace_back([&, c] { ok[c] = (c & 1 ? a : b).read(dst[c].data(), src.data(), n, 0); });
        for (auto &x : t) x.join();
        for (int c = 0; c < 4; ++c) CHECK(ok[c] && same(dst[c], src));
        CHECK(live == 2 * Readback::NBUF);  // one set for both owners
        device = 1;
        StateReader other;
        CHECK(other.read(dst[0].data(), src.data(), n, 0) && live == 4 * Readback::NBUF);
        device = 0;
    }
    CHECK(live == 0);  // gone with the last owner
    for (int at = 1; at <= Readback::NBUF; ++at) {
        std::vector<double> d(n);
        StateReader a, b;
        allocs = 0;
        fail_alloc_at = at;
        CHECK(!a.read(d.data(), src.data(), n, 0) && live == 0);
        fail_alloc_at = 0;
        CHECK(!a.read(d.data(), src.data(), n, 0) && live == 0);  // not tried again
        CHECK(b.read(d.data(), src.data(), n, 0) && same(d, src));
    }
    {
        std::vector<double> d(n);
        StateReader a;
        fail_copy = 1;
        CHECK(!a.read(d.data(), src.data(), n, 0) && live == 0);
        fail_copy = 0;
    }
    return 0;
}
int main()
{
    for (size_t n : {(size_t)1, (size_t)262144, (size_t)(4 * 524288 + 1), (size_t)5000011})
        if (whole<float>(n) || whole<double>(n)) return 1;
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_pieces_pool_and_failures(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I", str(tmp_path), "-I", CSRC,
                    str(tmp_path / "main.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
