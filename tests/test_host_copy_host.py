"""State out to host arrays (csrc/ttsh_hostcopy.h) on the CPU: the HIP calls it
makes are stood in for by a few lines that copy at once and keep count, and the
whole is built with AddressSanitizer and UndefinedBehaviorSanitizer.  Checked are
the values, and which pieces go through the ring and which are left to a plain
copy."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bacterial-droplet_amd", "csrc")

STUB = r"""
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum { hipEventDisableTiming = 2, hipHostMallocPortable = 1 };
typedef void* hipStream_t;
typedef void* hipEvent_t;
struct hipPointerAttribute_t { hipMemoryType type; int device; };
inline std::mutex g_mu;
inline std::map<const char*, size_t> g_pinned;
inline size_t g_pinned_bytes = 0, g_allocs = 0;
inline std::atomic<size_t> g_async{0}, g_looked{0};
inline bool g_no_memory = false;
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_no_memory) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    g_pinned[(char*)*p] = n;
    g_pinned_bytes += n;
    ++g_allocs;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p)
{
    std::lock_guard<std::mutex> lk(g_mu);
    g_pinned_bytes -= g_pinned[(char*)p];
    g_pinned.erase((char*)p);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    std::lock_guard<std::mutex> lk(g_mu);
    ++g_looked;
    auto it = g_pinned.upper_bound((const char*)p);
    const bool in = it != g_pinned.begin() && (--it, (const char*)p < it->first + it->second);
    a->type = in ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = e; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    ++g_async;
    return hipSuccess;
}
"""

DRIVER = r"""
#include "ttsh_hostcopy.h"
#include <cstdio>
using namespace ttsh;
#define CHECK(c) do { if (!(c)) { std::printf("failed: %s (line %d)\n", #c, __LINE__); return 1; } } while (0)

// seven fields of n floats to dst, each `stride` bytes after the one before
static std::vector<HostPiece> fields(const std::vector<float>& src, size_t n, char* dst, size_t stride)
{
    std::vector<HostPiece> p;
    for (int f = 0; f < 7; ++f) p.push_back(HostPiece{src.data() + f * n, dst + f * stride, n});
    return p;
}

int main()
{
    const size_t n = 400000;  // 11 MB of state
    std::vector<float> src(7 * n), a(7 * n);
    std::vector<double> b(7 * n);
    for (size_t i = 0; i < src.size(); ++i) src[i] = (float)(i % 100003) - 0.25f;
    {
        HostCopier hc;
        // pageable: everything through the ring
        auto p = fields(src, n, (char*)a.data(), 4 * n);
        CHECK(hc.copy(p, false, nullptr) == hipSuccess && p.empty() && g_allocs == 1);
        CHECK(g_pinned_bytes <= (size_t)16 << 20);  // a first read of a small state pins a small ring
        CHECK(std::memcmp(a.data(), src.data(), 28 * n) == 0);
        p = fields(src, n, (char*)b.data(), 8 * n);
        CHECK(hc.copy(p, true, nullptr) == hipSuccess && p.empty() && g_allocs == 1);
        for (size_t i = 0; i < src.size(); ++i) CHECK(b[i] == (double)src[i]);

        // pinned: FP32 is left to the plain copy, FP64 has to be widened
        char* pin = nullptr;
        CHECK(hipHostMalloc((void**)&pin, 56 * n, 0) == hipSuccess);
        const size_t copies = g_async, allocs = g_allocs;
        p = fields(src, n, pin, 4 * n);
        CHECK(hc.copy(p, false, nullptr) == hipSuccess && p.size() == 7);
        CHECK(g_async == copies && g_allocs == allocs);
        for (int f = 0; f < 7; ++f) CHECK(p[f].src == src.data() + f * n && p[f].dst == pin + 4 * f * n && p[f].n == n);
        p = fields(src, n, pin, 8 * n);
        CHECK(hc.copy(p, true, nullptr) == hipSuccess && p.empty());
        for (size_t i = 0; i < src.size(); ++i) CHECK(((double*)pin)[i] == (double)src[i]);

        // one pinned among pageable ones
        std::fill(a.begin(), a.end(), 0.f);
        p = fields(src, n, (char*)a.data(), 4 * n);
        p[2].dst = pin;
        CHECK(hc.copy(p, false, nullptr) == hipSuccess && p.size() == 1 && p[0].dst == pin);
        for (size_t i = 0; i < src.size(); ++i) CHECK(a[i] == (i / n == 2 ? 0.f : src[i]));

        // less than kMinBytes of pageable pieces: the plain copy
        p = fields(src, n, (char*)a.data(), 4 * n);
        for (int f = 0; f < 5; ++f) p[f].dst = pin + 4 * f * n;
        CHECK(hc.copy(p, false, nullptr) == hipSuccess && p.size() == 7);
        (void)hipHostFree(pin);

        // a small state: not even a look at where it goes
        const size_t looked = g_looked;
        p = fields(src, 1000, (char*)a.data(), 4000);
        CHECK(hc.copy(p, false, nullptr) == hipSuccess && p.size() == 7 && g_looked == looked);
    }
    CHECK(g_pinned_bytes == 0);  // given back with the last copier
    {
        // a large state takes a larger ring, which then serves small ones too
        HostCopier hc;
        const size_t m = 2500000;  // 70 MB
        std::vector<float> big(7 * m), out(7 * m);
        for (size_t i = 0; i < big.size(); ++i) big[i] = (float)(i % 99991);
        auto p = fields(src, n, (char*)a.data(), 4 * n);
        CHECK(hc.copy(p, false, nullptr) == hipSuccess && p.empty());
        const size_t small = g_pinned_bytes;
        p = fields(big, m, (char*)out.data(), 4 * m);
        CHECK(hc.copy(p, false, nullptr) == hipSuccess && p.empty() && big == out);
        CHECK(g_pinned_bytes > small);
        const size_t allocs = g_allocs;
        std::fill(a.begin(), a.end(), 0.f);
        p = fields(src, n, (char*)a.data(), 4 * n);
        CHECK(hc.copy(p, false, nullptr) == hipSuccess && p.empty() && a == src && g_allocs == allocs);
        // three at once; two rings stay, the larger ones
        HostCopier h3[3];
        std::vector<float> o3[3];
        std::vector<std::thread> th;
        for (int k = 0; k < 3; ++k)
            th.emplace_back([&, k] {
                o3[k].resize(7 * m);
                auto q = fields(big, m, (char*)o3[k].data(), 4 * m);
                if (h3[k].copy(q, false, nullptr) != hipSuccess || !q.empty()) o3[k].clear();
            });
        for (auto& t : th) t.join();
        for (auto& o : o3) CHECK(o == big);
        CHECK(g_pinned_bytes <= (size_t)64 << 20);
    }
    CHECK(g_pinned_bytes == 0);
    {
        HostCopier hc;
        g_no_memory = true;
        auto p = fields(src, n, (char*)a.data(), 4 * n);
        CHECK(hc.copy(p, false, nullptr) == hipSuccess && p.size() == 7);
    }
    std::printf("ok\n");
    return 0;
}
"""


@pytest.mark.parametrize("san", ["address,undefined", "thread"])
def test_pieces_and_values(tmp_path, san):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    (tmp_path / "driver.cpp").write_text(DRIVER)
    exe = tmp_path / "driver"
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-g", f"-fsanitize={san}", "-fno-sanitize-recover=all", "-I", str(tmp_path),
                        "-I", CSRC, str(tmp_path / "driver.cpp"), "-lpthread", "-o", str(exe)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
