"""DBuf (quantom_amd/csrc/device_buffer.h) when device memory runs out: the call that asked gets an error,
and the next one does not meet a size without memory behind it.  Compiled for the host with an
allocator of a fixed budget in HIP's place."""
import os
import shutil
import subprocess

import pytest

from tests.conftest import ROOT

HIP_INCLUDE = "/opt/rocm/include"

SRC = r"""
#include "device_buffer.h"
#include <cstdio>
#include <cstdlib>
#include <map>

static size_t budget = 1000;
static std::map<void*, size_t> held;
static hipError_t last = hipSuccess;
static size_t in_use() { size_t n = 0; for (auto& h : held) n += h.second; return n; }
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (in_use() + n > budget) { last = hipErrorOutOfMemory; return last; }
    *p = std::malloc(n);
    held[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p) { held.erase(p); std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
template <typename F> static bool fails(F&& f) {
    try { f(); } catch (const lima::LimaError& e) { return e.code == LIMA_E_HIP; }
    return false;
}
int main() {
    {
        lima::DBuf<float> b;
        CHECK(fails([&] { b.alloc(1000); }));                     // 4,000 bytes of 1,000
        CHECK(b.n == 0 && b.p == nullptr && last == hipSuccess);
        CHECK(fails([&] { b.alloc(1000); }) && b.n == 0);         // asked again, refused again
        b.alloc(100);
        CHECK(b.n == 100 && b.p);
        CHECK(fails([&] { b.grow(300); }));                       // as large as before
        CHECK(b.n == 100 && b.p && held[b.p] == 400 && last == hipSuccess);
        float* p = b.p;
        b.grow(50);
        CHECK(b.p == p && b.n == 100);
        b.grow(200);                                              // fits only once the former 400 are given back
        CHECK(b.n == 200 && held[b.p] == 800);
        p = b.p;
        b.upload(std::vector<float>(200));
        CHECK(b.p == p && b.n == 200);
        CHECK(fails([&] { b.upload(std::vector<float>(300)); }) && b.n == 0 && b.p == nullptr);
        b.alloc(0);
        CHECK(b.n == 0 && b.p == nullptr);
    }
    CHECK(held.empty());
    std::printf("ok\n");
    return 0;
}
"""


@pytest.mark.skipif(not os.path.isdir(os.path.join(HIP_INCLUDE, "hip")) or shutil.which("g++") is None, reason="HIP headers or g++ missing")
def test_a_failed_allocation_leaves_no_size(tmp_path):
    src = tmp_path / "buffer.cpp"
    src.write_text(SRC)
    exe = tmp_path / "buffer"
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", HIP_INCLUDE, "-I",
                    os.path.join(ROOT, "quantom_amd", "csrc"), str(src), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
