"""Device memory after a failed allocation (spice21_amd/csrc/devmem.h), on the CPU: the header compiled with g++ against
an allocator that fails on demand.  A request that failed leaves no memory, and the same request tries again."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "spice21_amd", "csrc")

PROGRAM = r"""
#include "devmem.h"
#include <cstdio>
#include <cstdlib>
static bool out_of_memory = false;
static int live = 0, calls = 0;
extern "C" hipError_t hipMalloc(void** p, size_t b) {
    calls++;
    *p = nullptr;
    if (out_of_memory) return hipErrorOutOfMemory;
    *p = std::malloc(b);
    live++;
    return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
    std::free(p);
    live--;
    return hipSuccess;
}
extern "C" const char* hipGetErrorString(hipError_t) { return "out of memory"; }
#define CHECK(x) \
    if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; }
int main() {
    {
        s21::DevMem m;
        m.keep(64);
        CHECK(m.p && m.bytes == 64 && calls == 1)
        void* const before = m.p;
        m.keep(64);
        CHECK(m.p == before && calls == 1)
        out_of_memory = true;
        for (int k = 0; k < 2; k++) {  // the second request for as much must not take the failed one's size for memory
            bool failed = false;
            try {
                m.keep(128);
            } catch (const s21::Error& e) {
                failed = e.code == S21_DEVICE;
            }
            CHECK(failed && !m.p && m.bytes == 0 && live == 0)
        }
        out_of_memory = false;
        m.keep(128);
        CHECK(m.p && m.bytes == 128 && live == 1)
        m.alloc(0);
        CHECK(!m.p && m.bytes == 0 && live == 0)
        m.alloc(8);
    }
    CHECK(live == 0)
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_a_failed_allocation_leaves_no_memory(tmp_path):
    src, exe = tmp_path / "devmem.cpp", tmp_path / "devmem"
    src.write_text(PROGRAM)
    b = subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC,
                        "-I" + os.path.join(CSRC, "..", "..", "include"),
                        str(src), "-o", str(exe)], capture_output=True, text=True, timeout=120)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
