"""HostPages (lh_hostcopy.h) on the host: contents stay as they are, and no
exception leaves it where memory or threads run out."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "luna.jl_amd", "csrc")
BODY = r"""
#include <hip/hip_runtime.h>
#include <new>
#include <stdio.h>
#include <stdlib.h>
static int left = -1;  // allocations until one fails
void* operator new(size_t n) {
    if (left >= 0 && left-- == 0) throw std::bad_alloc();
    return malloc(n);
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
#include "lh_hostcopy.h"
int main() {
    const size_t n = (size_t)40 << 20;
    unsigned char* p = (unsigned char*)aligned_alloc(4096, n);
    for (int k = -1; k < 24; k++) {
        for (size_t i = 0; i < n; i += 4096) p[i] = (unsigned char)(i >> 12);
        try {
            left = k;
            HostPages pages;
            pages.add(p + 100, n - 200);
            pages.start();
            pages.wait();
            left = -1;
        } catch (...) {
            left = -1;
            printf("an exception after %d allocations\n", k);
            return 1;
        }
        for (size_t i = 0; i < n; i += 4096)
            if (p[i] != (unsigned char)(i >> 12)) return 2;
    }
    return 0;
}
"""


def test_pages_survive_failures(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(BODY)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC, "-w", "-pthread",
                    str(src), "-o", str(exe), "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr[-300:])
