"""host_copy (csrc/host_copy.hpp) when threads cannot be had: the copy is whole and the process goes on. A small program
built here makes the k-th allocation after arming fail, for every k that the copy reaches, then none."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <new>
#include "host_copy.hpp"
static long armed = -1;
void *operator new(size_t n) {
    if (armed >= 0 && armed-- == 0) throw std::bad_alloc();
    if (void *p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
int main() {
    for (size_t bytes : {size_t(1000), size_t(4 << 20) + 3, size_t(23 << 20) + 77})
        for (long k = -1; k < 12; k++) {
            std::vector<uint8_t> a(bytes), b(bytes, 0);
            for (size_t i = 0; i < bytes; i++) a[i] = (uint8_t)(i * 2654435761u >> 13);
            armed = k;
            tah::host_copy(b.data(), a.data(), bytes);
            armed = -1;
            if (a != b) {
                std::printf("%zu bytes, allocation %ld: not whole\n", bytes, k);
                return 1;
            }
        }
    return 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="needs g++")
def test_allocations_that_fail(tmp_path):
    src, exe = tmp_path / "copy.cpp", tmp_path / "copy"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "tabicl-anywhere_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], timeout=60, capture_output=True, text=True)
    assert run.returncode == 0, run.stdout + run.stderr
