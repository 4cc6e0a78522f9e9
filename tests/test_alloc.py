"""An allocation that finds no memory is tried once more after what can be
released is released (csrc/grmp_alloc.h, compiled here by itself)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gradientrobustmultiphysics.jl_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "grmp_alloc.h"
// results of the attempts in order, releases made, and what the call returned
static void run(std::initializer_list<hipError_t> results)
{
    const hipError_t *next = results.begin();
    int released = 0;
    const hipError_t e = alloc_or_release([&] { return *next++; }, [&] { ++released; });
    std::printf("%d %d %d\n", (int)e, (int)(next - results.begin()), released);
}
int main()
{
    run({hipSuccess});
    run({hipErrorOutOfMemory, hipSuccess});
    run({hipErrorOutOfMemory, hipErrorOutOfMemory});
    run({hipErrorInvalidValue});
    return 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++") or not os.path.isdir("/opt/rocm/include/hip"), reason="needs g++ and HIP headers")
def test_out_of_memory_releases_and_retries(tmp_path):
    src, exe = tmp_path / "alloc.cpp", tmp_path / "alloc"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", CSRC, str(src), "-o",
                    str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    got = [tuple(map(int, line.split())) for line in out.splitlines()]
    oom, bad = 2, 1  # hipErrorOutOfMemory, hipErrorInvalidValue
    assert got == [(0, 1, 0), (0, 2, 1), (oom, 2, 1), (bad, 1, 0)]
