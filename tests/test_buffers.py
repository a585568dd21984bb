"""Device buffers on the host side."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

FAILED_ALLOCATION = r"""
#include "nsdg_internal.hpp"
#include <cstdio>
int main()
{
    nsdg::DBuf<double> b;
    bool threw = false;
    try {
        b.alloc(size_t(1) << 56); // 2^59 bytes: refused on any machine, with or without a GPU
    } catch (const nsdg::Error&) {
        threw = true;
    }
    std::printf("%d %zu %d\n", threw, b.n, b.p != nullptr);
    return 0;
}
"""


def test_a_failed_allocation_leaves_the_buffer_empty(tmp_path):
    """Buffers kept between calls are allocated when their size is too small: a size left
    behind by a failed allocation would pass a null pointer to the next call's kernels."""
    src, exe = tmp_path / "alloc.cpp", tmp_path / "alloc"
    src.write_text(FAILED_ALLOCATION)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "nextsimdg_amd", "csrc"), str(src), "-L/opt/rocm/lib", "-lamdhip64",
                    "-Wl,-rpath,/opt/rocm/lib", "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.stdout.split() == ["1", "0", "0"], out.stdout + out.stderr
