"""A device buffer whose allocation failed holds nothing (openems_amd/csrc/
oe_internal.h: DevBuf), so that the next call asks again instead of handing a
null pointer to a kernel.  Built with the host compiler; the allocator fails on
request."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "oe_internal.h"
#include <cstdio>
#include <cstdlib>
static size_t most = 1000;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
    if (n > most) return *p = (void*)8, hipErrorOutOfMemory;
    return *p = malloc(n), hipSuccess;
}
extern "C" hipError_t hipFree(void* p) { return free(p), hipSuccess; }
int main() {
    oe::DevBuf b;
    const bool first = b.alloc(500) == hipSuccess && b.p && b.bytes == 500;
    const bool failed = b.alloc(2000) != hipSuccess && !b.p && b.bytes == 0;
    most = 4000;
    const bool again = b.alloc(2000) == hipSuccess && b.p && b.bytes == 2000;
    const bool none = b.alloc(0) == hipSuccess && !b.p && b.bytes == 0;
    printf("%d%d%d%d\n", first, failed, again, none);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"),
                    reason="needs g++ and the HIP headers")
def test_a_failed_allocation_leaves_no_size(tmp_path):
    (tmp_path / "buf.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-w", "-I", os.path.join(ROOT, "openems_amd", "csrc"), "-I",
                    "/opt/rocm/include", "-I", os.path.join(ROOT, "include"), str(tmp_path / "buf.cpp"), "-o",
                    str(tmp_path / "buf")], check=True)
    assert subprocess.run([str(tmp_path / "buf")], capture_output=True, text=True).stdout == "1111\n"
