"""The staged read-back (openems_amd/csrc/oe_copy.hip) on the CPU: the file is
built with the host compiler against a runtime whose transfers are memcpy and
whose calls can be made to fail.  Without memory, events or threads for the
ring the runtime's own copy runs; a transfer that fails is an error; nothing
that was made is left behind."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#include "oe_internal.h"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <string>
#include <vector>
static std::string mode;
static long events, pins, copies, direct, fail_at = -1, last_error;
static const char *dst0, *dst1;
static char done;
extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (mode == "no_ring") return last_error = 1, hipErrorOutOfMemory;
    ++pins;
    *p = malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { return free(p), --pins, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (mode == "no_event" && events == 3) return last_error = 1, hipErrorOutOfMemory;
    ++events;
    *e = (hipEvent_t)&done;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return --events, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return rand() % 3 ? hipErrorNotReady : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return last_error = 0, hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (++copies == fail_at) return hipErrorUnknown;
    if ((char*)d >= dst0 && (char*)d < dst1) ++direct;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    if (mode == "no_attributes") return last_error = 1, hipErrorInvalidValue;
    a->type = mode == "pinned" && p == dst0 ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipMalloc(void**, size_t) { abort(); }
hipError_t hipFree(void*) { abort(); }
}
int main(int argc, char** argv) {
    mode = argv[1];
    fail_at = atol(argv[2]);
    std::vector<char> src, dst;
    std::vector<oe::HostCopy> c;
    size_t total = 0;
    for (int q = 3; q < argc; ++q) total += atol(argv[q]);
    src.resize(total);
    dst.resize(total);
    for (size_t q = 0; q < total; ++q) src[q] = (char)(q * 2654435761u >> 24);
    dst0 = dst.data();
    dst1 = dst0 + total;
    for (size_t q = 3, o = 0; q < (size_t)argc; o += atol(argv[q++])) c.push_back({dst.data() + o, src.data() + o, (size_t)atol(argv[q])});
    const hipError_t e = oe::copy_to_host(c.data(), (int)c.size(), nullptr);
    printf("%d %d %ld %ld %ld %ld\n", e == hipSuccess, src == dst, direct, events, pins, last_error);
}
"""


@pytest.fixture(scope="module")
def copy(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("needs g++ and the HIP headers")
    d = tmp_path_factory.mktemp("copy")
    (d / "run.cpp").write_text(RUNTIME)
    src = os.path.join(ROOT, "openems_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-w", "-I", src, "-I", "/opt/rocm/include", "-I",
                    os.path.join(ROOT, "include"), "-x", "c++", str(d / "run.cpp"), "-x", "c++", os.path.join(src, "oe_copy.hip"),
                    "-o", str(d / "run"), "-pthread"], check=True)

    def run(mode, *sizes, fail_at=-1):
        r = subprocess.run([str(d / "run"), mode, str(fail_at), *map(str, sizes)], capture_output=True, text=True, check=True,
                           timeout=60)
        ok, same, direct, events, pins, err = map(int, r.stdout.split())
        assert events == 0 and pins == 0 and err == 0, "left behind"
        return bool(ok), bool(same), direct

    return run


MB = 1 << 20
SIZES = [(12 * MB,), (5 * MB, 7 * MB + 4, 1), (2 * MB,) * 6, (40 * MB + 12, 3), (17 * MB, 17 * MB)]


@pytest.mark.parametrize("sizes", SIZES)
def test_ring_carries_all(copy, sizes):
    assert copy("ok", *sizes) == (True, True, 0)


@pytest.mark.parametrize("mode", ["no_ring", "no_event"])
@pytest.mark.parametrize("sizes", SIZES)
def test_without_a_ring_the_runtime_copies(copy, mode, sizes):
    assert copy(mode, *sizes) == (True, True, len(sizes))


@pytest.mark.parametrize("sizes", SIZES)
def test_a_pinned_destination_takes_the_transfers(copy, sizes):
    assert copy("pinned", *sizes) == (True, True, len(sizes))
    assert copy("no_attributes", *sizes) == (True, True, 0)


@pytest.mark.parametrize("sizes", [(12 * MB - 4,), (1,), (5 * MB, 6 * MB)])
def test_small_copies_are_the_runtimes(copy, sizes):
    assert copy("ok", *sizes) == (True, True, len(sizes))


@pytest.mark.parametrize("at", [1, 5, 9, 20])
def test_a_failed_transfer_is_an_error(copy, at):
    assert copy("ok", 40 * MB, fail_at=at)[0] is False
