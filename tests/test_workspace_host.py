"""The split-K workspace where its growth fails: csrc/workspace.cpp compiled for the host against a HIP
runtime of its own here, whose allocations fail on request."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ming-tts_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "mt_internal.hpp"
static bool fail_malloc, fail_memset;
static hipError_t last = hipSuccess;
static int frees;
extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) {
    if (fail_malloc) return last = hipErrorOutOfMemory;
    *p = malloc(n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return fail_memset ? last = hipErrorUnknown : hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipFree(void *p) { frees++; free(p); return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "refused"; }
}
namespace mt {
int set_error(int code, const char *, ...) { return code; }
}
#define CHECK(c) do { if (!(c)) { printf("%s\n", #c); return 1; } } while (0)
int main() {
    void *a, *b;
    uint32_t *ca, *cb;
    CHECK(mt::stream_workspace(nullptr, 1000, 4, &a, &ca) == 0);
    for (int memset_too = 0; memset_too < 2; memset_too++) {
        (memset_too ? fail_memset : fail_malloc) = true;
        CHECK(mt::stream_workspace(nullptr, 1 << 20, 4, &b, &cb) != 0);
        CHECK(hipGetLastError() == hipSuccess);  // the next launch's check finds nothing
        CHECK(mt::stream_workspace(nullptr, 1000, 4, &b, &cb) == 0);  // the stream keeps what it had
        CHECK(b == a && cb == ca);
        fail_malloc = fail_memset = false;
    }
    CHECK(frees == 1);
    CHECK(mt::stream_workspace(nullptr, 1 << 20, 4, &b, &cb) == 0 && b != a);
    CHECK(frees == 1);  // the old one is kept: graphs may hold its address
    printf("ok\n");
    return 0;
}
"""


def test_a_failed_growth_leaves_the_stream_as_it_was(tmp_path):
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "workspace_host"
    subprocess.run([f"{ROCM}/bin/hipcc", "--offload-host-only", "-no-hip-rt", "-std=c++17", "-O1", f"-I{CSRC}",
                    f"-I{os.path.join(CSRC, '..', '..', 'include')}", "-x", "hip", str(tmp_path / "main.cpp"),
                    "-x", "hip", os.path.join(CSRC, "workspace.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
