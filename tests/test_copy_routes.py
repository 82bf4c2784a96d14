"""Which arrays the library's kernels copy or read in place, and which go through
the runtime's copy, on the CPU: csrc/copies.hip's host code against a stand-in
for the HIP runtime that knows memory of two devices and of the host.  A kernel
must be given no pointer but the stream's own device's: without peer access it
could not read another's."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mohid_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

DRIVER = r"""
#include <stdio.h>
#include <string.h>
#include "mgpu_internal.h"

static char own[2][256], peer[2][256], host[2][256];     // device 0, device 1, not known
static int launches = 0, copied = 0, last = 0;
static CopySet got;
static dim3 grid, block;                               // of the launch under way

extern "C" {
hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *dev) { *dev = 0; return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    const char *c = (const char *)p;
    memset(a, 0, sizeof(*a));
    a->type = hipMemoryTypeDevice;
    if (c >= own[0] && c < own[0] + sizeof(own)) return hipSuccess;
    a->device = 1;
    if (c >= peer[0] && c < peer[0] + sizeof(peer)) return hipSuccess;
    last = 1;
    return hipErrorInvalidValue;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    memcpy(d, s, n);
    ++copied;
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const int e = last;
    last = 0;
    return e ? hipErrorInvalidValue : hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3 g, dim3, void **args, size_t, hipStream_t) {
    memcpy(&got, args[0], sizeof(got));
    ++launches;
    return g.y == (unsigned)got.n ? hipSuccess : hipErrorInvalidValue;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
    grid = g;
    block = b;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s) {
    *g = grid;
    *b = block;
    *n = 0;
    *s = nullptr;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *,
                           void *, void *, int *) {}
void __hipUnregisterFatBinary(void **) {}
}
void mgpu_set_error(const char *what, hipError_t) { printf("error %s\n", what); }

int main() {
    if (!on_device(own[1] + 8, nullptr) || on_device(peer[0], nullptr) ||
        on_device(host[0], nullptr) || last)
        return 1;
    CopySet c;
    c.add(own[0], own[1], 64, own[0]);
    c.add(peer[0], own[1] + 64, 64, peer[0]);       // a field on another device
    c.add(host[0], own[1] + 128, 64, host[0]);      // memory the runtime does not describe
    c.add(own[0] + 64, peer[1], 64, peer[1]);       // fluxes asked for on another device
    c.add(own[0] + 128, own[1] + 192, 64, nullptr);
    if (launch_copy_set(c, nullptr)) return 2;
    if (launches != 1 || copied != 3 || got.n != 2 || last) return 3;
    if (got.src[0] != own[0] || got.dst[0] != own[1] || got.src[1] != own[0] + 128 ||
        got.dst[1] != own[1] + 192 || got.bytes[1] != 64)
        return 4;
    CopySet e;
    e.add(peer[0], own[1], 64, peer[0]);
    if (launch_copy_set(e, nullptr) || launches != 1 || copied != 4) return 5;
    return 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc missing")
def test_kernels_get_only_the_streams_own_memory(tmp_path):
    (tmp_path / "driver.hip").write_text(DRIVER)
    flags = [HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "--offload-host-only", "-fPIC",
             "-I" + CSRC, "-I" + os.path.join(ROOT, "include")]
    objs = []
    for f in (os.path.join(CSRC, "copies.hip"), str(tmp_path / "driver.hip")):
        objs.append(str(tmp_path / (os.path.basename(f)[:-4] + ".o")))
        subprocess.run([*flags, "-c", f, "-o", objs[-1]], check=True, timeout=300)
    exe = str(tmp_path / "driver")
    # the device code is not there: nothing refers to it in the stand-in runtime
    subprocess.run(["g++", *objs, "-o", exe, "-Wl,--unresolved-symbols=ignore-all"], check=True,
                   timeout=120)
    assert subprocess.run([exe], timeout=60).returncode == 0
