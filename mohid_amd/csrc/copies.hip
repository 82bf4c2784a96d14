// Copies between a caller's device arrays and a handle's own.
#include "mgpu_internal.h"

namespace {

// The arrays of a set, one grid row each, 16 bytes a load where both ends
// allow it, four loads in flight a lane.
template <typename T>
__device__ __forceinline__ void copy_units(const T *__restrict__ a, T *__restrict__ b, long n) {
    const long nt = (long)gridDim.x * blockDim.x;
    long q = blockIdx.x * (long)blockDim.x + threadIdx.x;
    for (; q + 3 * nt < n; q += 4 * nt) {
        const T v0 = a[q], v1 = a[q + nt], v2 = a[q + 2 * nt], v3 = a[q + 3 * nt];
        b[q] = v0;
        b[q + nt] = v1;
        b[q + 2 * nt] = v2;
        b[q + 3 * nt] = v3;
    }
    for (; q < n; q += nt) b[q] = a[q];
}

__global__ void __launch_bounds__(256) copy_set_kernel(CopySet c) {
    const int m = blockIdx.y;
    const char *a = static_cast<const char *>(c.src[m]);
    char *b = static_cast<char *>(c.dst[m]);
    const long n = c.bytes[m];
    if ((((uintptr_t)a | (uintptr_t)b) & 15) == 0) {
        copy_units(reinterpret_cast<const uint4 *>(a), reinterpret_cast<uint4 *>(b), n / 16);
        if (blockIdx.x == 0 && threadIdx.x < (n % 16) / 4) {
            const long q = n / 16 * 4 + threadIdx.x;
            reinterpret_cast<uint32_t *>(b)[q] = reinterpret_cast<const uint32_t *>(a)[q];
        }
    } else {
        copy_units(reinterpret_cast<const uint32_t *>(a), reinterpret_cast<uint32_t *>(b), n / 4);
    }
}

}  // namespace

bool on_device(const void *p, hipStream_t s) {
    // a process that sees one device needs no look-up (0.4 us each, 22 arrays in a
    // set_geometry and a set_hydro: 12 of 433 us of a small coupled step)
    static const bool only = [] {
        int n = 0;
        return hipGetDeviceCount(&n) == hipSuccess && n == 1;
    }();
    if (only) return true;
    int dev = 0;
    hipPointerAttribute_t a;
    if (hipStreamGetDevice(s, &dev) == hipSuccess && hipPointerGetAttributes(&a, p) == hipSuccess)
        return a.type == hipMemoryTypeDevice && a.device == dev;
    (void)hipGetLastError();   // memory the runtime does not know: not an error here
    return false;
}

int launch_copy_set(const CopySet &all, hipStream_t s) {
    // arrays of another device (or of the host) go through the runtime's copy,
    // which needs no peer access
    CopySet c;
    for (int m = 0; m < all.n; ++m) {
        if (!all.caller[m] || on_device(all.caller[m], s))
            c.add(all.src[m], all.dst[m], (size_t)all.bytes[m], all.caller[m]);
        else
            HIPCHK(hipMemcpyAsync(all.dst[m], all.src[m], (size_t)all.bytes[m],
                                  hipMemcpyDeviceToDevice, s));
    }
    if (c.n <= 0) return MGPU_SUCCESS;
    long most = 0;
    for (int m = 0; m < c.n; ++m) most = c.bytes[m] > most ? c.bytes[m] : most;
    long blocks = (most / 64 + 255) / 256 + 1;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(copy_set_kernel, dim3((unsigned)blocks, c.n), dim3(256), 0, s, c);
    HIPCHK(hipGetLastError());
    return MGPU_SUCCESS;
}
