// Compares the kernel weight's root (pm_sqrt_w) with sqrtf over every float from
// 2^-96 to 2^64, and its weight with sigma over every smaller one (0 and the
// subnormal ones too).  Prints the number of differences of both.
#include <hip/hip_runtime.h>
#include <stdio.h>

#include "pm_device.h"

__global__ __launch_bounds__(256) void k_root(uint32_t first, uint32_t n, unsigned long long *bad)
{
    unsigned long long d = 0;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
        const float x = __uint_as_float(first + i);
        d += __float_as_uint(pm_sqrt_w(x)) != __float_as_uint(sqrtf(x)) ? 1ull : 0ull;
    }
    if (d) atomicAdd(bad, d);
}

__global__ __launch_bounds__(256) void k_weight(uint32_t n, float inv_h, float sig, unsigned long long *bad)
{
    unsigned long long d = 0;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
        const float x = __uint_as_float(i);
        d += pm_W_in(x, inv_h, sig) != sig || pm_W_sel(x, inv_h, sig) != sig ? 1ull : 0ull;
    }
    if (d) atomicAdd(bad, d);
}

static uint32_t bits(float f) { union { float f; uint32_t u; } v = { f }; return v.u; }

int main()
{
    unsigned long long *bad = nullptr, host[2] = { 1, 1 };
    if (hipMalloc((void **)&bad, sizeof(host)) != hipSuccess) return 2;
    if (hipMemset(bad, 0, sizeof(host)) != hipSuccess) return 2;
    const uint32_t lo = bits(0x1p-96f), hi = bits(0x1p64f);
    hipLaunchKernelGGL(k_root, dim3(8192), dim3(256), 0, 0, lo, hi - lo + 1, bad);
    const float inv_h[] = { 1.0e-3f, 10.0f, 1.0e5f, 0x1.fp33f };
    for (float f : inv_h) hipLaunchKernelGGL(k_weight, dim3(8192), dim3(256), 0, 0, lo, f, 1.7f, bad + 1);
    if (hipGetLastError() != hipSuccess || hipMemcpy(host, bad, sizeof(host), hipMemcpyDeviceToHost) != hipSuccess) return 2;
    printf("%llu %llu\n", host[0], host[1]);
    return hipFree(bad) == hipSuccess ? 0 : 2;
}
