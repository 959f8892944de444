// pm_gauss.hip -- screen-space depth smoothing: GaussRenderPass
// (GaussRenderPass.cpp:8-48 kernel table, 347-358 uniforms; gauss.frag).
//
// out(x, y) = sum_{i=-N..N} sum_{j=-N..N} K(|i|, |j|) depth(x + i, y + j),
// i (the horizontal offset) outer, j inner, as gauss.frag loops, each term
// accumulated with one fused multiply-add (gauss.frag's `sum += k * t` carries
// no `precise`, so the shader compiler may fuse it; fused here and in the
// oracle, so both round the same way); the depth texture is addressed
// clamp-to-edge (BilateralBuffer.cpp:246-248) at texel centres (Spread = 1,
// GaussRenderPass.h:66), so every tap is a texel value.
//
// A 256-thread workgroup takes a 32x32 output tile (contiguous runs of tiles per
// XCD) and stages the edge-clamped window in LDS; each thread computes 4
// vertically adjacent outputs, so a column's 4 + 2N values are read from LDS
// once per horizontal offset and used by all 4; the weights are uniform and come
// through scalar loads.  N is a template argument for every window the entry
// points take (0..31).  HBM traffic is one read of the image (plus the halo) and
// one write; the FMAs bound it from N = 8 up: (2N + 1)^2 per pixel in the fixed
// order of the sum, at 78.6 TFLOP/s without packed math (15.2 us at N = 8 and
// 1920x1080; 24.2 measured: all 2,040 workgroups are resident at once, eight to a
// CU, so they stage their windows together before the first FMA and no other's
// arithmetic covers that; VALU busy 59 % of the launch).  1920x1080 with one output per thread and the
// weights in LDS (two LDS reads per FMA), and now: N = 3 30.1 and 8.7 us, N = 12
// 240 and 46.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

#include "pmarch.h"

namespace pm {

static constexpr int kTW = 32, kR = 4, kTH = 8 * kR;

// The horizontal offsets are a loop, not unrolled: unrolled, the compiler
// hoists every column's LDS reads ahead of the arithmetic (~350 VGPRs at N = 8,
// one wave per SIMD).  A wave stages whole rows of the window: the clamped row
// is a scalar and the clamped column is found once, so a value costs a load and
// a store (with a division and two clamps per value N = 8 took 25.5 us, now 24.2).
template <int N>
__global__ __launch_bounds__(256) void k_depth_smooth(const float *__restrict__ in, float *__restrict__ out, uint32_t W,
                                                      uint32_t H, const float *__restrict__ K)
{
    constexpr int tw = kTW + 2 * N, th = kTH + 2 * N;
    __shared__ float tile[tw * th];
    // Workgroups are dispatched to the 8 XCDs round-robin (blockIdx % 8 names
    // the XCD): each XCD takes a contiguous run of row-major tiles, so the
    // halos that neighbouring tiles share are read once into that XCD's L2.
    const uint32_t tiles_x = (W + kTW - 1) / kTW, T = tiles_x * ((H + kTH - 1) / kTH), per = (T + 7) / 8;
    const uint32_t t = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (t >= T) return;                            // whole workgroup, before the barrier
    const int x0 = (int)(t % tiles_x) * kTW, y0 = (int)(t / tiles_x) * kTH;
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
#pragma unroll
    for (int c = 0; c < tw; c += 64) {
        const int tx = c + lane, gx = min(max(x0 + tx - N, 0), (int)W - 1);
        if (tx < tw) {
#pragma unroll 4
            for (int ty = wave; ty < th; ty += 4) {
                const int gy = min(max(y0 + ty - N, 0), (int)H - 1);
                tile[ty * tw + tx] = in[(size_t)gy * W + (size_t)gx];
            }
        }
    }
    __syncthreads();
    const int lx = (int)threadIdx.x % kTW, ly = (int)threadIdx.x / kTW;
    float s[kR];
#pragma unroll
    for (int m = 0; m < kR; m++) s[m] = 0.0f;
#pragma unroll 1
    for (int i = -N; i <= N; i++) {
        // rows ly kR .. ly kR + kR - 1 + 2N of window column lx + N + i
        float v[kR + 2 * N];
        const float *col = tile + (ly * kR) * tw + (lx + N + i);
#pragma unroll
        for (int k = 0; k < kR + 2 * N; k++) v[k] = col[k * tw];
        const float *kr = K + (i < 0 ? -i : i) * (N + 1);     // uniform: scalar loads
        float kw[N + 1];
#pragma unroll
        for (int q = 0; q <= N; q++) kw[q] = kr[q];
#pragma unroll
        for (int m = 0; m < kR; m++)
#pragma unroll
            for (int j = -N; j <= N; j++) s[m] = __builtin_fmaf(kw[j < 0 ? -j : j], v[m + j + N], s[m]);
    }
    const int x = x0 + lx;
    if (x >= (int)W) return;
#pragma unroll
    for (int m = 0; m < kR; m++) {
        const int y = y0 + ly * kR + m;
        if (y < (int)H) out[(size_t)y * W + (size_t)x] = s[m];
    }
}

using SmoothKernel = void (*)(const float *, float *, uint32_t, uint32_t, const float *);

template <int... N> static SmoothKernel smooth_kernel(int n, std::integer_sequence<int, N...>)
{
    static constexpr SmoothKernel table[] = { k_depth_smooth<N>... };
    return table[n];
}

hipError_t launch_depth_smooth(const float *in, float *out, uint32_t W, uint32_t H, int N, const float *K,
                               hipStream_t st)
{
    if (N < 0 || N > 31) return hipErrorInvalidValue;
    const uint32_t T = ((W + kTW - 1) / kTW) * ((H + kTH - 1) / kTH);
    hipLaunchKernelGGL(smooth_kernel(N, std::make_integer_sequence<int, 32>{}), dim3(8 * ((T + 7) / 8)), dim3(256), 0, st,
                       in, out, W, H, K);
    return hipGetLastError();
}

}  // namespace pm
