// pm_mlp.hip -- training and batch inference of the step-proposal MLP, the
// coarse occupancy grid its features read, and the trace logger that turns
// plain-march results into (features, distance-to-crossing) pairs.
//
// Training step for a batch of B samples (B a multiple of 64):
//   k_mlp_train : four waves per 64 samples -- forward, loss, backward with BF16
//                 MFMA GEMMs (FP32 accumulate) -> per-workgroup partial gradients
//   k_mlp_adam  : sums the partials in a fixed order (deterministic) and applies
//                 Adam to the FP32 master weights, then refreshes the BF16 copies
#include "pm_features.h"
#include "pm_internal.h"
#include "pm_mlp.h"

namespace pm {

// ------------------------------------------------------------ coarse grid --

__global__ __launch_bounds__(256) void k_coarse_counts(GridDev g, CoarseDev cg, uint32_t *__restrict__ out)
{
    uint32_t c = blockIdx.x * 256 + threadIdx.x;
    if (c >= (uint32_t)cg.nx * cg.ny * cg.nz) return;
    int32_t X = c % cg.nx, Y = (c / cg.nx) % cg.ny, Z = c / (cg.nx * cg.ny);
    uint32_t sum = 0;
    for (int z = 4 * Z; z < 4 * Z + 4 && z < g.nz; z++)
        for (int y = 4 * Y; y < 4 * Y + 4 && y < g.ny; y++) {
            int x0 = 4 * X, x1 = min(4 * X + 4, g.nx);
            uint32_t row = (uint32_t)g.nx * ((uint32_t)y + (uint32_t)g.ny * (uint32_t)z);
            sum += g.cell_start[row + x1] - g.cell_start[row + x0];
        }
    out[c] = sum;
}

hipError_t launch_coarse_counts(const GridDev &g, const CoarseDev &cg, uint32_t *out, hipStream_t st)
{
    uint32_t n = (uint32_t)cg.nx * cg.ny * cg.nz;
    hipLaunchKernelGGL(k_coarse_counts, dim3((n + 255) / 256), dim3(256), 0, st, g, cg, out);
    return hipGetLastError();
}

// ------------------------------------------------------------ trace logger --

__device__ __forceinline__ uint32_t hash32(uint32_t x)
{
    x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16;
    return x;
}

// One thread per selected ray.  Rays are selected by hash(pixel ^ seed) % ray_stride == 0;
// samples k = k0, k0 + k_stride, ... (k0 = hash % k_stride) before the crossing.
__global__ __launch_bounds__(256) void k_trace(TraceArgs a)
{
    uint32_t idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= a.W * a.H) return;
    uint32_t hsh = hash32(idx ^ a.seed);
    if (hsh % a.ray_stride != 0) return;
    const GridDev &g = a.g;
    uint32_t px = idx % a.W, py = idx / a.W;
    float cx = (float)px * (2.0f / (float)a.W) - 1.0f, cy = (float)py * (2.0f / (float)a.H) - 1.0f;
    float w[4];
    for (int r = 0; r < 4; r++) w[r] = (a.M[r] * cx + a.M[4 + r] * cy) + (a.M[8 + r] * 1.0f + a.M[12 + r] * 1.0f);
    float dun[3] = { w[0] / w[3] - a.cam[0], w[1] / w[3] - a.cam[1], w[2] / w[3] - a.cam[2] };
    float inv = 1.0f / sqrtf((dun[0] * dun[0] + dun[1] * dun[1]) + dun[2] * dun[2]);
    float d[3] = { dun[0] * inv, dun[1] * inv, dun[2] * inv };
    float tn = 0.0f, tf = INFINITY;
    for (int ax = 0; ax < 3; ax++) {
        if (d[ax] != 0.0f) {
            float iv = 1.0f / d[ax];
            float t0 = (g.bmin[ax] - a.cam[ax]) * iv, t1 = (g.bmax[ax] - a.cam[ax]) * iv;
            tn = fmaxf(tn, fminf(t0, t1));
            tf = fminf(tf, fmaxf(t0, t1));
        } else if (a.cam[ax] < g.bmin[ax] || a.cam[ax] > g.bmax[ax]) {
            return;
        }
    }
    if (tn > tf) return;
    float thit = a.t_hit[idx];
    float tend = thit >= 0.0f ? thit : tf;
    uint32_t k = (hsh >> 8) % a.k_stride;
    for (;; k += a.k_stride) {
        float t = tn + (float)k * a.step;
        if (t >= tend) break;
        float q[3] = { a.cam[0] + t * d[0], a.cam[1] + t * d[1], a.cam[2] + t * d[2] };
        // the features the learned march computes at a sample below iso: its
        // (compensated) density, grad rho over the fine stencil, the 27-cell count
        uint32_t cand = 0;
        const float rho = pm_density32(g, q[0], q[1], q[2], true, cand);
        if (rho >= a.iso) break;                 // at or past the crossing
        uint32_t row = atomicAdd(a.count, 1u);
        if (row >= a.cap) break;
        float gx, gy, gz;
        grad_feat(g, q[0], q[1], q[2], gx, gy, gz, cand);
        float f[PM_MLP_IN];
        float gmag = sqrtf((gx * gx + gy * gy) + gz * gz);
        mlp_features(g, a.cg, a.cam, d, t, tn, tf, rho, gmag, (float)pm_cand27(g, q[0], q[1], q[2]), a.iso, f);
        for (int j = 0; j < PM_MLP_IN; j++) a.feat[(uint64_t)row * PM_MLP_IN + j] = f[j];
        float dist = (tend - t) * g.inv_h;
        a.label[row] = log2f(1.0f + fminf(dist, 255.0f));
        a.is_hit[row] = thit >= 0.0f ? 1 : 0;
        a.meta[2 * (uint64_t)row] = idx;
        a.meta[2 * (uint64_t)row + 1] = k;
    }
}

hipError_t launch_trace(const TraceArgs &a, hipStream_t st)
{
    uint32_t n = a.W * a.H;
    hipLaunchKernelGGL(k_trace, dim3((n + 255) / 256), dim3(256), 0, st, a);
    return hipGetLastError();
}

// --------------------------------------------------------------- training --

// LDS row strides in bf16: 16-byte rows that start in different banks (at the
// plain 32 and 64 every row starts in the same one).
static constexpr int kXS = PM_MLP_K1 + 8, kHS = PM_MLP_H + 8;

struct TrainLds {
    uint16_t X[64 * kXS];
    uint16_t XT[PM_MLP_K1 * kHS];
    uint16_t H1[64 * kHS], H1T[64 * kHS];
    uint16_t G2[64 * kHS], G2T[64 * kHS];
    uint16_t G1T[64 * kHS];
    float Y[4][64], DY[64];
};

// Four bf16 of one unit's consecutive samples, as one 8-byte store.
__device__ __forceinline__ void store_bf16x4(uint16_t *p, const uint16_t *v)
{
    *(uint2 *)p = make_uint2((uint32_t)v[0] | ((uint32_t)v[1] << 16), (uint32_t)v[2] | ((uint32_t)v[3] << 16));
}

// acc[m] += A[16 m .. 16 m + 15][.] B^T for one 16-row tile of B held in
// registers (32 KT values of K); A in LDS, row stride lda.
template <int MT, int KT>
__device__ __forceinline__ void train_gemm(const uint16_t *A, int lda, const pm_bf16x8 (&b)[KT], pm_f32x4 (&acc)[MT])
{
    const int l = threadIdx.x & 63, row = l & 15, kb = l >> 4;
#pragma unroll
    for (int kk = 0; kk < KT; kk++)
#pragma unroll
        for (int m = 0; m < MT; m++)
            acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_bf16x8(A + (16 * m + row) * lda + 32 * kk + 8 * kb),
                                                             b[kk], acc[m], 0, 0, 0);
}

// Four waves per 64 samples; wave w takes units 16 w .. 16 w + 15 of every
// layer, all 64 samples.  One wave's chain of loads, MFMAs, activations and LDS
// round trips bounds a small batch, so it is cut in four, the weights are
// loaded before the inputs, and the samples' rows come in 16-byte loads.  At
// most kTrainBlocks workgroups: beyond 64 kTrainBlocks samples a workgroup
// takes several groups of 64 and keeps its sums in registers, which bounds the
// partial gradients written here and read by k_mlp_adam (25 KB a workgroup).
// 4,096 rows: 21.6 us with one wave per 64 samples, 10.8 now; 65,536 rows: 52.9
// and 28.8.
__global__ __launch_bounds__(256) void k_mlp_train(TrainArgs a)
{
    __shared__ TrainLds S;
    const int l = threadIdx.x & 63, col = l & 15, kb = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), u = 16 * w + col;
    const MlpDev &net = a.net;
    float *part = a.partial + (uint64_t)blockIdx.x * (PM_MLP_NPARAM + 1);

    // this wave's weights: rows u of W1, W2 and W2^T
    pm_bf16x8 bw1[1], bw2[2], bw2t[2];
    bw1[0] = load_bf16x8(net.W1 + u * PM_MLP_K1 + 8 * kb);
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
        bw2[kk] = load_bf16x8(net.W2 + u * PM_MLP_H + 32 * kk + 8 * kb);
        bw2t[kk] = load_bf16x8(net.W2T + u * PM_MLP_H + 32 * kk + 8 * kb);
    }
    const float b1 = net.p[PM_MLP_OFF_B1 + u], b2 = net.p[PM_MLP_OFF_B2 + u], w3 = net.p[PM_MLP_OFF_W3 + u],
                b3 = net.p[PM_MLP_OFF_B3];

    const pm_f32x4 zero = { 0.f, 0.f, 0.f, 0.f };
    pm_f32x4 gW2[4] = { zero, zero, zero, zero }, gW1[2] = { zero, zero };
    float gw3 = 0.f, gb2 = 0.f, gb1 = 0.f, gb3 = 0.f, loss = 0.f;

    for (uint32_t grp = blockIdx.x; grp < a.ngroups; grp += gridDim.x) {
        // inputs: four threads per sample, eight of the 32 columns each
        {
            const int s = (int)threadIdx.x >> 2, q = (int)threadIdx.x & 3;
            const uint32_t sample = a.idx ? a.idx[grp * 64 + s] : grp * 64 + s;
            float f[8] = { 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f };
            if (q < 3) {
                const float4 *src = (const float4 *)(a.feat + (uint64_t)sample * PM_MLP_IN) + 2 * q;
                const float4 v0 = src[0], v1 = src[1];
                f[0] = v0.x; f[1] = v0.y; f[2] = v0.z; f[3] = v0.w;
                f[4] = v1.x; f[5] = v1.y; f[6] = v1.z; f[7] = v1.w;
            }
            uint16_t h[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                h[j] = f2bf(f[j]);
                S.XT[(8 * q + j) * kHS + s] = h[j];
            }
            store_bf16x4(&S.X[s * kXS + 8 * q], h);
            store_bf16x4(&S.X[s * kXS + 8 * q + 4], h + 4);
        }
        const uint32_t mine = a.idx ? a.idx[grp * 64 + l] : grp * 64 + l;
        const float t = a.label[mine];
        __syncthreads();

        // layer 1
        pm_f32x4 z1[4] = { zero, zero, zero, zero };
        train_gemm<4, 1>(S.X, kXS, bw1, z1);
#pragma unroll
        for (int mi = 0; mi < 4; mi++) {
            uint16_t hb[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                z1[mi][r] += b1;
                hb[r] = f2bf(mlp_act(z1[mi][r]));
                S.H1[(16 * mi + 4 * kb + r) * kHS + u] = hb[r];
            }
            store_bf16x4(&S.H1T[u * kHS + 16 * mi + 4 * kb], hb);
        }
        __syncthreads();

        // layer 2 and output: this wave's 16 units of every sample's sum
        pm_f32x4 z2[4] = { zero, zero, zero, zero };
        train_gemm<4, 2>(S.H1, kHS, bw2, z2);
        float a2[4][4];
#pragma unroll
        for (int mi = 0; mi < 4; mi++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                z2[mi][r] += b2;
                a2[mi][r] = mlp_act(z2[mi][r]);
                float v = w3 * a2[mi][r];
                v += __shfl_xor(v, 1, 64);
                v += __shfl_xor(v, 2, 64);
                v += __shfl_xor(v, 4, 64);
                v += __shfl_xor(v, 8, 64);
                if (col == 0) S.Y[w][16 * mi + 4 * kb + r] = v;
            }
        __syncthreads();

        // loss: wt * (y - t)^2, wt = w_over when the prediction is too long
        // (every wave for sample l; wave 0 keeps it)
        const float y = ((S.Y[0][l] + S.Y[1][l]) + (S.Y[2][l] + S.Y[3][l])) + b3;
        const float diff = y - t, wt = diff > 0.0f ? a.w_over : 1.0f;
        const float dy = 2.0f * wt * diff * a.inv_batch;
        loss += wt * diff * diff * a.inv_batch;
        gb3 += dy;
        if (w == 0) S.DY[l] = dy;
        __syncthreads();

        // output layer and layer-2 pre-activation gradients
        float dw3 = 0.f, db2 = 0.f, db1 = 0.f;
#pragma unroll
        for (int mi = 0; mi < 4; mi++) {
            uint16_t gb[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int s = 16 * mi + 4 * kb + r;
                const float dys = S.DY[s];
                dw3 += dys * a2[mi][r];
                const float dz = dys * w3 * mlp_act_grad(z2[mi][r]);
                db2 += dz;
                gb[r] = f2bf(dz);
                S.G2[s * kHS + u] = gb[r];
            }
            store_bf16x4(&S.G2T[u * kHS + 16 * mi + 4 * kb], gb);
        }
        gw3 += dw3;
        gb2 += db2;
        __syncthreads();

        // dW2[o][i] = sum_s dZ2[s][o] A1[s][i], columns i = u
        pm_bf16x8 b[2];
#pragma unroll
        for (int kk = 0; kk < 2; kk++) b[kk] = load_bf16x8(S.H1T + u * kHS + 32 * kk + 8 * kb);
        train_gemm<4, 2>(S.G2T, kHS, b, gW2);

        // dA1[s][i] = sum_o dZ2[s][o] W2[o][i]; dZ1 = dA1 * act'(Z1)
        pm_f32x4 dA1[4] = { zero, zero, zero, zero };
        train_gemm<4, 2>(S.G2, kHS, bw2t, dA1);
#pragma unroll
        for (int mi = 0; mi < 4; mi++) {
            uint16_t gb[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float dz = dA1[mi][r] * mlp_act_grad(z1[mi][r]);
                db1 += dz;
                gb[r] = f2bf(dz);
            }
            store_bf16x4(&S.G1T[u * kHS + 16 * mi + 4 * kb], gb);
        }
        gb1 += db1;
        wave_lds_sync();               // G1T rows 16 w .. 16 w + 15 are this wave's own

        // dW1[i][f] = sum_s dZ1[s][i] X[s][f], rows i of this wave (A and B swapped
        // in train_gemm's terms: its result's rows are f, its columns i = u)
#pragma unroll
        for (int kk = 0; kk < 2; kk++) b[kk] = load_bf16x8(S.G1T + u * kHS + 32 * kk + 8 * kb);
        train_gemm<2, 2>(S.XT, kHS, b, gW1);
        __syncthreads();               // the next group's inputs overwrite X and XT
    }

    gw3 += __shfl_xor(gw3, 16, 64);
    gw3 += __shfl_xor(gw3, 32, 64);
    gb2 += __shfl_xor(gb2, 16, 64);
    gb2 += __shfl_xor(gb2, 32, 64);
    gb1 += __shfl_xor(gb1, 16, 64);
    gb1 += __shfl_xor(gb1, 32, 64);
    if (kb == 0) {
        part[PM_MLP_OFF_W3 + u] = gw3;
        part[PM_MLP_OFF_B2 + u] = gb2;
        part[PM_MLP_OFF_B1 + u] = gb1;
    }
#pragma unroll
    for (int mi = 0; mi < 4; mi++)
#pragma unroll
        for (int r = 0; r < 4; r++) part[PM_MLP_OFF_W2 + (16 * mi + 4 * kb + r) * PM_MLP_H + u] = gW2[mi][r];
#pragma unroll
    for (int mi = 0; mi < 2; mi++)
#pragma unroll
        for (int r = 0; r < 4; r++) part[PM_MLP_OFF_W1 + u * PM_MLP_K1 + 16 * mi + 4 * kb + r] = gW1[mi][r];

    // db3 and the loss: wave sums
    if (w == 0) {
        for (int off = 32; off > 0; off >>= 1) {
            gb3 += __shfl_xor(gb3, off, 64);
            loss += __shfl_xor(loss, off, 64);
        }
        if (l == 0) {
            part[PM_MLP_OFF_B3] = gb3;
            part[PM_MLP_NPARAM] = loss;
        }
    }
}

// Sum of the workgroups' partials for every parameter and the loss; with apply
// != 0, one Adam step on the FP32 master and the BF16 copies.  A workgroup
// takes 64 parameters (a 256-byte run of every partial) and wave k the partials
// k, k + 16, ...; wave 0 adds the 16 sums in order, so the result does not
// depend on timing.  One thread per parameter left 25 workgroups with a serial
// chain over all partials: 15.2 us for 4,096 rows and 238 for 65,536, now 3.3 and 4.1.
__global__ __launch_bounds__(1024) void k_mlp_adam(AdamArgs a)
{
    __shared__ float sum[16][64];
    const uint32_t l = threadIdx.x & 63, k = threadIdx.x >> 6, i = blockIdx.x * 64 + l;
    float g = 0.0f;
    if (i <= PM_MLP_NPARAM)
#pragma unroll 8
        for (uint32_t w = k; w < a.nparts; w += 16) g += a.partial[(uint64_t)w * (PM_MLP_NPARAM + 1) + i];
    sum[k][l] = g;
    __syncthreads();
    if (k != 0 || i > PM_MLP_NPARAM) return;
    float gsum = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; j++) gsum += sum[j][l];
    if (i == PM_MLP_NPARAM) {
        a.loss_out[0] = gsum;
        return;
    }
    if (a.grad_out) a.grad_out[i] = gsum;
    if (!a.apply) return;
    float m = a.b1 * a.m[i] + (1.0f - a.b1) * gsum;
    float v = a.b2 * a.v[i] + (1.0f - a.b2) * gsum * gsum;
    a.m[i] = m;
    a.v[i] = v;
    float mh = m / a.bc1, vh = v / a.bc2;
    float p = a.p[i] - a.lr * mh / (sqrtf(vh) + a.eps);
    if (i < PM_MLP_OFF_B1 && (i % PM_MLP_K1) >= PM_MLP_IN) p = 0.0f;   // padding inputs stay zero
    a.p[i] = p;
}

__global__ __launch_bounds__(256) void k_mlp_sync_bf16(const float *__restrict__ p, uint16_t *__restrict__ W1,
                                                       uint16_t *__restrict__ W2, uint16_t *__restrict__ W2T)
{
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < PM_MLP_H * PM_MLP_K1) W1[i] = f2bf(p[PM_MLP_OFF_W1 + i]);
    if (i < PM_MLP_H * PM_MLP_H) {
        uint16_t b = f2bf(p[PM_MLP_OFF_W2 + i]);
        uint32_t o = i / PM_MLP_H, in = i % PM_MLP_H;
        W2[i] = b;
        W2T[in * PM_MLP_H + o] = b;
    }
}

hipError_t launch_mlp_train(const TrainArgs &a, uint32_t nblocks, hipStream_t st)
{
    hipLaunchKernelGGL(k_mlp_train, dim3(nblocks), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_mlp_adam(const AdamArgs &a, hipStream_t st)
{
    hipLaunchKernelGGL(k_mlp_adam, dim3((PM_MLP_NPARAM + 1 + 63) / 64), dim3(1024), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_mlp_sync(const float *p, uint16_t *W1, uint16_t *W2, uint16_t *W2T, hipStream_t st)
{
    hipLaunchKernelGGL(k_mlp_sync_bf16, dim3((PM_MLP_H * PM_MLP_H + 255) / 256), dim3(256), 0, st, p, W1, W2, W2T);
    return hipGetLastError();
}

// ---------------------------------------------------------- batch forward --

__global__ __launch_bounds__(64) void k_mlp_forward(MlpDev net, const float *__restrict__ feat, uint32_t n,
                                                    float *__restrict__ y)
{
    __shared__ uint16_t X[64 * PM_MLP_K1];
    __shared__ uint16_t H[64 * 64];
    __shared__ float Y[64];
    const int l = threadIdx.x;
    uint32_t s = blockIdx.x * 64 + l;
    for (int j = 0; j < PM_MLP_K1; j++)
        X[l * PM_MLP_K1 + j] = (j < PM_MLP_IN && s < n) ? f2bf(feat[(uint64_t)s * PM_MLP_IN + j]) : (uint16_t)0;
    wave_lds_sync();
    float out = mlp_wave_forward(net, X, H, Y);
    if (s < n) y[s] = out;
}

hipError_t launch_mlp_forward(const MlpDev &net, const float *feat, uint32_t n, float *y, hipStream_t st)
{
    hipLaunchKernelGGL(k_mlp_forward, dim3((n + 63) / 64), dim3(64), 0, st, net, feat, n, y);
    return hipGetLastError();
}

}  // namespace pm
