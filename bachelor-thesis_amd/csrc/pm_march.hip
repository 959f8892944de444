// pm_march.hip -- the per-pixel iso-surface march on CDNA4.
//
// Replaces RayMarcher::PerPixel_Isotropic (RayMarcher.cpp:256-344) and the
// ThreadPool that drives it (ThreadPool.cpp:38-55).
//
// Work mapping: one wave64 per 8x8 pixel tile, one ray per lane.  A tile
// pre-pass lists the tiles a ray of which can hit; the march kernel takes one
// listed tile per wave up to each ray's hit bracket or miss, the finish kernel
// then takes the same tiles through bisection, FP64 step, normal and outputs.
// In each kernel every lane does the same kind of work at the same time: the
// march ends where its rays' work would diverge.  (One kernel that bisected a
// ray's hit while other lanes of the wave still marched took 23 density
// evaluations per wave at the median, 1.11 ms at 1080p on the 1 M dam break;
// split, 0.33 + 0.46 ms, now 0.28 + 0.25.)  Schedule 1 (k_march_simple) marches one ray per lane
// to its end with a direct walk for every sample: the plain form the product
// is checked against.
#include "pm_features.h"
#include "pm_internal.h"
#include "pm_ray.h"
#include "pm_tiles.h"

namespace pm {

// FP32 density through the lane's candidate list (compensated or plain sum).
// CAP: 36 candidates -- near the surface a stencil holds about 41, so most
// samples take their list once or twice -- and 10 KB of LDS per wave, which
// keeps 16 waves on a CU.
static constexpr int kListCap = 36;
static constexpr int kListWords = (kListCap + kListPad) * 64;   // per wave
// The finish kernel's list of a whole segment, unfiltered row by row: in the
// 1 M dam break the filtered lists hold up to 41 candidates and a row up to
// about 10 more.  Measured there (finish kernel): 36 slots 433 us, 48 355,
// 52 226, 56 223, 60 231 (15 KB of LDS at 56 leave ten waves on a CU).
static constexpr int kFinCap = 56, kFinWords = (kFinCap + kListPad) * 64;

struct DensList {
    const GridDev *g;
    uint32_t *lst;
    bool comp;
    __device__ float operator()(float x, float y, float z, uint32_t &cand) const
    {
        return pm_density32_list<kListCap>(*g, x, y, z, comp, lst, cand);
    }
};

static constexpr int kLdsCap = 32;   // floats per lane of the six-sample walk's compaction

// Tile pre-pass: the 8x8 tiles one of whose rays enters the padded AABB (the ray
// set-up and slab test of ray_setup, bit for bit) -- in reference mode, one of
// whose pixels has a depth other than 1.  The march takes only these active
// tiles; the others' pixels are misses.
__device__ __forceinline__ bool tile_ray_active(const MarchLaunch &L, uint32_t px, uint32_t py)
{
    if (px >= L.W || py >= L.H) return false;
    if (L.s.mode == PM_MODE_REFERENCE) return L.depth[py * L.W + px] != 1.0f;
    const float cx = (float)px * (2.0f / (float)L.W) - 1.0f;
    const float cy = (float)py * (2.0f / (float)L.H) - 1.0f;
    float wx, wy, wz, d[3], tn, tf;
    pm_unproject(L.M, cx, cy, 1.0f, wx, wy, wz);
    pm_normalize(wx - L.cam[0], wy - L.cam[1], wz - L.cam[2], d[0], d[1], d[2]);
    const float o[3] = { L.cam[0], L.cam[1], L.cam[2] };
    return pm_slab(o, d, L.g.bmin, L.g.bmax, tn, tf);
}

// Two launches list the active tiles in row order and write the misses of the
// others: tile_buf[0, count) the tiles, tile_buf[T] = count, then (64-bit
// aligned) one mask of active tiles per 64.  The first takes 64 tiles per
// workgroup, four per wave; the second adds up the masks before its own, which
// at these sizes (507 masks at 1080p) is cheaper than a scan's launches.  Beyond
// kSumMasks masks a launch between them sums the masks 64 at a time, and the
// second adds up those (32768x16384, nothing hit: 8.1 ms without, 4.5 with; 7680x4320,
// 8,100 masks: 353 and 323 us).  Bound
// by the miss writes (36 B per ray).  (Flags, a three-launch scan, a compaction
// and the misses were six launches: 45 us at 1080p, 17 at 96x64.  One launch
// that appended each workgroup's tiles with an atomic saved 3 us more but lost
// the row order: march kernel of the 640x480 lattice cube 228 -> 337 us, finish
// kernel of the 4K pool 3.6 -> 4.0 ms.)
__device__ __forceinline__ unsigned long long *tile_masks(const MarchLaunch &L, uint32_t T)
{
    return (unsigned long long *)(L.tile_buf + ((T + 2u) & ~1u));
}

__global__ __launch_bounds__(1024) void k_tile_masks(MarchLaunch L, uint32_t T)
{
    __shared__ uint32_t nib[16];
    const uint32_t wave = threadIdx.x >> 6, j = threadIdx.x & 63u, tiles_x = (L.W + 7) / 8;
    const uint32_t t0 = blockIdx.x * 64 + wave * 4;
    if (blockIdx.x == 0 && threadIdx.x < (uint32_t)kCtrWords) L.counters[threadIdx.x] = 0ull;   // the march's, before it
    uint32_t m = 0;
    for (uint32_t k = 0; k < 4 && t0 + k < T; k++) {
        const uint32_t t = t0 + k;
        const uint32_t px = (t % tiles_x) * 8 + (j & 7u), py = (t / tiles_x) * 8 + (j >> 3);
        if (__ballot(tile_ray_active(L, px, py)) != 0) m |= 1u << k;
        else if (px < L.W && py < L.H) write_miss(L, py * L.W + px);
    }
    if (j == 0) nib[wave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long mask = 0;
        for (uint32_t w = 0; w < 16; w++) mask |= (unsigned long long)nib[w] << (4 * w);
        tile_masks(L, T)[blockIdx.x] = mask;
    }
}

static constexpr uint32_t kSumMasks = 4096;
__device__ __forceinline__ uint32_t *mask_sums(const MarchLaunch &L, uint32_t T)
{
    return (uint32_t *)(tile_masks(L, T) + (T + 63) / 64);
}

// The active tiles of 64 masks, a wave each.
__global__ __launch_bounds__(64) void k_mask_sums(MarchLaunch L, uint32_t T)
{
    const uint32_t i = blockIdx.x * 64 + threadIdx.x;
    uint32_t n = i < (T + 63) / 64 ? (uint32_t)__popcll(tile_masks(L, T)[i]) : 0u;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    if (threadIdx.x == 0) mask_sums(L, T)[blockIdx.x] = n;
}

// summed: k_mask_sums ran.
__global__ __launch_bounds__(64) void k_tile_list(MarchLaunch L, uint32_t T, int summed)
{
    const unsigned long long *masks = tile_masks(L, T);
    const uint32_t b = blockIdx.x, lane = threadIdx.x, first = summed ? b & ~63u : 0u;
    uint32_t before = 0;
    if (summed) {
        const uint32_t *sums = mask_sums(L, T);
        for (uint32_t i = lane; i < b / 64; i += 64) before += sums[i];
    }
    for (uint32_t i = first + lane; i < b; i += 64) before += (uint32_t)__popcll(masks[i]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
    const unsigned long long m = masks[b];
    if ((m >> lane) & 1ull) L.tile_buf[before + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = b * 64 + lane;
    if (b == gridDim.x - 1 && lane == 0) L.tile_buf[T] = before + (uint32_t)__popcll(m);
}

// The flags and the misses on their own (a batch lists its tiles on the host):
// tile_buf[t] = 1 for an active tile, tile_buf[T] = 0.
__global__ __launch_bounds__(256) void k_tile_flags(MarchLaunch L, uint32_t T)
{
    // one wave per tile, one lane per ray
    const uint32_t t = blockIdx.x * 4 + (threadIdx.x >> 6), j = threadIdx.x & 63u;
    if (t > T) return;   // whole wave
    const uint32_t tiles_x = (L.W + 7) / 8;
    const bool enters = t < T && tile_ray_active(L, (t % tiles_x) * 8 + (j & 7u), (t / tiles_x) * 8 + (j >> 3));
    const unsigned long long m = __ballot(enters);
    if (j == 0) L.tile_buf[t] = m != 0ull ? 1u : 0u;
}

// Pixels of the inactive tiles are written as misses here.  (They are not
// counted on the device: one counter for every wave would serialise on a
// single address; the host knows the ray total.)
__global__ __launch_bounds__(256) void k_miss_tiles(MarchLaunch L, uint32_t T)
{
    const uint32_t t = blockIdx.x * 4 + (threadIdx.x >> 6), j = threadIdx.x & 63u;
    if (t >= T) return;   // whole wave
    if (L.tile_buf[t] == 0) {
        const uint32_t tiles_x = (L.W + 7) / 8;
        const uint32_t px = (t % tiles_x) * 8 + (j & 7u), py = (t / tiles_x) * 8 + (j >> 3);
        if (px < L.W && py < L.H) write_miss(L, py * L.W + px);
    }
}

// Schedule 1: one 8x8 tile per wave, one ray per lane to its end -- march,
// bisection, FP64 step, normal, outputs -- every sample with its own direct
// walk (no compaction, no lists, no hit records).  The plain form of the
// configured march the product is checked against.
__global__ __launch_bounds__(256) void k_march_simple(MarchLaunch L)
{
    uint32_t px, py;
    Counts cn;
    const pm_settings &s = L.s;
    const GridDev &g = L.g;
    const bool comp = s.compensated != 0;
    if (pm_tile(L.W, L.H, px, py) && px < L.W && py < L.H) {
        RayState r{};
        cn.rays++;
        r.idx = py * L.W + px;
        float d[3];
        pm_ray_dir(L, px, py, d);
        r.d0 = d[0]; r.d1 = d[1]; r.d2 = d[2];
        r.id0 = 1.0f / d[0]; r.id1 = 1.0f / d[1]; r.id2 = 1.0f / d[2];
        const float o[3] = { L.cam[0], L.cam[1], L.cam[2] };
        bool hit = false;
        if (pm_slab(o, d, g.bmin, g.bmax, r.tn, r.tf)) {
            cn.in_aabb++;
            r.k = 0;
            for (;;) {
                const float t = r.tn + (float)r.k * s.step;
                if (t > r.tf || (s.max_steps > 0 && r.k >= s.max_steps)) break;
                const float qx = o[0] + t * d[0], qy = o[1] + t * d[1], qz = o[2] + t * d[2];
                int kn = r.k;
                if (s.skip_mode == PM_SKIP_BOUND) kn = pm_skip_bound(g, o[0], o[1], o[2], r, qx, qy, qz, L.inv_step);
                else if (s.skip_mode == PM_SKIP_EMPTY) kn = pm_skip_empty(g, o[0], o[1], o[2], r, qx, qy, qz, s.step);
                if (kn != r.k) { r.k = kn; continue; }
                uint32_t cand = 0;
                const float rho = pm_density32(g, qx, qy, qz, comp, cand);
                cn.samples++; cn.march++; cn.cand += cand; cn.mcand += cand;
                if (rho >= s.iso) { hit = true; break; }
                r.k++;
            }
        }
        if (!hit) {
            write_miss(L, r.idx);
        } else {
            const bool fp64 = s.final_fp64 && s.bisect_iters > 0;
            const int n32 = fp64 ? s.bisect_iters - 1 : s.bisect_iters;
            float lo = r.tn + (float)(r.k - 1) * s.step, hi = r.tn + (float)r.k * s.step;
            float xs[3], th;
            if (r.k == 0) {
                th = r.tn;
                xs[0] = o[0] + th * d[0]; xs[1] = o[1] + th * d[1]; xs[2] = o[2] + th * d[2];
            } else {
                for (int it = 0; it < n32; it++) {
                    const float tm = (lo + hi) * 0.5f;
                    uint32_t cand = 0;
                    const float rho = pm_density32(g, o[0] + tm * d[0], o[1] + tm * d[1], o[2] + tm * d[2], comp, cand);
                    cn.samples++; cn.cand += cand;
                    if (rho >= s.iso) hi = tm; else lo = tm;
                }
                if (fp64) {
                    const double tmd = ((double)lo + (double)hi) * 0.5;
                    const double rho = pm_density64(g, (double)o[0] + tmd * (double)d[0], (double)o[1] + tmd * (double)d[1],
                                                    (double)o[2] + tmd * (double)d[2]);
                    cn.samples++;
                    double dlo = lo, dhi = hi;
                    if (rho >= (double)s.iso) dhi = tmd; else dlo = tmd;
                    const double tt = (dlo + dhi) * 0.5;
#pragma unroll
                    for (int a = 0; a < 3; a++) xs[a] = (float)((double)o[a] + tt * (double)d[a]);
                    th = (float)tt;
                } else {
                    th = (lo + hi) * 0.5f;
                    xs[0] = o[0] + th * d[0]; xs[1] = o[1] + th * d[1]; xs[2] = o[2] + th * d[2];
                }
            }
            float nx, ny, nz;
            if (s.normal_mode == PM_NORMAL_GRADW) {
                float sx, sy, sz;
                uint32_t cand = 0;
                pm_sum_gradw(g, xs[0], xs[1], xs[2], sx, sy, sz, cand);
                cn.cand += cand;
                pm_normalize(sx, sy, sz, nx, ny, nz);
            } else {
                float gv[3];
                for (int j = 0; j < 6; j++) {
                    float q[3] = { xs[0], xs[1], xs[2] };
                    q[j >> 1] = (j & 1) ? xs[j >> 1] - s.normal_eps : xs[j >> 1] + s.normal_eps;
                    uint32_t cand = 0;
                    const float rho = pm_density32(g, q[0], q[1], q[2], comp, cand);
                    cn.samples++; cn.cand += cand;
                    if (j & 1) gv[j >> 1] -= rho; else gv[j >> 1] = rho;
                }
                const float dd = (gv[0] * gv[0] + gv[1] * gv[1]) + gv[2] * gv[2];
                nx = ny = nz = 0.0f;
                if (dd > 0.0f) {
                    const float inv = 1.0f / sqrtf(dd);
                    nx = -gv[0] * inv; ny = -gv[1] * inv; nz = -gv[2] * inv;
                }
            }
            L.pos[r.idx] = make_float4(xs[0], xs[1], xs[2], 1.0f);
            L.nrm[r.idx] = make_float4(nx, ny, nz, 1.0f);
            if (L.t) L.t[r.idx] = th;
            cn.hits++;
        }
    }
    flush_counts(L.counters, cn);
}

// ---- learned step proposal with certified jumps ----
// An upper bound U of the density over every point within `margin` of the
// segment [a, b]: the sum over the particles near the segment of W at their
// distance to the segment less the margin.  W falls with the distance, so
// rho(q) <= U for every such q.  The walk covers the march-grid cells near the
// segment's box (pm_box_begin); it stops once every lane's U reached lim.
// INFINITY when those cells leave the grid (nothing is certified).
__device__ __forceinline__ float pm_segment_bound(const GridDev &g, const float a[3], const float b[3], float margin,
                                                  float lim, uint32_t &cand)
{
    float lo[3], hi[3], u[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        lo[k] = fminf(a[k], b[k]) - margin;
        hi[k] = fmaxf(a[k], b[k]) + margin;
        u[k] = b[k] - a[k];
    }
    BoxWalk w;
    if (!pm_box_begin(g, lo, hi, w)) return INFINITY;
    const float uu = (u[0] * u[0] + u[1] * u[1]) + u[2] * u[2];
    const float iuu = uu > 0.0f ? 1.0f / uu : 0.0f;
    float U = 0.0f;
    const int nr = w.ny * w.nz;
    int jy = 0, jz = 0;
    _Pragma("unroll 1") for (int r = 0; __ballot(r < nr && U < lim) != 0; r++) {
        uint32_t rb, re;
        pm_box_row(g, w, jy, jz, rb, re);
        if (++jy == w.ny) { jy = 0; jz++; }
        if (!(U < lim)) continue;
        cand += re - rb;
        for (uint32_t i = rb; i < re; i++) {
            const float4 p = g.fsorted[i];
            const float ax = p.x - a[0], ay = p.y - a[1], az = p.z - a[2];
            const float sp = fminf(fmaxf(((ax * u[0] + ay * u[1]) + az * u[2]) * iuu, 0.0f), 1.0f);
            const float dx = ax - sp * u[0], dy = ay - sp * u[1], dz = az - sp * u[2];
            const float dist = sqrtf((dx * dx + dy * dy) + dz * dz) - margin;
            if (dist < g.h) {
                const float dl = fmaxf(dist, 0.0f);
                U += pm_W_in(dl * dl, g.inv_h, g.sig);
            }
        }
    }
    return U;
}

// A step proposal for every lane in PH_PROPOSE (want), all at once: features at
// the lane's current sample k (its density rho is known; one fine-stencil pass
// for grad rho), one MLP evaluation for the whole wave (BF16 MFMA), a jump of
// n samples, and the certificate of the samples k+1 .. k+n-1 it passes over:
// the segment bound U < iso (1 - 2^-9), which covers the rounding of the bound
// and of the samples' own FP32 densities.  A certified lane next evaluates
// sample k+n exactly; the others step to k+1 and ask for no proposal until the
// exact skip next moves them.  Every sample the learned march does not
// evaluate lies below iso, so its first crossing -- and its image -- are the
// plain march's.  Called by all 64 lanes together, with the ray's state passed
// in and out by value.  (Kept inline: as a call, the kernel reserved 0.8 KB of
// stack per lane for the registers live across it and ran 30 % slower even
// without proposals.)
struct Proposal {
    int k, lrn;
    uint32_t mlp, cert, cskip, cand;
};

__device__ __forceinline__ Proposal wave_propose(const MarchLaunch &L, bool want, int k, float tn, float tf, float d0,
                                              float d1, float d2, float rho, uint16_t *X, uint16_t *H, float *Y)
{
    const int l = threadIdx.x & 63;
    const pm_settings &s = L.s;
    const GridDev &g = L.g;
    Proposal o{ k, 1, 0u, 0u, 0u, 0u };
    float f[PM_MLP_IN];
#pragma unroll
    for (int j = 0; j < PM_MLP_IN; j++) f[j] = 0.0f;
    const float t = tn + (float)k * s.step;
    if (want) {
        const float q0 = L.cam[0] + t * d0, q1 = L.cam[1] + t * d1, q2 = L.cam[2] + t * d2;
        float gx, gy, gz;
        uint32_t cand = 0;
        grad_feat(g, q0, q1, q2, gx, gy, gz, cand);
        o.cand += cand;
        const float d[3] = { d0, d1, d2 };
        mlp_features(g, L.cg, L.cam, d, t, tn, tf, rho, sqrtf((gx * gx + gy * gy) + gz * gz),
                     (float)pm_cand27(g, q0, q1, q2), s.iso, f);
    }
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < PM_MLP_K1; j++) X[l * PM_MLP_K1 + j] = j < PM_MLP_IN ? f2bf(f[j]) : (uint16_t)0;
    wave_lds_sync();
    const float y = mlp_wave_forward_halves(L.net, X, H, Y);
    wave_lds_sync();
    int n = 0;
    if (want) {
        o.mlp = 1;
        const float dist = g.h * (exp2f(fminf(y, 8.0f)) - 1.0f);
        const float sk = fminf(floorf(L.mlp_alpha * dist * L.inv_step), (float)L.mlp_max_skip);
        int kmax = (int)floorf((tf - tn) * L.inv_step);           // last sample inside the AABB
        while (kmax > 0 && tn + (float)kmax * s.step > tf) kmax--;
        if (sk >= (float)L.mlp_min_skip && k + (int)sk <= kmax) n = (int)sk;
        if (n < 2) {
            o.lrn = 0;
            o.k = k + 1;
        }
    }
    const bool cert = want && n >= 2;
    if (__ballot(cert) == 0) return o;
    const float lim = s.iso * (1.0f - 0x1p-9f);
    if (cert) {
        const float ta = tn + (float)(k + 1) * s.step, tb = tn + (float)(k + n - 1) * s.step;
        const float a[3] = { L.cam[0] + ta * d0, L.cam[1] + ta * d1, L.cam[2] + ta * d2 };
        const float b[3] = { L.cam[0] + tb * d0, L.cam[1] + tb * d1, L.cam[2] + tb * d2 };
        // the lattice samples between a and b lie within a few ulps of the
        // segment; the margin covers them and the rounding of the distances
        float m = g.h;
#pragma unroll
        for (int c = 0; c < 3; c++) m = fmaxf(m, fmaxf(fabsf(a[c]), fabsf(b[c])));
        uint32_t cand = 0;
        const float U = pm_segment_bound(g, a, b, m * 0x1p-18f, lim, cand);
        o.cand += cand;
        o.cert = 1;
        if (U < lim) {
            o.k = k + n;
            o.cskip = (uint32_t)(n - 1);
        } else {
            o.k = k + 1;
            o.lrn = 0;
        }
    }
    return o;
}

// The proposals of a wave and their transitions (all 64 lanes).
__device__ __forceinline__ void wave_propose_step(const MarchLaunch &L, RayState &r, Counts &cn, float *region)
{
    const bool want = r.phase == PH_PROPOSE;
    const Proposal o = wave_propose(L, want, r.k, r.tn, r.tf, r.d0, r.d1, r.d2, r.rho, (uint16_t *)region,
                                    (uint16_t *)region + 64 * PM_MLP_K1, region + 2048);
    if (want) {
        r.k = o.k;
        r.lrn = o.lrn;
        r.phase = PH_MARCH;
        cn.mlp += o.mlp;
        cn.cert += o.cert;
        cn.cskip += o.cskip;
        cn.cand += o.cand;
    }
}

// ---- finish ----
// Per hit record: the bisection of the bracket (the last step in FP64 when the
// settings ask for it), the normal (the six central differences in one fused
// walk, or the sum of gradW) and the pixel's outputs.  Every lane of a wave does the same kind of work
// and none of the march's state is held, so this runs packed and short; the
// march kernels keep only the phases that decide where the hit is.
template <bool INSTR, bool LIST>
__device__ __forceinline__ void finish_hit(const MarchLaunch &L, uint32_t px, uint32_t py, uint4 rec, uint32_t *lst,
                                           Counts &cn)
{
    const pm_settings &s = L.s;
    const GridDev &g = L.g;
    const uint32_t idx = py * L.W + px;
    float lo = __uint_as_float(rec.y), hi = __uint_as_float(rec.z);
    float d[3];
    pm_ray_dir(L, px, py, d);
    const float o0 = L.cam[0], o1 = L.cam[1], o2 = L.cam[2];
    float xs[3], th;
    const bool comp = s.compensated != 0;
    const bool fp64 = s.final_fp64 && s.bisect_iters > 0;
    const bool bracket = (rec.x & 2u) != 0;
    const float e = s.normal_mode == PM_NORMAL_CDIFF ? s.normal_eps : 0.0f;
    int n = 0;
    bool listed = false;
    if (LIST) {
        const float o[3] = { o0, o1, o2 };
        listed = pm_list_segment<kFinCap>(g, o, d, lo, hi, fabsf(e), lst, n);
    }
    if (bracket) {
        const int n32 = fp64 ? s.bisect_iters - 1 : s.bisect_iters;
#pragma unroll 1
        for (int it = 0; it < n32; it++) {
            const float tm = (lo + hi) * 0.5f;
            const float qx = o0 + tm * d[0], qy = o1 + tm * d[1], qz = o2 + tm * d[2];
            uint32_t cand = 0, nsup = 0;
            float rho;
            if (listed) {
                float sum = 0.0f, c = 0.0f;
                pm_list_density(g, lst, n, qx, qy, qz, sum, c, nsup);
                rho = comp ? sum + c : sum;
                cand = pm_stencil_cand(g, qx, qy, qz);
            } else {
                rho = pm_density32_list<kListCap>(g, qx, qy, qz, comp, lst, cand);
            }
            count_sample<INSTR>(g, qx, qy, qz, cand, false, cn);
            if (rho >= s.iso) hi = tm; else lo = tm;
        }
        if (!fp64) lo = hi = (lo + hi) * 0.5f;
    }
    if (bracket && fp64) {
        // the last bisection step in double (RayMarcher.cpp:316-326 in FP64)
        const double tmd = ((double)lo + (double)hi) * 0.5;
        const double x = (double)o0 + tmd * (double)d[0];
        const double y = (double)o1 + tmd * (double)d[1];
        const double z = (double)o2 + tmd * (double)d[2];
        const double rho = listed ? pm_list_density64(g, lst, n, x, y, z) : pm_density64(g, x, y, z);
        cn.samples++;
        if (INSTR) {
            cn.cst += pm_stencil_cand(g, (float)x, (float)y, (float)z);
            cn.c27 += pm_cand27(g, (float)x, (float)y, (float)z);
        }
        double dlo = lo, dhi = hi;
        if (rho >= (double)s.iso) dhi = tmd; else dlo = tmd;
        const double tt = (dlo + dhi) * 0.5;
        xs[0] = (float)((double)o0 + tt * (double)d[0]);
        xs[1] = (float)((double)o1 + tt * (double)d[1]);
        xs[2] = (float)((double)o2 + tt * (double)d[2]);
        th = (float)tt;
    } else {
        th = lo;
        xs[0] = o0 + th * d[0]; xs[1] = o1 + th * d[1]; xs[2] = o2 + th * d[2];
    }
    float nx, ny, nz;
    if (s.normal_mode == PM_NORMAL_GRADW) {
        float sx, sy, sz;
        uint32_t cand = 0;
        pm_sum_gradw(g, xs[0], xs[1], xs[2], sx, sy, sz, cand);
        pm_normalize(sx, sy, sz, nx, ny, nz);
    } else {
        float gv[3];
        if (listed) {
            float v[6];
            pm_list_cdiff6(g, lst, n, xs, e, comp, v);
            cn.samples += 6;
            cn.cand += pm_box_cand(g, xs, e);
            gv[0] = v[0] - v[1]; gv[1] = v[2] - v[3]; gv[2] = v[4] - v[5];
        } else {
            const Cdiff6 o = pm_cdiff6_lds<kLdsCap>(g, xs[0], xs[1], xs[2], e, (float *)lst, comp);
            if (o.cand != 0xffffffffu) {
                cn.samples += 6;
                cn.cand += o.cand;
                gv[0] = o.v[0] - o.v[1]; gv[1] = o.v[2] - o.v[3]; gv[2] = o.v[4] - o.v[5];
            } else {
                // the fused walk's cells leave the grid: +x, -x, +y, -y, +z, -z one at a time
#pragma unroll 1
                for (int k = 0; k < 6; k++) {
                    const float ek = (k & 1) ? -e : e;
                    const float q0 = k < 2 ? xs[0] + ek : xs[0], q1 = (k >> 1) == 1 ? xs[1] + ek : xs[1],
                                q2 = k > 3 ? xs[2] + ek : xs[2];
                    uint32_t cand = 0;
                    const float rho = pm_density32_list<kListCap>(g, q0, q1, q2, comp, lst, cand);
                    cn.samples++;
                    cn.cand += cand;
#pragma unroll
                    for (int a = 0; a < 3; a++)
                        if ((k >> 1) == a) gv[a] = (k & 1) ? gv[a] - rho : rho;
                }
            }
        }
        if (INSTR) {
#pragma unroll 1
            for (int k = 0; k < 6; k++) {
                float q[3] = { xs[0], xs[1], xs[2] };
                q[k >> 1] = (k & 1) ? xs[k >> 1] - e : xs[k >> 1] + e;
                cn.cst += pm_stencil_cand(g, q[0], q[1], q[2]);
                cn.c27 += pm_cand27(g, q[0], q[1], q[2]);
            }
        }
        // RayMarcher.cpp:331-338 with central differences
        const float dd = (gv[0] * gv[0] + gv[1] * gv[1]) + gv[2] * gv[2];
        nx = ny = nz = 0.0f;
        if (dd > 0.0f) {
            const float inv = 1.0f / sqrtf(dd);
            nx = -gv[0] * inv; ny = -gv[1] * inv; nz = -gv[2] * inv;
        }
    }
    L.pos[idx] = make_float4(xs[0], xs[1], xs[2], 1.0f);
    L.nrm[idx] = make_float4(nx, ny, nz, 1.0f);
    if (L.t) L.t[idx] = th;
}

// One 8x8 tile per wave, one pixel per lane: the lanes whose pixel holds a
// hit record finish it.
template <bool INSTR, bool LIST>
__device__ __forceinline__ void finish_tile(const MarchLaunch &L, uint32_t tile, uint32_t *lst, Counts &cn)
{
    const uint32_t lane = threadIdx.x & 63, tiles_x = (L.W + 7) / 8;
    const uint32_t px = (tile % tiles_x) * 8 + (lane & 7u), py = (tile / tiles_x) * 8 + (lane >> 3);
    if (px >= L.W || py >= L.H) return;
    const uint4 rec = L.hit_rec[py * L.W + px];
    if (rec.x & 1u) finish_hit<INSTR, LIST>(L, px, py, rec, lst, cn);
}

// Schedule 0: a wave per active 8x8 tile (or several, tile_split), one ray per
// lane or lane group up to the ray's hit or miss.  As rays end, the others spread over the idle lanes (lane
// groups), so the tile's last rays take several samples per step.  The tiles
// come from the list by position: no queue.  (Persistent waves that drew tiles
// from counters spent 0.30 of 0.64 ms at 1080p on the counters: 4,096 waves
// each found all eight bands empty, one serialised atomic per band.)
// LEARNED adds the step proposals; its LDS region holds either the lanes'
// candidate lists or the network's activations (never both at once).
// INSTR adds the per-sample counts of instrumented launches.
template <bool LEARNED, bool INSTR>
__device__ __forceinline__ void march_part(const MarchLaunch &L, uint32_t tile, uint32_t i, uint32_t sub, float *region,
                                           Counts &cn)
{
    const uint32_t lane = threadIdx.x;
    uint32_t *lst = (uint32_t *)region + lane;
    const bool comp = L.s.compensated != 0;
    uint32_t px, py;
    part_pixel(tile, (L.W + 7) / 8, i, sub, lane >> sub, px, py);
    RayState r{};
    r.phase = PH_DONE;
    int G = 1 << sub;
    if (px < L.W && py < L.H) ray_setup(L, r, px, py, cn, (lane & (uint32_t)(G - 1)) == 0);
    while (__ballot(r.phase != PH_DONE) != 0) {
        // The network is batched across the wave (the wave pays for it
        // whenever any lane needs it): it runs once half of the busy
        // lanes wait for a proposal, or when few rays are left; waiting
        // lanes sit out.  Lane groups take no proposals: the learned march
        // groups its last 16 rays only.
        const int nbusy = __popcll(__ballot(r.phase != PH_DONE));
        if (LEARNED && G == 1) {
            const int nwant = __popcll(__ballot(r.phase == PH_PROPOSE));
            if (nwant > 0 && (2 * nwant >= nbusy || nbusy <= 16)) wave_propose_step(L, r, cn, region);
        }
        if (!LEARNED || nbusy <= 16) regroup(r, G, region);
        if (G == 1) {
            if (r.phase == PH_MARCH) ray_step<INSTR, 16>(L, r, DensList{ &L.g, lst, comp }, cn);
        } else {
            group_step<INSTR>(L, r, G, DensList{ &L.g, lst, comp }, cn);
        }
    }
}

template <bool LEARNED, bool INSTR>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_march_tiles(MarchLaunch L)
{
    // the lanes' candidate lists, or X[64][32] + H[32][64] bf16 + Y[64]
    static_assert(kListWords >= 2112, "network region");
    __shared__ float region[kListWords];
    const uint32_t T = ((L.W + 7) / 8) * ((L.H + 7) / 8);
    const uint32_t *order = L.tile_buf;
    const uint32_t TA = order[T];
    Counts cn;
    bool any = false;
    const uint32_t sub = LEARNED ? 0u : tile_split(TA);
    for (uint32_t w = blockIdx.x; w < tile_waves_of(TA << sub); w += gridDim.x) {
        const uint32_t i = xcd_tile(w);
        if (i >= TA << sub) continue;
        any = true;
        march_part<LEARNED, INSTR>(L, order[i >> sub], i, sub, region, cn);
    }
    if (any) flush_counts(L.counters, cn);
}

// PerPixel_Isotropic (RayMarcher.cpp:256-344): start on the depth-buffer
// surface, fixed step vector, MaxSteps samples, first sample with rho >= iso,
// normal = normalize(sum gradW) (or central differences on request).
struct RefCounts {
    uint32_t rays = 0, in = 0, hits = 0, samples = 0, ms = 0;
    unsigned long long cand = 0;
};

__device__ __forceinline__ void ref_pixel(const MarchLaunch &L, uint32_t px, uint32_t py, bool active, RefCounts &rc)
{
    const GridDev &g = L.g;
    const pm_settings &s = L.s;
    const uint32_t idx = py * L.W + px;
    const bool comp = s.compensated != 0;
    uint32_t c_rays = 0, c_in = 0, c_hits = 0, c_samples = 0, c_ms = 0;
    unsigned long long c_cand = 0;
    if (active) {
        c_rays = 1;
        float z = L.depth[idx];
        float4 P = make_float4(0.f, 0.f, 0.f, 0.f), N = make_float4(0.f, 0.f, 0.f, 0.f);
        float tout = -1.0f;
        if (z != 1.0f) {
            c_in = 1;
            float cx = (float)px * (2.0f / (float)L.W) - 1.0f;
            float cy = (float)py * (2.0f / (float)L.H) - 1.0f;
            float p0, p1, p2, d0, d1, d2;
            pm_unproject(L.M, cx, cy, z, p0, p1, p2);
            pm_normalize(p0 - L.cam[0], p1 - L.cam[1], p2 - L.cam[2], d0, d1, d2);
            float st0 = s.step * d0, st1 = s.step * d1, st2 = s.step * d2;
            for (int i = 0; i < s.max_steps; i++) {
                p0 += st0; p1 += st1; p2 += st2;
                if (s.skip_mode == PM_SKIP_DG_BOX || s.skip_mode == PM_SKIP_DG_CONS) {   // RayMarcher.cpp:284-304
                    float nmin[3], nmax[3];
                    while (pm_dg_query(g, p0, p1, p2, nmin, nmax)) {
                        float pin[3] = { p0, p1, p2 }, stv[3] = { st0, st1, st2 }, q[3];
                        pm_intersect_aabb(pin, stv, nmin, nmax, q);
                        p0 = q[0] + st0; p1 = q[1] + st1; p2 = q[2] + st2;
                    }
                }
                uint32_t cand = 0;
                float rho = pm_density32(g, p0, p1, p2, comp, cand);
                c_samples++; c_ms++; c_cand += cand;
                if (rho >= s.iso) {
                    float nx, ny, nz;
                    if (s.normal_mode == PM_NORMAL_GRADW) {
                        float sx, sy, sz;
                        uint32_t c2 = 0;
                        pm_sum_gradw(g, p0, p1, p2, sx, sy, sz, c2);
                        pm_normalize(sx, sy, sz, nx, ny, nz);
                    } else {
                        float gv[3];
                        float pp[3] = { p0, p1, p2 };
                        for (int a = 0; a < 3; a++) {
                            float xp[3] = { pp[0], pp[1], pp[2] }, xm[3] = { pp[0], pp[1], pp[2] };
                            xp[a] = pp[a] + s.normal_eps;
                            xm[a] = pp[a] - s.normal_eps;
                            uint32_t c3 = 0;
                            float rp = pm_density32(g, xp[0], xp[1], xp[2], comp, c3);
                            float rm = pm_density32(g, xm[0], xm[1], xm[2], comp, c3);
                            c_samples += 2; c_cand += c3;
                            gv[a] = rp - rm;
                        }
                        float dd = (gv[0] * gv[0] + gv[1] * gv[1]) + gv[2] * gv[2];
                        nx = ny = nz = 0.0f;
                        if (dd > 0.0f) {
                            float inv = 1.0f / sqrtf(dd);
                            nx = -gv[0] * inv; ny = -gv[1] * inv; nz = -gv[2] * inv;
                        }
                    }
                    P = make_float4(p0, p1, p2, 1.0f);
                    N = make_float4(nx, ny, nz, 1.0f);
                    float v0 = p0 - L.cam[0], v1 = p1 - L.cam[1], v2 = p2 - L.cam[2];
                    tout = sqrtf((v0 * v0 + v1 * v1) + v2 * v2);
                    c_hits = 1;
                    break;
                }
            }
        }
        L.pos[idx] = P;
        L.nrm[idx] = N;
        if (L.t) L.t[idx] = tout;
    }
    rc.rays += c_rays; rc.in += c_in; rc.hits += c_hits; rc.samples += c_samples; rc.ms += c_ms;
    rc.cand += c_cand;
}

__global__ __launch_bounds__(256) void k_march_reference(MarchLaunch L)
{
    uint32_t px, py;
    if (!pm_tile(L.W, L.H, px, py)) return;
    RefCounts rc;
    ref_pixel(L, px, py, px < L.W && py < L.H, rc);
    flush_counters(L.counters, rc.rays, rc.in, rc.hits, rc.samples, rc.cand, rc.ms);
}

// The product's reference march: the active tiles of the tile pre-pass (those
// with a pixel whose depth is not 1; the pre-pass wrote the others' misses), a
// wave per tile or part of one.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_ref_tiles(MarchLaunch L)
{
    __shared__ float region[kListWords];
    __shared__ float4 hits[64];
    uint32_t *lst = (uint32_t *)region + threadIdx.x;
    const pm_settings &s = L.s;
    const GridDev &g = L.g;
    const uint32_t tiles_x = (L.W + 7) / 8, T = tiles_x * ((L.H + 7) / 8);
    const uint32_t *order = L.tile_buf;
    const uint32_t TA = order[T], sub = tile_split(TA);
    const DensList dens{ &g, lst, s.compensated != 0 };
    Counts cn;
    bool any = false;
    auto normal = [&](const float p[3], float &nx, float &ny, float &nz) {
        if (s.normal_mode == PM_NORMAL_GRADW) {
            float sx, sy, sz;
            uint32_t cand = 0;
            pm_sum_gradw(g, p[0], p[1], p[2], sx, sy, sz, cand);
            pm_normalize(sx, sy, sz, nx, ny, nz);
            return;
        }
        float gv[3];
#pragma unroll 1
        for (int k = 0; k < 6; k++) {
            const float e = (k & 1) ? -s.normal_eps : s.normal_eps;
            uint32_t cand = 0;
            const float rho = dens(k < 2 ? p[0] + e : p[0], (k >> 1) == 1 ? p[1] + e : p[1], k > 3 ? p[2] + e : p[2], cand);
            cn.samples++;
            cn.cand += cand;
#pragma unroll
            for (int a = 0; a < 3; a++)
                if ((k >> 1) == a) gv[a] = (k & 1) ? gv[a] - rho : rho;
        }
        cdiff_normal(gv, nx, ny, nz);
    };
    for (uint32_t w = blockIdx.x; w < tile_waves_of(TA << sub); w += gridDim.x) {
        const uint32_t i = xcd_tile(w);
        if (i >= TA << sub) continue;
        any = true;
        ref_part(L, order[i >> sub], tiles_x, i, sub, region, hits, dens, normal, cn);
    }
    if (any) flush_counters(L.counters, cn.rays, cn.in_aabb, cn.hits, cn.samples, cn.cand, cn.march);
}

// The march of a batch: as k_march_tiles, over the active tiles of all views
// (B.tiles, the largest view first), each tile with its own job's grid and
// camera.  The tiles are the work items because their number bounds a small
// batch: persistent waves that drew runs of 16 tiles from a counter left most of
// the chip idle on eight views of 0.6 MP in all.  March and finish: those 4.68 ->
// 0.55 ms; one view of 0.03 MP 2.0 -> 0.28; 64 views, 23 MP, 8.4 -> 5.2; 64
// views, 45 MP of two 1,024,000-particle frames, 14.0 -> 7.4, learned 14.7 -> 8.1.
template <bool LEARNED>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_march_batch(BatchLaunch B)
{
    __shared__ float region[kListWords];
    Counts cn;
    bool any = false;
    const uint32_t sub = LEARNED ? 0u : tile_split(B.ntiles);
    for (uint32_t w = blockIdx.x; w < tile_waves_of(B.ntiles << sub); w += gridDim.x) {
        const uint32_t i = xcd_tile(w);
        if (i >= B.ntiles << sub) continue;
        any = true;
        const BatchTile bt = B.tiles[i >> sub];
        march_part<LEARNED, false>(B.jobs[__builtin_amdgcn_readfirstlane(bt.job)], bt.tile, i, sub, region, cn);
    }
    if (any) flush_counts(B.base.counters, cn);
}

// The hits of the launch, counted by its march.
__device__ __forceinline__ uint32_t marched_hits(const MarchLaunch &L)
{
    uint32_t n = 0;                               // at most 2^30 pixels
#pragma unroll
    for (int k = 0; k < kCtrSlots; k++) n += (uint32_t)(L.counters[k * kCtrStride + C_BOX_HITS] >> 32);
    return n;
}

// A wave per active tile, of the view or of the batch.
// LIST: a hit's samples share one candidate list.  It pays where the lists fit
// (GridDev::sparse, at most 2.1 particles per occupied h/2 cell); in denser frames
// most lists overflow after they were built, and their LDS costs waves, so those
// walk for each sample.  March and finish at 1920x1080, walk -> list, lattices of
// 524,288 with Gaussian jitter: 1.4 per cell 846 -> 681 us, 1.8 1138 -> 992, 2.0
// 1242 -> 1184 (at 3840x2160 2937 -> 2644), 2.04 1298 -> 1314 (an image full of hits
// 3730 -> 3657), 2.13 1417 -> 1450 (3896 -> 3939), 2.3 1453 -> 1638, 2.9 1740 -> 2005.
// The finish of the 1 M dam break, 1.4 per cell: 466 -> 223 us (now 254: the
// statistics count every sample's own stencil); of the 4 M pool, 8 per cell: 3.1 ms
// walking, 5.3 to 7.0 with lists of 44 to 92 slots.
// Registers are capped for four waves per SIMD (three with lists).
// beyond: nothing is done for launches of at most so many hits (k_finish_groups
// takes them).
template <bool BATCH, bool INSTR, bool LIST>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(LIST ? 3 : 4, 8))) void k_finish(MarchLaunch L0, const MarchLaunch *__restrict__ jobs,
                                                const BatchTile *__restrict__ tiles, uint32_t ntiles, uint32_t beyond)
{
    if (beyond != 0 && marched_hits(L0) <= beyond) return;
    __shared__ uint32_t lds[LIST ? kFinWords : kListWords];
    uint32_t *lst = lds + threadIdx.x;
    Counts cn;
    bool any = false;
    if (BATCH) {
        for (uint32_t w = blockIdx.x; w < tile_waves_of(ntiles); w += gridDim.x) {
            const uint32_t i = xcd_tile(w);
            if (i >= ntiles) continue;
            const BatchTile bt = tiles[i];
            finish_tile<INSTR, LIST>(jobs[__builtin_amdgcn_readfirstlane(bt.job)], bt.tile, lst, cn);
            any = true;
        }
    } else {
        const uint32_t T = ((L0.W + 7) / 8) * ((L0.H + 7) / 8);
        const uint32_t *order = L0.tile_buf, TA = order[T];
        for (uint32_t w = blockIdx.x; w < tile_waves_of(TA); w += gridDim.x) {
            const uint32_t i = xcd_tile(w);
            if (i >= TA) continue;
            finish_tile<INSTR, LIST>(L0, order[i], lst, cn);
            any = true;
        }
    }
    if (any) flush_counts(L0.counters, cn);
}

// The finish of a small image: four lanes per hit, so the bisection takes four
// rounds instead of seven (ten samples), the six central differences two, and a tile's hits
// are spread over four waves.  It does more work in all (ten samples for
// seven, the FP64 sample by one lane of four), so it gains where a hit's own
// serial chain bounds the launch and loses once the waves fill the chip:
// - a sparse frame (k_finish with a list otherwise): the line lies where an image
//   full of hits still gains.  96x64 lattice 87 -> 59 us;
//   256x192 (768 tiles) dam 131 -> 86, full lattice 94 -> 71; 288x224 (1008) dam
//   134 -> 85 but full lattice 96 -> 110, 360x360 (2025) 115 -> 195;
// - a dense frame, where one hit's walks take milliseconds: the chip's 4,096 waves
//   hold 65,536 hits of four lanes, and a quarter more still gains; in an uneven
//   frame (most: the fullest h/2 cell over the mean) up to four times as many do,
//   its longest hits outlasting the others.  March and finish, k_finish -> groups:
//     even, 3.3 per cell (most 3.3): 27,000 hits 923 -> 631 us, 64,000 966 -> 889,
//     99,000 1047 -> 1033, 134,000 1172 -> 1258, 570,000 2519 -> 3559; 9.8 per cell
//     (2.1): 64,000 2213 -> 2036, 81,000 2244 -> 2286, 134,000 2782 -> 3164;
//     clustered pools of 5.5 to 6.2 per cell, few hits and (near) many: most 5.9,
//     101,000 1371 -> 1097 and (112,000) 1060 -> 1125; 9.2, 134,000 1690 -> 1437 and
//     (149,000) 1255 -> 1329; 17, 192,000 4103 -> 2618 and (199,000) 1645 -> 1947.
//   (By the image's tiles alone, up to 16,384, groups took images full of hits too:
//   the 100,000-particle pool at 1280x800 4889 us, k_finish 2348.)
//   Without lists the LDS holds 16 waves a CU (sized for lists, ten: 176,000 hits of
//   the even frame 1748 us, now 1462).
//   The march has counted the hits by then, so both kernels are launched where
//   the tiles could hold more, and one of them ends at once.
static constexpr uint32_t kGroupTiles = 800, kGroupTilesDense = 16384, kGroupHits = 81920;

uint32_t group_hits(uint64_t n, uint32_t cells, uint32_t most)
{
    const double over = (double)most * (double)cells / (double)n / 8.0;
    return (uint32_t)(kGroupHits * (1.0 + fmin(over * over, 3.0)));
}

// FP32 density of one of a hit's samples from the hit's list, or by its own walk.
struct FinishDens {
    const GridDev *g;
    uint32_t *lst;
    int n;
    bool listed, comp, count;
    __device__ float operator()(float x, float y, float z, uint32_t &cand) const
    {
        uint32_t c = 0, nsup = 0;
        float rho;
        if (listed) {
            float sum = 0.0f, cc = 0.0f;
            pm_list_density(*g, lst, n, x, y, z, sum, cc, nsup);
            rho = comp ? sum + cc : sum;
            if (count) c = pm_stencil_cand(*g, x, y, z);
        } else {
            rho = pm_density32_list<kListCap>(*g, x, y, z, comp, lst, c);
        }
        if (count) cand += c;
        return rho;
    }
};

// upto: nothing is done for launches of more hits (k_finish takes them).
template <bool LIST>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_finish_groups(MarchLaunch L, uint32_t upto)
{
    if (upto != 0 && marched_hits(L) > upto) return;
    __shared__ uint32_t lds[LIST ? kFinWords : kListWords];
    const uint32_t lane = threadIdx.x;
    uint32_t *lst = lds + lane;
    const pm_settings &s = L.s;
    const GridDev &g = L.g;
    const uint32_t tiles_x = (L.W + 7) / 8, T = tiles_x * ((L.H + 7) / 8), sub = 2;
    const uint32_t *order = L.tile_buf, TA = order[T];
    constexpr int G = 4;
    const uint32_t gbase = lane & ~(uint32_t)(G - 1);
    const bool lead = lane == gbase, comp = s.compensated != 0, fp64 = s.final_fp64 && s.bisect_iters > 0;
    const float e = s.normal_mode == PM_NORMAL_CDIFF ? s.normal_eps : 0.0f;
    const float o[3] = { L.cam[0], L.cam[1], L.cam[2] };
    Counts cn;
    bool any = false;
    for (uint32_t w = blockIdx.x; w < tile_waves_of(TA << sub); w += gridDim.x) {
        const uint32_t i = xcd_tile(w);
        if (i >= TA << sub) continue;
        uint32_t px, py;
        part_pixel(order[i >> sub], tiles_x, i, sub, lane >> sub, px, py);
        const bool inside = px < L.W && py < L.H;
        const uint32_t idx = inside ? py * L.W + px : 0u;
        const uint4 rec = L.hit_rec[idx];
        const bool hit = inside && (rec.x & 1u), bracket = hit && (rec.x & 2u);
        if (__ballot(hit) == 0) continue;
        any = true;
        float lo = __uint_as_float(rec.y), hi = __uint_as_float(rec.z);
        float d[3];
        pm_ray_dir(L, px, py, d);
        FinishDens dens{ &g, lst, 0, false, comp, true };
        if (LIST && hit) dens.listed = pm_list_segment<kFinCap>(g, o, d, lo, hi, fabsf(e), lst, dens.n);
        if (__ballot(bracket) != 0) {
            float l = lo, h = hi;
            group_bisect(L, d, l, h, fp64 ? s.bisect_iters - 1 : s.bisect_iters, bracket, G, dens, cn);
            if (bracket) { lo = l; hi = h; }
            if (bracket && !fp64) lo = hi = (lo + hi) * 0.5f;
        }
        float th = lo, xs[3] = { o[0] + lo * d[0], o[1] + lo * d[1], o[2] + lo * d[2] };
        if (bracket && fp64 && lead) {
            double dlo = lo, dhi = hi;
            const double tm = (dlo + dhi) * 0.5;
            const double x = (double)o[0] + tm * (double)d[0], y = (double)o[1] + tm * (double)d[1],
                         z = (double)o[2] + tm * (double)d[2];
            const double rho = dens.listed ? pm_list_density64(g, lst, dens.n, x, y, z) : pm_density64(g, x, y, z);
            cn.samples++;
            if (rho >= (double)s.iso) dhi = tm; else dlo = tm;
            const double tt = (dlo + dhi) * 0.5;
            xs[0] = (float)((double)o[0] + tt * (double)d[0]);
            xs[1] = (float)((double)o[1] + tt * (double)d[1]);
            xs[2] = (float)((double)o[2] + tt * (double)d[2]);
            th = (float)tt;
        }
#pragma unroll
        for (int a = 0; a < 3; a++) xs[a] = __shfl(xs[a], (int)gbase, 64);   // the leader's point
        float nx = 0.f, ny = 0.f, nz = 0.f;
        if (s.normal_mode == PM_NORMAL_GRADW) {
            if (hit && lead) {
                float sx, sy, sz;
                uint32_t cand = 0;
                pm_sum_gradw(g, xs[0], xs[1], xs[2], sx, sy, sz, cand);
                pm_normalize(sx, sy, sz, nx, ny, nz);
            }
        } else {
            // counted as the six-sample walk's box, or where that leaves the grid sample by sample
            const uint32_t box = hit ? pm_box_cand(g, xs, e) : 0u;
            dens.count = box == 0xffffffffu;
            if (hit && lead && !dens.count) cn.cand += box;
            float gv[3];
            group_cdiff(xs, e, hit, G, dens, gv, cn);
            cdiff_normal(gv, nx, ny, nz);
        }
        if (hit && lead) {
            L.pos[idx] = make_float4(xs[0], xs[1], xs[2], 1.0f);
            L.nrm[idx] = make_float4(nx, ny, nz, 1.0f);
            if (L.t) L.t[idx] = th;
        }
    }
    if (any) flush_counters(L.counters, cn.rays, cn.in_aabb, cn.hits, cn.samples, cn.cand, cn.march);
}

static hipError_t launch_finish(const MarchLaunch &L0, hipStream_t st)
{
    const uint32_t T = ((L0.W + 7) / 8) * ((L0.H + 7) / 8);
    const uint32_t need = tile_waves_of(T);
    const dim3 grid(need < kMaxWaves ? need : kMaxWaves), blk(64);
    uint32_t upto = 0;
    if (T < (L0.g.sparse ? kGroupTiles : kGroupTilesDense) && !L0.s.instrument) {
        if (!L0.g.sparse && (uint64_t)T * 64 > L0.g.group_hits) upto = L0.g.group_hits;
        hipLaunchKernelGGL(L0.g.sparse ? k_finish_groups<true> : k_finish_groups<false>, dim3(tile_waves_of(T << 2)), blk, 0, st, L0, upto);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess || upto == 0) return e;
    }
    if (L0.s.instrument) hipLaunchKernelGGL((k_finish<false, true, true>), grid, blk, 0, st, L0, nullptr, nullptr, 0u, 0u);
    else if (L0.g.sparse) hipLaunchKernelGGL((k_finish<false, false, true>), grid, blk, 0, st, L0, nullptr, nullptr, 0u, 0u);
    else hipLaunchKernelGGL((k_finish<false, false, false>), grid, blk, 0, st, L0, nullptr, nullptr, 0u, upto);
    return hipGetLastError();
}

hipError_t launch_march_batch(const BatchLaunch &B, hipStream_t st)
{
    const uint32_t need = tile_waves_of(B.ntiles << (B.base.s.learned ? 0u : tile_split(B.ntiles)));
    const dim3 grid(need < kMaxWaves ? need : kMaxWaves), blk(64);
    if (need == 0) return hipSuccess;   // no tile to march
    if (B.base.s.learned) hipLaunchKernelGGL((k_march_batch<true>), grid, blk, 0, st, B);
    else hipLaunchKernelGGL((k_march_batch<false>), grid, blk, 0, st, B);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const uint32_t nf = tile_waves_of(B.ntiles);
    const dim3 fgrid(nf < kMaxWaves ? nf : kMaxWaves);
    if (B.sparse) hipLaunchKernelGGL((k_finish<true, false, true>), fgrid, blk, 0, st, B.base, B.jobs, B.tiles, B.ntiles, 0u);
    else hipLaunchKernelGGL((k_finish<true, false, false>), fgrid, blk, 0, st, B.base, B.jobs, B.tiles, B.ntiles, 0u);
    return hipGetLastError();
}

__global__ void k_zero_u64(unsigned long long *p, uint32_t n)
{
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0ull;
}

hipError_t launch_zero_u64(unsigned long long *p, uint32_t n, hipStream_t st)
{
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(128), 0, st, p, n);
    return hipGetLastError();
}

__global__ void k_init_counters(unsigned long long *p, uint32_t n, unsigned long long rays0)
{
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) p[i] = i == (uint32_t)C_RAYS ? rays0 : 0ull;   // slot 0 holds rays0
}

hipError_t launch_init_counters(unsigned long long *p, uint32_t n, unsigned long long rays0, hipStream_t st)
{
    hipLaunchKernelGGL(k_init_counters, dim3(1), dim3(64), 0, st, p, n, rays0);
    return hipGetLastError();
}

hipError_t launch_tile_flags(const MarchLaunch &L, uint32_t T, hipStream_t st)
{
    hipLaunchKernelGGL(k_tile_flags, dim3((T + 1 + 3) / 4), dim3(256), 0, st, L, T);
    return hipGetLastError();
}

hipError_t launch_miss_tiles(const MarchLaunch &L, uint32_t T, hipStream_t st)
{
    hipLaunchKernelGGL(k_miss_tiles, dim3((T + 3) / 4), dim3(256), 0, st, L, T);
    return hipGetLastError();
}

// The configured isotropic march of one view: schedule 1, or the tile
// pre-pass, the march and the finish of its tiles
// (L.tile_buf and L.hit_rec set).
hipError_t launch_tile_prepass(const MarchLaunch &L, hipStream_t st)
{
    const uint32_t tiles = ((L.W + 7) / 8) * ((L.H + 7) / 8);
    const uint32_t groups = (tiles + 63) / 64;
    hipLaunchKernelGGL(k_tile_masks, dim3(groups), dim3(1024), 0, st, L, tiles);
    const int summed = groups > kSumMasks;
    if (summed) hipLaunchKernelGGL(k_mask_sums, dim3((groups + 63) / 64), dim3(64), 0, st, L, tiles);
    hipLaunchKernelGGL(k_tile_list, dim3(groups), dim3(64), 0, st, L, tiles, summed);
    return hipGetLastError();
}

static hipError_t launch_march_config(const MarchLaunch &L, hipStream_t st)
{
    const uint32_t tiles = ((L.W + 7) / 8) * ((L.H + 7) / 8);
    if (L.s.schedule == 1 && !L.s.learned) {
        hipLaunchKernelGGL(k_march_simple, dim3((tiles + 3) / 4), dim3(256), 0, st, L);
        return hipGetLastError();
    }
    hipError_t e = launch_tile_prepass(L, st);
    if (e != hipSuccess) return e;
    // a wave per tile that may be active; beyond kMaxWaves each takes several
    const uint32_t need = tile_waves_of(tiles << kMaxSplit);
    const dim3 grid(need < kMaxWaves ? need : kMaxWaves), blk(64);
    const bool instr = L.s.instrument != 0;
    if (L.s.learned) {
        if (instr) hipLaunchKernelGGL((k_march_tiles<true, true>), grid, blk, 0, st, L);
        else hipLaunchKernelGGL((k_march_tiles<true, false>), grid, blk, 0, st, L);
    } else {
        if (instr) hipLaunchKernelGGL((k_march_tiles<false, true>), grid, blk, 0, st, L);
        else hipLaunchKernelGGL((k_march_tiles<false, false>), grid, blk, 0, st, L);
    }
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_finish(L, st);
}

hipError_t launch_march(const MarchLaunch &L, hipStream_t st)
{
    if (L.s.anisotropic) return launch_march_aniso(L, st);
    if (L.s.mode == PM_MODE_REFERENCE) {
        const uint32_t tiles = ((L.W + 7) / 8) * ((L.H + 7) / 8);
        if (L.tile_buf && L.s.schedule == 0) {
            hipError_t e = launch_tile_prepass(L, st);
            if (e != hipSuccess) return e;
            const uint32_t need = tile_waves_of(tiles << kMaxSplit);
            hipLaunchKernelGGL(k_ref_tiles, dim3(need < kMaxWaves ? need : kMaxWaves), dim3(64), 0, st, L);
            return hipGetLastError();
        }
        hipLaunchKernelGGL(k_march_reference, dim3((tiles + 3) / 4), dim3(256), 0, st, L);
        return hipGetLastError();
    }
    return launch_march_config(L, st);
}

// ---- point queries used by the parity tests ----

__global__ __launch_bounds__(256) void k_density(GridDev g, const float *__restrict__ q, uint32_t nq, int comp,
                                                 float *__restrict__ rho)
{
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nq) return;
    uint32_t cand = 0;
    rho[i] = pm_density32(g, q[3 * i], q[3 * i + 1], q[3 * i + 2], comp != 0, cand);
}

__global__ __launch_bounds__(256) void k_density64(GridDev g, const double *__restrict__ q, uint32_t nq,
                                                   double *__restrict__ rho)
{
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nq) return;
    rho[i] = pm_density64(g, q[3 * i], q[3 * i + 1], q[3 * i + 2]);
}

__global__ __launch_bounds__(256) void k_neighbor_counts(GridDev g, const float *__restrict__ q, uint32_t nq,
                                                         uint32_t *__restrict__ counts, uint32_t *__restrict__ ncand)
{
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nq) return;
    float qx = q[3 * i], qy = q[3 * i + 1], qz = q[3 * i + 2];
    int32_t cx, cy, cz;
    uint32_t cnt = 0, cand = 0;
    if (pm_stencil(g, qx, qy, qz, cx, cy, cz)) {
        for (int dz = -1; dz <= 1; dz++)
            for (int dy = -1; dy <= 1; dy++) {
                uint32_t base = (uint32_t)(cx - 1) + (uint32_t)g.nx * ((uint32_t)(cy + dy) + (uint32_t)g.ny * (uint32_t)(cz + dz));
                uint32_t b = g.cell_start[base], e = g.cell_start[base + 3];
                cand += e - b;
                for (uint32_t j = b; j < e; j++) {
                    float4 p = g.sorted[j];
                    float dx = qx - p.x, dy2 = qy - p.y, dz2 = qz - p.z;
                    float r2 = (dx * dx + dy2 * dy2) + dz2 * dz2;
                    if (r2 < g.h2) cnt++;
                }
            }
    }
    counts[i] = cnt;
    if (ncand) ncand[i] = cand;
}

hipError_t launch_density(const GridDev &g, const float *q, uint32_t nq, int compensated, float *rho, hipStream_t st)
{
    hipLaunchKernelGGL(k_density, dim3((nq + 255) / 256), dim3(256), 0, st, g, q, nq, compensated, rho);
    return hipGetLastError();
}

hipError_t launch_density64(const GridDev &g, const double *q, uint32_t nq, double *rho, hipStream_t st)
{
    hipLaunchKernelGGL(k_density64, dim3((nq + 255) / 256), dim3(256), 0, st, g, q, nq, rho);
    return hipGetLastError();
}

hipError_t launch_neighbor_counts(const GridDev &g, const float *q, uint32_t nq, uint32_t *counts, uint32_t *ncand,
                                  hipStream_t st)
{
    hipLaunchKernelGGL(k_neighbor_counts, dim3((nq + 255) / 256), dim3(256), 0, st, g, q, nq, counts, ncand);
    return hipGetLastError();
}

}  // namespace pm
