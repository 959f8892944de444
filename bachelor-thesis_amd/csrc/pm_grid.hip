// pm_grid.hip -- GPU uniform grid: the replacement of CompactNSearch's
// add_point_set / z_sort / sort_field / update_point_sets (Dataset.cpp:49-76)
// and of Frame::ComputeAABB (Dataset.cpp:78-92).
//
// Pipeline (one stream, no host round trip except the extent read-back):
//   bounds reduce -> histogram (atomics) -> exclusive scan -> indices placed
//   cell by cell -> per-cell sort by input index into cell-major float4.
// The per-cell sort makes the stored order deterministic (cell, input index),
// which is the canonical neighbour order the density sums follow.
// All passes are HBM-bound streaming passes over n particles or C cells.
#include "pm_internal.h"

#include <float.h>

namespace pm {

static constexpr int kThreads = 256;

uint32_t bounds_partials(uint64_t n)
{
    uint64_t b = (n + kThreads - 1) / kThreads;
    if (b > 1024) b = 1024;
    if (b < 1) b = 1;
    return (uint32_t)b;
}

// Minimum and maximum that keep a NaN, so one anywhere shows in the bounds (and
// the frame is refused: it has no cell).
__device__ __forceinline__ float bounds_min(float a, float b) { return b < a || b != b ? b : a; }
__device__ __forceinline__ float bounds_max(float a, float b) { return b > a || b != b ? b : a; }

__global__ __launch_bounds__(kThreads) void k_bounds_partial(const float *__restrict__ xyz, uint64_t n,
                                                             float *__restrict__ partial)
{
    float mn[3] = { FLT_MAX, FLT_MAX, FLT_MAX }, mx[3] = { -FLT_MAX, -FLT_MAX, -FLT_MAX };
    for (uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kThreads) {
        for (int a = 0; a < 3; a++) {
            float v = xyz[3 * i + a];
            mn[a] = bounds_min(mn[a], v);
            mx[a] = bounds_max(mx[a], v);
        }
    }
    __shared__ float red[6][kThreads];
    for (int a = 0; a < 3; a++) { red[a][threadIdx.x] = mn[a]; red[3 + a][threadIdx.x] = mx[a]; }
    __syncthreads();
    for (int s = kThreads / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            for (int a = 0; a < 3; a++) {
                red[a][threadIdx.x] = bounds_min(red[a][threadIdx.x], red[a][threadIdx.x + s]);
                red[3 + a][threadIdx.x] = bounds_max(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + s]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) partial[6 * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

__global__ __launch_bounds__(kThreads) void k_bounds_final(const float *__restrict__ partial, uint32_t np,
                                                           float *__restrict__ out)
{
    __shared__ float red[6][kThreads];
    float v[6] = { FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX };
    for (uint32_t i = threadIdx.x; i < np; i += kThreads)
        for (int a = 0; a < 3; a++) {
            v[a] = bounds_min(v[a], partial[6 * i + a]);
            v[3 + a] = bounds_max(v[3 + a], partial[6 * i + 3 + a]);
        }
    for (int a = 0; a < 6; a++) red[a][threadIdx.x] = v[a];
    __syncthreads();
    for (int s = kThreads / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int a = 0; a < 3; a++) {
                red[a][threadIdx.x] = bounds_min(red[a][threadIdx.x], red[a][threadIdx.x + s]);
                red[3 + a][threadIdx.x] = bounds_max(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) out[threadIdx.x] = red[threadIdx.x][0];
}

hipError_t launch_bounds_reduce(const float *xyz, uint64_t n, float *partial, uint32_t npartial, float *out,
                                hipStream_t st)
{
    hipLaunchKernelGGL(k_bounds_partial, dim3(npartial), dim3(kThreads), 0, st, xyz, n, partial);
    hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(kThreads), 0, st, partial, npartial, out);
    return hipGetLastError();
}

__global__ void k_fill_u32(uint32_t *__restrict__ p, uint64_t n, uint32_t v)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Both grids of a frame are built together from one histogram, the march grid's:
// a cell of h is 2x2x2 cells of h/2 (the keys are floor-like and 2/h is exact, so
// key(x, 1/h) = key(x, 2/h) >> 1, of negative coordinates too), so its count is
// the sum of eight and its particles are four runs of the march grid's order.
// The atomics bound the build (25 G/s): one per particle, which also gives the
// particle its place, where a histogram and a cursor for each grid took four.  Only the 4-byte index is placed; the particle
// itself is read by the ranking pass, which ranks it in both grids.  A launch's
// workgroups take contiguous runs of particles per XCD (xcd_run): neighbours in
// the input meet in the same cells, and their atomics and stores in one L2.
// 1.02 M particles: both sorts 250 us in 18 launches, now 105 in 7 (count 41, place
// 14, rank 28); the 4 M pool's, unevenly dense, 1,630 us, now 513 (rank 264).

// The blockIdx-th of `blocks` work items, contiguous runs for each of the 8 XCDs
// (workgroups are dispatched round-robin over them); >= blocks: none.
__device__ __forceinline__ uint64_t xcd_run(uint64_t blocks)
{
    const uint64_t per = (blocks + 7) / 8;
    return (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
}

// Cell of the march grid relative to its origin.
__device__ __forceinline__ void fine_cell(const GridBuildArgs &a, float x, float y, float z, int32_t k[3])
{
    k[0] = pm_key(x, a.inv_hf) - a.fo[0];
    k[1] = pm_key(y, a.inv_hf) - a.fo[1];
    k[2] = pm_key(z, a.inv_hf) - a.fo[2];
}

__device__ __forceinline__ uint32_t fine_lin(const GridBuildArgs &a, int32_t x, int32_t y, int32_t z)
{
    return (uint32_t)x + (uint32_t)a.fn[0] * ((uint32_t)y + (uint32_t)a.fn[1] * (uint32_t)z);
}

__global__ __launch_bounds__(kThreads) void k_cell_count(GridBuildArgs a)
{
    const uint64_t i = xcd_run((a.n + kThreads - 1) / kThreads) * kThreads + threadIdx.x;
    if (i >= a.n) return;
    int32_t k[3];
    fine_cell(a, a.xyz[3 * i + 0], a.xyz[3 * i + 1], a.xyz[3 * i + 2], k);
    a.slot[i] = atomicAdd(&a.counts[fine_lin(a, k[0], k[1], k[2])], 1u);
}

// ---- exclusive scan of u32 (len up to 2^31), 1024 elements per block ----
static constexpr int kScanPer = 4;
static constexpr int kScanBlock = kThreads * kScanPer;

static inline uint32_t scan_blocks(uint32_t len) { return (len + kScanBlock - 1) / kScanBlock; }

// Per block of the scan its sum, and its number of nonzero elements (11 bits) with
// its largest element (21 bits, at most kScanMax).
static constexpr uint32_t kScanMax = (1u << 21) - 1u;
size_t scan_tmp_size(uint32_t ncells, uint32_t fncells)
{
    return 2 * ((size_t)scan_blocks(ncells + 1) + scan_blocks(fncells + 1));
}

// Exclusive scan of one value per thread: within waves by shuffles, then over the
// waves' sums (sh: one u32 per wave).
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *sh, uint32_t &total)
{
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    uint32_t incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(incl, off, 64);
        if ((int)lane >= off) incl += o;
    }
    __syncthreads();                               // sh may still be read from the last call
    if (lane == 63) sh[wave] = incl;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for (uint32_t w = 0; w < nw; w++) {
        const uint32_t s = sh[w];
        before += w < wave ? s : 0u;
        total += s;
    }
    return before + incl - v;
}

// Particles in cell c of the search grid: its eight march-grid cells.  Particles
// lie at least two cells inside the search grid; its border cells, whose march
// cells may lie outside the march grid, hold none.
__device__ __forceinline__ uint32_t dense_count(const GridBuildArgs &a, uint32_t c)
{
    const int32_t x = (int32_t)(c % (uint32_t)a.dn[0]), yz = (int32_t)(c / (uint32_t)a.dn[0]);
    const int32_t y = yz % a.dn[1], z = yz / a.dn[1];
    if (x < 2 || y < 2 || z < 2 || x > a.dn[0] - 3 || y > a.dn[1] - 3 || z > a.dn[2] - 3) return 0;
    const int32_t fx = 2 * (x + a.dorg[0]) - a.fo[0], fy = 2 * (y + a.dorg[1]) - a.fo[1], fz = 2 * (z + a.dorg[2]) - a.fo[2];
    uint32_t s = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const uint32_t row = fine_lin(a, fx, fy + (r & 1), fz + (r >> 1));
        s += a.counts[row] + a.counts[row + 1];
    }
    return s;
}

// Blocks 0 .. nb0 - 1 scan the search grid's counts, the others the march grid's.
__global__ __launch_bounds__(kThreads) void k_scan_blocks(GridBuildArgs a, uint32_t nb0)
{
    __shared__ uint32_t sh[kThreads / 64], occ, top;
    const bool fine = blockIdx.x >= nb0;
    const uint32_t ncells = fine ? a.fncells : a.ncells, blk = blockIdx.x - (fine ? nb0 : 0u);
    uint32_t *out = fine ? a.fcell_start : a.cell_start;
    const uint32_t base = blk * kScanBlock + threadIdx.x * kScanPer;
    uint32_t v[kScanPer], sum = 0, cells = 0, most = 0;
    for (int j = 0; j < kScanPer; j++) {
        v[j] = base + j >= ncells ? 0u : (fine ? a.counts[base + j] : dense_count(a, base + j));
        sum += v[j];
        cells += v[j] != 0;
        most = max(most, v[j]);
    }
    if (threadIdx.x == 0) occ = top = 0;
    uint32_t total;
    uint32_t ex = block_excl_scan(sum, sh, total);
    for (int j = 0; j < kScanPer; j++) {
        if (base + j <= ncells) out[base + j] = ex;
        ex += v[j];
    }
    for (int off = 32; off > 0; off >>= 1) {
        cells += __shfl_xor(cells, off, 64);
        most = max(most, (uint32_t)__shfl_xor(most, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&occ, cells);
        atomicMax(&top, min(most, kScanMax));
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        a.scan_tmp[2 * blockIdx.x] = total;
        a.scan_tmp[2 * blockIdx.x + 1] = occ | top << 11;
    }
}

// One workgroup per grid: its blocks' sums in place, its occupied cells and the
// largest count of one.
__global__ __launch_bounds__(1024) void k_scan_sums(GridBuildArgs a, uint32_t nb0, uint32_t nb1)
{
    __shared__ uint32_t sh[16], occ, top;
    const uint32_t first = blockIdx.x ? nb0 : 0u, nb = blockIdx.x ? nb1 : nb0;
    uint32_t carry = 0, cells = 0, most = 0;
    if (threadIdx.x == 0) occ = top = 0;
    for (uint32_t base = 0; base < nb; base += 1024) {
        const uint32_t i = base + threadIdx.x;
        uint2 *p = (uint2 *)a.scan_tmp + first + i;
        const uint2 v = i < nb ? *p : make_uint2(0u, 0u);
        cells += v.y & 2047u;
        most = max(most, v.y >> 11);
        uint32_t total;
        const uint32_t ex = block_excl_scan(v.x, sh, total);
        if (i < nb) p->x = ex + carry;
        carry += total;
    }
    for (int off = 32; off > 0; off >>= 1) {
        cells += __shfl_xor(cells, off, 64);
        most = max(most, (uint32_t)__shfl_xor(most, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&occ, cells);
        atomicMax(&top, most);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        a.occupied[2 * blockIdx.x] = occ;
        a.occupied[2 * blockIdx.x + 1] = top;
    }
}

__global__ __launch_bounds__(kThreads) void k_scan_add(GridBuildArgs a, uint32_t nb0)
{
    const bool fine = blockIdx.x >= nb0;
    const uint32_t ncells = fine ? a.fncells : a.ncells, blk = blockIdx.x - (fine ? nb0 : 0u);
    uint32_t *out = fine ? a.fcell_start : a.cell_start;
    const uint32_t base = blk * kScanBlock + threadIdx.x * kScanPer;
    const uint32_t add = a.scan_tmp[2 * blockIdx.x];
    for (int j = 0; j < kScanPer; j++)
        if (base + j <= ncells) out[base + j] += add;
}

// The particles' indices in the march grid's order, arbitrary inside a cell.
__global__ __launch_bounds__(kThreads) void k_place(GridBuildArgs a)
{
    const uint64_t i = xcd_run((a.n + kThreads - 1) / kThreads) * kThreads + threadIdx.x;
    if (i >= a.n) return;
    int32_t k[3];
    fine_cell(a, a.xyz[3 * i + 0], a.xyz[3 * i + 1], a.xyz[3 * i + 2], k);
    a.index[a.fcell_start[fine_lin(a, k[0], k[1], k[2])] + a.slot[i]] = (uint32_t)i;
}

// Order inside each cell by input index: a particle goes to its cell's start +
// (number of particles of the cell with a smaller index), in both grids.  One
// thread per particle, read-only over its own cells: no dependent swaps and no
// atomics, so dense cells cost O(k) per particle in parallel rather than an
// O(k^2) serial insertion sort.
__global__ __launch_bounds__(kThreads) void k_cell_rank(GridBuildArgs a)
{
    const uint64_t s = xcd_run((a.n + kThreads - 1) / kThreads) * kThreads + threadIdx.x;
    if (s >= a.n) return;
    const uint32_t key = a.index[s];
    const float x = a.xyz[3 * (uint64_t)key], y = a.xyz[3 * (uint64_t)key + 1], z = a.xyz[3 * (uint64_t)key + 2];
    int32_t k[3];
    fine_cell(a, x, y, z, k);
    // search-grid cell, and its first march-grid cell
    const int32_t d[3] = { (k[0] + a.fo[0]) >> 1, (k[1] + a.fo[1]) >> 1, (k[2] + a.fo[2]) >> 1 };
    const int32_t f[3] = { 2 * d[0] - a.fo[0], 2 * d[1] - a.fo[1], 2 * d[2] - a.fo[2] };
    const uint32_t own = fine_lin(a, k[0], k[1], k[2]);
    uint32_t rank = 0, frank = 0, own_b = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const uint32_t row = fine_lin(a, f[0], f[1] + (r & 1), f[2] + (r >> 1));
        const uint32_t b = a.fcell_start[row], m = a.fcell_start[row + 1], e = a.fcell_start[row + 2];
        uint32_t lo = 0, hi = 0;
        for (uint32_t j = b; j < m; j++) lo += a.index[j] < key ? 1u : 0u;
        for (uint32_t j = m; j < e; j++) hi += a.index[j] < key ? 1u : 0u;
        rank += lo + hi;
        if (row == own) { frank = lo; own_b = b; }
        if (row + 1 == own) { frank = hi; own_b = m; }
    }
    const uint32_t c = (uint32_t)(d[0] - a.dorg[0]) +
                       (uint32_t)a.dn[0] * ((uint32_t)(d[1] - a.dorg[1]) + (uint32_t)a.dn[1] * (uint32_t)(d[2] - a.dorg[2]));
    const float4 v = make_float4(x, y, z, __uint_as_float(key));
    a.fsorted[own_b + frank] = v;
    a.sorted[a.cell_start[c] + rank] = v;
}

hipError_t launch_grid_build(const GridBuildArgs &a, hipStream_t st)
{
    const uint32_t fill = (a.fncells + kThreads - 1) / kThreads;
    hipLaunchKernelGGL(k_fill_u32, dim3(fill < 65535 ? fill : 65535), dim3(kThreads), 0, st, a.counts,
                       (uint64_t)a.fncells, 0u);
    const uint32_t pblocks = 8 * (uint32_t)(((a.n + kThreads - 1) / kThreads + 7) / 8);
    hipLaunchKernelGGL(k_cell_count, dim3(pblocks), dim3(kThreads), 0, st, a);
    const uint32_t nb0 = scan_blocks(a.ncells + 1), nb1 = scan_blocks(a.fncells + 1);
    hipLaunchKernelGGL(k_scan_blocks, dim3(nb0 + nb1), dim3(kThreads), 0, st, a, nb0);
    hipLaunchKernelGGL(k_scan_sums, dim3(2), dim3(1024), 0, st, a, nb0, nb1);
    hipLaunchKernelGGL(k_scan_add, dim3(nb0 + nb1), dim3(kThreads), 0, st, a, nb0);
    hipLaunchKernelGGL(k_place, dim3(pblocks), dim3(kThreads), 0, st, a);
    hipLaunchKernelGGL(k_cell_rank, dim3(pblocks), dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

// empty27[c] = 1 when cells c-1..c+1 on every axis hold no particle (border
// cells count missing neighbours as empty).
__global__ __launch_bounds__(kThreads) void k_empty27(const uint32_t *__restrict__ cs, int32_t nx, int32_t ny, int32_t nz,
                                                      uint8_t *__restrict__ out)
{
    uint32_t c = blockIdx.x * kThreads + threadIdx.x;
    if (c >= (uint32_t)nx * ny * nz) return;
    int32_t x = c % nx, y = (c / nx) % ny, z = c / (nx * ny);
    int32_t x0 = x > 0 ? x - 1 : 0, x1 = x < nx - 1 ? x + 1 : nx - 1;
    uint32_t cnt = 0;
    for (int dz = -1; dz <= 1; dz++)
        for (int dy = -1; dy <= 1; dy++) {
            int32_t yy = y + dy, zz = z + dz;
            if (yy < 0 || yy >= ny || zz < 0 || zz >= nz) continue;
            uint32_t row = (uint32_t)nx * ((uint32_t)yy + (uint32_t)ny * (uint32_t)zz);
            cnt += cs[row + x1 + 1] - cs[row + x0];
        }
    out[c] = cnt == 0;
}

hipError_t launch_empty27(const uint32_t *cs, int32_t nx, int32_t ny, int32_t nz, uint8_t *out, hipStream_t st)
{
    uint32_t n = (uint32_t)nx * ny * nz;
    hipLaunchKernelGGL(k_empty27, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, st, cs, nx, ny, nz, out);
    return hipGetLastError();
}

// Distance field of empty27: clear[c] is the Chebyshev distance, in cells, from
// c to the nearest cell whose 27-neighbourhood holds a particle, at most
// kClearMax (cells outside the grid hold none).  A ray inside a cell with
// clear = D > 0 may cross the (2 D - 1)^3 cells around it at once.  The
// Chebyshev distance is separable: along x, then min over d of max(|d|, .) along
// y and along z.  A pass loads at most 2 kClearMax - 1 bytes per cell, fewer where
// a particle is near; mostly empty grids, which load them all, bound it.  (y and
// z in one pass over the 15 x 15 rows around a cell took up to 224 loads: a grid of
// 64 M nearly empty cells 7.5 ms, now 1.3.)
static constexpr int kClearMax = 8;

__global__ __launch_bounds__(kThreads) void k_clear_x(const uint8_t *__restrict__ empty27, int32_t nx, uint32_t n,
                                                      uint8_t *__restrict__ out)
{
    const uint32_t c = blockIdx.x * kThreads + threadIdx.x;
    if (c >= n) return;
    const int32_t x = (int32_t)(c % (uint32_t)nx);
    int D = 0;
    for (; D < kClearMax; D++) {
        const bool lo = x - D >= 0 && !empty27[c - (uint32_t)D], hi = x + D < nx && !empty27[c + (uint32_t)D];
        if (lo || hi) break;
    }
    out[c] = (uint8_t)D;
}

// Along the axis of `len` cells `stride` apart.
__global__ __launch_bounds__(kThreads) void k_clear_axis(const uint8_t *__restrict__ in, uint32_t stride, uint32_t len,
                                                         uint32_t n, uint8_t *__restrict__ out)
{
    const uint32_t c = blockIdx.x * kThreads + threadIdx.x;
    if (c >= n) return;
    const int32_t i = (int32_t)(c / stride % len);
    int D = in[c];
    for (int r = 1; r < D; r++) {                  // none at distance >= D matters
        const int lo = i - r >= 0 ? in[c - (uint32_t)r * stride] : kClearMax;
        const int hi = i + r < (int32_t)len ? in[c + (uint32_t)r * stride] : kClearMax;
        D = min(D, max(r, min(lo, hi)));
    }
    out[c] = (uint8_t)D;
}

hipError_t launch_clear(const uint8_t *empty27, int32_t nx, int32_t ny, int32_t nz, uint8_t *tmp, uint8_t *out,
                        hipStream_t st)
{
    const uint32_t n = (uint32_t)nx * ny * nz;
    const dim3 grid((n + kThreads - 1) / kThreads), blk(kThreads);
    hipLaunchKernelGGL(k_clear_x, grid, blk, 0, st, empty27, nx, n, out);
    hipLaunchKernelGGL(k_clear_axis, grid, blk, 0, st, (const uint8_t *)out, (uint32_t)nx, (uint32_t)ny, n, tmp);
    hipLaunchKernelGGL(k_clear_axis, grid, blk, 0, st, (const uint8_t *)tmp, (uint32_t)nx * (uint32_t)ny, (uint32_t)nz, n, out);
    return hipGetLastError();
}

// Density bound per sub-box.  Every cell of the dense grid is split into
// 8x8x8 sub-boxes (eighth boxes); sub-box (fx, fy, fz) holds the points whose
// u = inv_h * x lies in [key + f/8, key + (f+1)/8) on every axis, and quarter
// box s = f / 2 (4x4x4 per cell) the eight sub-boxes with the same s.  For a
// box B widened by delta (which covers the rounding of u and of the march's
// sample positions), U = sum over the cell's 27-cell stencil of W(dist(x_j, B))
// bounds the density at every point of B, since W falls with r and the
// stencil holds every particle within h.  A sub-box's bit is set when U of its
// quarter box, or else its own U, is below the limit iso (1 - 2^-9); the margin
// covers the rounding of both sums.  Two rules spare sub-box sums that would
// find no bit: a cell whose centre row (dz = dy = 0) alone takes every quarter
// box's U past the limit lies inside the fluid and gets no bit, and neither
// does a quarter box whose U reaches 4 x the limit (a clear bit only means the
// sample is evaluated) -- except for the zero-density bound (iso = PM_ZERO_ISO),
// where a quarter box's U only says that some particle lies within h of it,
// not near which of its sub-boxes.  A cell's 512 bits are 64 bytes: byte
// l = sx + 4 sy + 16 sz belongs to quarter box s and its bit
// (fx & 1) + 2 (fy & 1) + 4 (fz & 1) to the sub-box inside it, so a byte of
// 0xff marks a quarter box the march can cross in one jump.  Each U sums the
// centre row (dz = dy = 0) first, then the other eight in (dz, dy) order,
// particles in storage order.  Border cells (no stencil, zero density) and
// cells with an empty 27-neighbourhood get every bit.  One wave per cell: lane
// l takes quarter box l, all lanes read the same particle; the quarter boxes'
// sums come first (one W per particle), the eight sub-box sums only for the
// quarter boxes between the limit and 4 x the limit, and each walk stops once
// every box it sums has reached the value that decides it.
// Squared distance along one axis from x to [lo, hi] (0 inside).
__device__ __forceinline__ float bound_e2(float lo, float hi, float x)
{
    const float e = fmaxf(fmaxf(lo - x, x - hi), 0.0f);
    return e * e;
}

// W at the distance from particle p to the box [l, h] (0 outside the support).
__device__ __forceinline__ float bound_term(const GridDev &g, float4 p, float lx, float hx, float ly, float hy, float lz,
                                            float hz)
{
    const float d2 = (bound_e2(lx, hx, p.x) + bound_e2(ly, hy, p.y)) + bound_e2(lz, hz, p.z);
    return d2 < g.h2 ? pm_W_sel(d2, g.inv_h, g.sig) : 0.0f;
}

// The eight sub-box bounds of one quarter box, one particle at a time.
struct BoundEighths {
    float lo[3][2], hi[3][2];   // per axis, the two sub-boxes' widened ends
    float U[8];

    __device__ void init(const GridDev &g, const int32_t k[3], const int32_t s[3], float delta)
    {
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int b = 0; b < 2; b++) {
                lo[a][b] = ((float)k[a] + 0.125f * (float)(2 * s[a] + b)) * g.h - delta;
                hi[a][b] = ((float)k[a] + 0.125f * (float)(2 * s[a] + b + 1)) * g.h + delta;
            }
#pragma unroll
        for (int f = 0; f < 8; f++) U[f] = 0.0f;
    }
    __device__ void add(const GridDev &g, float4 p)
    {
        const float ex0 = bound_e2(lo[0][0], hi[0][0], p.x), ex1 = bound_e2(lo[0][1], hi[0][1], p.x);
        const float ey0 = bound_e2(lo[1][0], hi[1][0], p.y), ey1 = bound_e2(lo[1][1], hi[1][1], p.y);
        const float ez0 = bound_e2(lo[2][0], hi[2][0], p.z), ez1 = bound_e2(lo[2][1], hi[2][1], p.z);
        // no sub-box within h: all eight terms are 0
        if (!((fminf(ex0, ex1) + fminf(ey0, ey1)) + fminf(ez0, ez1) < g.h2)) return;
#pragma unroll
        for (int f = 0; f < 8; f++) {
            const float d2 = ((f & 1 ? ex1 : ex0) + (f & 2 ? ey1 : ey0)) + (f & 4 ? ez1 : ez0);
            U[f] += d2 < g.h2 ? pm_W_sel(d2, g.inv_h, g.sig) : 0.0f;
        }
    }
    __device__ bool below(float lim) const
    {
        bool b = false;
#pragma unroll
        for (int f = 0; f < 8; f++) b = b || U[f] < lim;
        return b;
    }
};

// Row r of the bound walk's order: the centre row, then (dz, dy) in order.
__device__ __forceinline__ uint32_t bound_row(const GridDev &g, int32_t x, int32_t y, int32_t z, int r)
{
    const int dz = r == 0 ? 0 : (r - 1 + (r > 4)) / 3 - 1, dy = r == 0 ? 0 : (r - 1 + (r > 4)) % 3 - 1;
    return (uint32_t)x - 1u + (uint32_t)g.nx * ((uint32_t)(y + dy) + (uint32_t)g.ny * (uint32_t)(z + dz));
}

// The byte of quarter box `lane` of cell c (one wave; each lane stores its own).
// quarter_only: every byte 0xff or 0 (the quarter boxes' bounds alone).
__device__ __forceinline__ uint32_t bound_cell(const GridDev &g, float iso, bool quarter_only, uint32_t c, uint32_t lane)
{
    const uint32_t nx = (uint32_t)g.nx, ny = (uint32_t)g.ny;
    const int32_t x = (int32_t)(c % nx), y = (int32_t)((c / nx) % ny), z = (int32_t)(c / (nx * ny));
    if (x < 1 || y < 1 || z < 1 || x > g.nx - 2 || y > g.ny - 2 || z > g.nz - 2 || g.empty27[c]) return 0xffu;
    const int32_t k[3] = { x + g.ox, y + g.oy, z + g.oz };
    int32_t km = abs(k[0]) > abs(k[1]) ? abs(k[0]) : abs(k[1]);
    km = (km > abs(k[2]) ? km : abs(k[2])) + 1;
    const float delta = g.h * (0x1p-10f + (float)km * 0x1p-18f);
    const int32_t sq[3] = { (int32_t)(lane & 3u), (int32_t)((lane >> 2) & 3u), (int32_t)(lane >> 4) };
    const float lim = iso * (1.0f - 0x1p-9f), lim4 = iso == PM_ZERO_ISO ? INFINITY : 4.0f * lim;
    // the quarter box's bound; inside the fluid the centre row alone takes
    // every quarter box past the limit
    const float lx = ((float)k[0] + 0.25f * (float)sq[0]) * g.h - delta, hx = ((float)k[0] + 0.25f * (float)(sq[0] + 1)) * g.h + delta;
    const float ly = ((float)k[1] + 0.25f * (float)sq[1]) * g.h - delta, hy = ((float)k[1] + 0.25f * (float)(sq[1] + 1)) * g.h + delta;
    const float lz = ((float)k[2] + 0.25f * (float)sq[2]) * g.h - delta, hz = ((float)k[2] + 0.25f * (float)(sq[2] + 1)) * g.h + delta;
    float Uq = 0.0f;
    for (int r = 0; r < 9; r++) {
        const uint32_t row = bound_row(g, x, y, z, r);
        const uint32_t b = g.cell_start[row], e = g.cell_start[row + 3];
        // all lanes take the same particles (scalar loads); 8 in flight
        uint32_t j = b;
        for (; j + 8 <= e; j += 8) {
            const float4 *src = g.sorted + j;
            float4 p[8];
#pragma unroll
            for (int u = 0; u < 8; u++) p[u] = src[u];
#pragma unroll
            for (int u = 0; u < 8; u++) Uq += bound_term(g, p[u], lx, hx, ly, hy, lz, hz);
            if (r == 0 && __ballot(Uq < lim) == 0) return 0u;   // inside the fluid
        }
        for (; j < e; j++) Uq += bound_term(g, g.sorted[j], lx, hx, ly, hy, lz, hz);
        if (r == 0 && __ballot(Uq < lim) == 0) return 0u;       // inside the fluid
        if (__ballot(Uq < (quarter_only ? lim : lim4)) == 0) break;
    }
    const bool whole = Uq < lim;
    if (quarter_only) return whole ? 0xffu : 0u;
    const bool eighths = !whole && Uq < lim4;
    if (__ballot(eighths) == 0) return whole ? 0xffu : 0u;
    // the eight sub-boxes of the quarter boxes left at or above the limit
    BoundEighths B;
    B.init(g, k, sq, delta);
    for (int r = 0; r < 9; r++) {
        if (eighths) {
            const uint32_t row = bound_row(g, x, y, z, r);
            const uint32_t b = g.cell_start[row], e = g.cell_start[row + 3];
            uint32_t j = b;
            for (; j + 4 <= e; j += 4) {
                const float4 *src = g.sorted + j;
                float4 p[4];
#pragma unroll
                for (int u = 0; u < 4; u++) p[u] = src[u];
#pragma unroll
                for (int u = 0; u < 4; u++) B.add(g, p[u]);
            }
            for (; j < e; j++) B.add(g, g.sorted[j]);
        }
        if (__ballot(eighths && B.below(lim)) == 0) break;
    }
    if (whole) return 0xffu;
    if (!eighths) return 0u;
    uint32_t m = 0;
#pragma unroll
    for (int f = 0; f < 8; f++) m |= (B.U[f] < lim ? 1u : 0u) << f;
    return m;
}

// One wave per cell; bits[64 c + l] is the byte of quarter box l.  The weights'
// VALU instructions bound it: the cell is a scalar, so the particles come through scalar loads without an address in a
// VGPR, the weight takes no branch, and the centre row ends once it has decided.
// Quarter boxes of the 1.02 M dam break 410 -> 366 us, every sub-box of the 4 M
// pool 3.42 -> 3.15 ms.  Slower: one row in one vector load handed round by
// readlane, and sums of a cheaper form of the spline that leave only values near
// a limit to this one (no branch past particles out of reach: 477 us).
__global__ __launch_bounds__(256) void k_bound_grid(GridDev g, float iso, int quarter_only, uint8_t *__restrict__ out)
{
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t c = blockIdx.x * 4 + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (c >= (uint32_t)g.nx * (uint32_t)g.ny * (uint32_t)g.nz) return;   // whole wave
    out[64 * (uint64_t)c + lane] = (uint8_t)bound_cell(g, iso, quarter_only != 0, c, lane);
}

hipError_t launch_bound_grid(const GridDev &g, float iso, bool quarter_only, uint64_t *out, hipStream_t st)
{
    uint32_t n = (uint32_t)g.nx * g.ny * g.nz;
    hipLaunchKernelGGL(k_bound_grid, dim3((n + 3) / 4), dim3(256), 0, st, g, iso, quarter_only ? 1 : 0, (uint8_t *)out);
    return hipGetLastError();
}

// Reference DensityGrid node flags (Dataset.cpp:94-164).  Node (x,y,z) covers
// [bmin + (x,y,z) h, +h); its centre is bmin + ((x,y,z) + 0.5) h.  Two flags:
//   box  : some particle with |x_j - centre|_inf < h and count * W(0) > 1
//          (one reading of find_neighbors_box, whose source is absent);
//   cons : some particle with |x_j - centre|_inf < 1.5 h (1.001 margin), i.e.
//          a cleared node has zero density everywhere inside it.
__global__ __launch_bounds__(kThreads) void k_densitygrid(GridDev g, int32_t dnx, int32_t dny, int32_t dnz,
                                                          uint8_t *__restrict__ flag_box, uint8_t *__restrict__ flag_cons,
                                                          uint32_t *__restrict__ count_box)
{
    uint32_t id = blockIdx.x * kThreads + threadIdx.x;
    if (id >= (uint32_t)dnx * dny * dnz) return;
    int32_t k[3] = { (int32_t)(id % dnx), (int32_t)((id / dnx) % dny), (int32_t)(id / (dnx * dny)) };
    float c[3];
    const float cw = 1.0f * g.h;
    for (int a = 0; a < 3; a++) c[a] = g.bmin[a] + ((float)k[a] + 0.5f) * cw;
    const int32_t org[3] = { g.ox, g.oy, g.oz }, dim[3] = { g.nx, g.ny, g.nz };
    uint32_t res[2] = { 0u, 0u };
    const float R[2] = { g.h, 1.5f * g.h * 1.001f };
    for (int w = 0; w < 2; w++) {
        int32_t lo[3], hi[3];
        bool empty = false;
        for (int a = 0; a < 3; a++) {
            lo[a] = pm_key(c[a] - R[w], g.inv_h) - org[a];
            hi[a] = pm_key(c[a] + R[w], g.inv_h) - org[a];
            if (lo[a] < 0) lo[a] = 0;
            if (hi[a] > dim[a] - 1) hi[a] = dim[a] - 1;
            if (lo[a] > hi[a]) empty = true;
        }
        if (empty) continue;
        uint32_t cnt = 0;
        for (int32_t z = lo[2]; z <= hi[2]; z++)
            for (int32_t y = lo[1]; y <= hi[1]; y++) {
                uint32_t row = (uint32_t)g.nx * ((uint32_t)y + (uint32_t)g.ny * (uint32_t)z);
                uint32_t b = g.cell_start[row + lo[0]], e = g.cell_start[row + hi[0] + 1];
                for (uint32_t i = b; i < e; i++) {
                    float4 p = g.sorted[i];
                    if (fabsf(p.x - c[0]) < R[w] && fabsf(p.y - c[1]) < R[w] && fabsf(p.z - c[2]) < R[w]) cnt++;
                }
            }
        res[w] = cnt;
    }
    count_box[id] = res[0];
    flag_box[id] = (float)res[0] * g.sig > 1.0f;
    flag_cons[id] = res[1] > 0;
}

hipError_t launch_densitygrid(const GridDev &g, int32_t dnx, int32_t dny, int32_t dnz, uint8_t *flag_box, uint8_t *flag_cons,
                              uint32_t *count_box, hipStream_t st)
{
    uint32_t n = (uint32_t)dnx * dny * dnz;
    hipLaunchKernelGGL(k_densitygrid, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, st, g, dnx, dny, dnz, flag_box,
                       flag_cons, count_box);
    return hipGetLastError();
}

// Streaming copy (read n float4, write n float4): the measured-bandwidth
// reference point for the roofline and for scaling HBM byte counters.
__global__ __launch_bounds__(kThreads) void k_stream_copy(const float4 *__restrict__ src, float4 *__restrict__ dst,
                                                          uint64_t n)
{
    for (uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kThreads)
        dst[i] = src[i];
}

hipError_t launch_stream_copy(const void *src, void *dst, uint64_t bytes, hipStream_t st)
{
    uint64_t n = bytes / 16;
    uint64_t blocks = (n + kThreads - 1) / kThreads;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_stream_copy, dim3((uint32_t)blocks), dim3(kThreads), 0, st, (const float4 *)src, (float4 *)dst, n);
    return hipGetLastError();
}

}  // namespace pm
