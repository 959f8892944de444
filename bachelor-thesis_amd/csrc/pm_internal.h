// pm_internal.h -- host-side launchers shared by the kernels and the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pm_device.h"
#include "pm_mlp.h"
#include "pmarch.h"

namespace pm {

// Per-launch counters (u64 each), accumulated by the march kernels, in the
// order of pm_stats.  C_BOX_HITS: the rays in the box and 2^32 times the hits, one
// atomic for both (a march of 800x600, a few samples per ray: 134 us, with an atomic
// for each 168; a slot's share of the largest batch, 2^33 rays, is 2^30).
enum Counter {
    C_RAYS = 0, C_BOX_HITS, C_SAMPLES, C_CAND, C_MARCH_SAMPLES, C_MLP, C_MARCH_CAND, C_CERT, C_CERT_SKIP,
    C_CAND_STENCIL, C_CAND27, C_COUNT
};
// The counters live in kCtrSlots copies, one per XCD (a workgroup adds to
// slot blockIdx % 8), kCtrStride u64 (one 128-byte line) apart: atomics of
// different XCDs never meet on one address.  The host sums the slots.
constexpr int kCtrSlots = 8, kCtrStride = 16, kCtrWords = kCtrSlots * kCtrStride;

// Coarse occupancy grid of the step-proposal features: 4x4x4 dense cells.
struct CoarseDev {
    const uint32_t *count;
    int32_t nx, ny, nz;
};

// Anisotropic density parameters (PerPixel_Anisotropic, RayMarcher.cpp:346-423):
// h = ParticleRadius, hx = ParticleRadiusExt, sig = 8/pi (Kernel.cpp:57-61),
// the clamp knobs k_n, k_r, k_s, N_eps (RayMarcher.h:22-25); FP32 and FP64.
struct AnParF {
    using T = float;
    float h, h2, hinv, hx, R2x, hxinv, sig, k_n, k_r, k_s;
    int32_t n_eps;
};
struct AnParD {
    using T = double;
    double h, h2, hinv, hx, R2x, hxinv, sig, k_n, k_r, k_s;
    int32_t n_eps;
};
struct AnisoDev {
    AnParF f;
    AnParD d;
};

struct MarchLaunch {
    GridDev g;
    pm_settings s;
    float M[16];
    float cam[3];
    uint32_t W, H;
    const float *depth;   // device, reference mode
    float4 *pos;
    float4 *nrm;
    float *t;             // may be null
    unsigned long long *counters;
    uint32_t *band_ctr;        // per-XCD tile counters and the hit-list length (anisotropic march, schedule 1)
    // learned step proposal
    CoarseDev cg;
    MlpDev net;
    float mlp_alpha;           // fraction of the predicted distance that is skipped
    int32_t mlp_min_skip;      // below this many steps the ray continues step by step
    int32_t mlp_max_skip;      // longest jump, in steps
    float mlp_gate_rho;        // a sample asks for a proposal only below this density
    // the active tiles of the tile pre-pass (tile_words(T) u32: the list, its
    // length at T, masks); null = every tile
    uint32_t *tile_buf;
    float inv_step;            // 1 / s.step (bound skip)
    // per pixel: the hit handed from the march to the finish (1 | bracket << 1,
    // lo, hi, 0), zeros for a miss; written for every pixel of a marched tile
    // (the anisotropic march's schedule 1: its list of hits)
    uint4 *hit_rec;
    AnisoDev an;               // s.anisotropic
};

// Batched launch: many (view, frame) jobs in one march and one finish; every job
// is a complete MarchLaunch in device memory (read through a wave-uniform
// pointer, so its fields stay in scalar registers and the scalar cache).
// An active 8x8 tile of one job.
struct BatchTile {
    uint32_t job, tile;
};
struct BatchLaunch {
    MarchLaunch base;          // settings, counters and network (each job repeats them)
    const MarchLaunch *jobs;
    const BatchTile *tiles;    // the active tiles of all jobs
    uint32_t ntiles;
    int sparse;                // every job's frame is (GridDev::sparse)
};
hipError_t launch_bound_grid(const GridDev &g, float iso, bool quarter_only, uint64_t *out, hipStream_t st);
hipError_t launch_march_batch(const BatchLaunch &B, hipStream_t st);
hipError_t launch_zero_u64(unsigned long long *p, uint32_t n, hipStream_t st);
// counters[0..n) = 0 except counters[C_RAYS] = rays0 (rays answered without marching)
hipError_t launch_init_counters(unsigned long long *p, uint32_t n, unsigned long long rays0, hipStream_t st);
// Tile pre-pass pieces: flags (tile_buf[t] = 1 if a ray of tile t enters the
// AABB, t < T; tile_buf[T] = 0) and the misses of the inactive tiles.
hipError_t launch_tile_flags(const MarchLaunch &L, uint32_t T, hipStream_t st);
hipError_t launch_miss_tiles(const MarchLaunch &L, uint32_t T, hipStream_t st);

// Grid build: bounds of n float3 points (device) into out[6] (device).
hipError_t launch_bounds_reduce(const float *xyz, uint64_t n, float *partial, uint32_t npartial,
                                float *out, hipStream_t st);
uint32_t bounds_partials(uint64_t n);

// The search grid (cells of h) and the march grid (cells of h/2) of a frame.
struct GridBuildArgs {
    const float *xyz;      // device AoS float3
    uint64_t n;
    float inv_hf;          // 2 / h
    int32_t fo[3], fn[3];  // march grid: origin, cells per axis
    int32_t dorg[3], dn[3];   // search grid
    uint32_t ncells, fncells;
    uint32_t *counts;      // fncells, zeroed by the build
    uint32_t *slot;        // n: place inside the march-grid cell, arbitrary order
    uint32_t *index;       // n: input indices, march cell by march cell
    float4 *sorted, *fsorted;             // n
    uint32_t *cell_start, *fcell_start;   // ncells + 1, fncells + 1
    uint32_t *scan_tmp;    // scan_tmp_size of both grids
    uint32_t *occupied;    // [4]: search cells that hold a particle, the most in one; march cells, the most in one
};
size_t scan_tmp_size(uint32_t ncells, uint32_t fncells);
hipError_t launch_grid_build(const GridBuildArgs &a, hipStream_t st);

// The tile pre-pass (L.tile_buf set): the list of the active tiles and the misses
// of the others.  Its words: the list, one 64-bit mask per 64 tiles, one sum per 64
// masks.
inline size_t tile_words(uint64_t T)
{
    const uint64_t masks = (T + 63) / 64;
    return (size_t)(((T + 2) & ~1ull) + 2 * masks + (masks + 63) / 64);
}
hipError_t launch_tile_prepass(const MarchLaunch &L, hipStream_t st);
hipError_t launch_march(const MarchLaunch &L, hipStream_t st);
// GridDev::group_hits of a frame of n particles in `cells` march cells, at most
// `most` in one.
uint32_t group_hits(uint64_t n, uint32_t cells, uint32_t most);
// The anisotropic march: march, finish and normals kernels over the active tiles,
// or the reference march of a tile; schedule 1: its own forms.
hipError_t launch_march_aniso(const MarchLaunch &L, hipStream_t st);
hipError_t launch_density_aniso(const GridDev &g, const AnParF &a, const float *q, uint32_t nq, int compensated,
                                float *rho, hipStream_t st);
hipError_t launch_density_aniso64(const GridDev &g, const AnParD &a, const double *q, uint32_t nq, double *rho,
                                  hipStream_t st);
hipError_t launch_aniso_matrix(const GridDev &g, const AnParF &a, const float *q, uint32_t nq, float *G, float *det,
                               uint32_t *next, hipStream_t st);
hipError_t launch_density(const GridDev &g, const float *q, uint32_t nq, int compensated, float *rho,
                          hipStream_t st);
hipError_t launch_density64(const GridDev &g, const double *q, uint32_t nq, double *rho, hipStream_t st);
hipError_t launch_neighbor_counts(const GridDev &g, const float *q, uint32_t nq, uint32_t *counts,
                                  uint32_t *ncand, hipStream_t st);

hipError_t launch_stream_copy(const void *src, void *dst, uint64_t bytes, hipStream_t st);
// Gaussian depth smoothing (GaussRenderPass): K = the (N + 1)^2 table of pm_gauss_kernel.
// The depth-sprite pass: View, Projection (column-major), the march's inverse
// projection-view and camera for the pixel rays, the particle radius and the
// particles' bounds.
struct SpriteLaunch {
    float view[16], proj[16], inv_pv[16], cam[3];
    float lo[3], hi[3];
    float radius;
    uint32_t W, H;
};
// tmax: one u32 per 8x8 pixel tile.
hipError_t launch_depth_sprites(const SpriteLaunch &S, const float4 *pts, uint32_t n, uint32_t *depth, uint32_t *tmax,
                                hipStream_t st);
hipError_t launch_depth_smooth(const float *in, float *out, uint32_t W, uint32_t H, int N, const float *K,
                               hipStream_t st);
hipError_t launch_empty27(const uint32_t *cs, int32_t nx, int32_t ny, int32_t nz, uint8_t *out, hipStream_t st);
// The distance field of empty27 (GridDev::clear); tmp: one byte per cell.
hipError_t launch_clear(const uint8_t *empty27, int32_t nx, int32_t ny, int32_t nz, uint8_t *tmp, uint8_t *out,
                        hipStream_t st);
hipError_t launch_densitygrid(const GridDev &g, int32_t dnx, int32_t dny, int32_t dnz, uint8_t *flag_box, uint8_t *flag_cons,
                              uint32_t *count_box, hipStream_t st);

hipError_t launch_coarse_counts(const GridDev &g, const CoarseDev &cg, uint32_t *out, hipStream_t st);

struct TraceArgs {
    GridDev g;
    CoarseDev cg;
    float M[16];
    float cam[3];
    uint32_t W, H;
    float step, iso;
    const float *t_hit;       // plain-march t per pixel (-1 = miss)
    uint32_t ray_stride, k_stride, seed;
    uint32_t *count;          // rows written so far (device)
    uint32_t cap;
    float *feat;              // [cap][24]
    float *label;             // [cap]
    uint8_t *is_hit;          // [cap]
    uint32_t *meta;           // [cap][2]: pixel index, sample index k
};
hipError_t launch_trace(const TraceArgs &a, hipStream_t st);

struct TrainArgs {
    MlpDev net;
    const float *feat;
    const float *label;
    const uint32_t *idx;      // batch sample ids (NULL: 0..B-1)
    float inv_batch, w_over;
    uint32_t ngroups;         // B / 64
    float *partial;           // [nblocks][NPARAM + 1]
};
static constexpr uint32_t kTrainBlocks = 512;   // most workgroups of k_mlp_train: two per CU fit its LDS
struct AdamArgs {
    const float *partial;
    uint32_t nparts;
    float *p, *m, *v;
    float lr, b1, b2, eps, bc1, bc2;
    int apply;
    float *grad_out;          // optional summed gradient
    float *loss_out;
};
hipError_t launch_mlp_train(const TrainArgs &a, uint32_t nblocks, hipStream_t st);
hipError_t launch_mlp_adam(const AdamArgs &a, hipStream_t st);
hipError_t launch_mlp_sync(const float *p, uint16_t *W1, uint16_t *W2, uint16_t *W2T, hipStream_t st);
hipError_t launch_mlp_forward(const MlpDev &net, const float *feat, uint32_t n, float *y, hipStream_t st);

// Scratch of pm_march_device_noalloc (pm_noalloc.hip): the static device
// array of the device (looked up once per device), and its layout for a W x H
// march (false beyond the limits).
struct NoAllocScratch {
    uint4 *hit_rec;
    uint32_t *tiles;
    unsigned long long *counters;
    uint32_t *band;
};
hipError_t noalloc_scratch_init(int device, void **out);
bool noalloc_layout(void *base, uint32_t W, uint32_t H, NoAllocScratch &s);
size_t noalloc_scratch_bytes();

// Host restatement of the CompactNSearch key, for the grid extent.
inline int32_t host_key(float x, float inv_h)
{
    float v = inv_h * x;
    return x >= 0.0f ? (int32_t)v : (int32_t)v - 1;
}

}  // namespace pm
