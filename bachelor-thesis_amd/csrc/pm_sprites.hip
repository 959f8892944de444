// pm_sprites.hip -- the depth-sprite pass that gives the reference march its
// ray starts: DepthRenderPass (DepthRenderPass.cpp:243-250 uniforms View,
// Projection, Radius), the sprite quads of AdvancedRenderer::CollectRenderData
// (AdvancedRenderer.cpp:455-474: p + R (+-x +-y) with x, y the first two rows
// of View, CameraController3D.cpp:80; UV (-1, -1) at p + R (-x + y)), depth.vert
// and depth.frag, depth test LESS against a clear of 1.0.
//
// Fragment at the centre of pixel (px, py), NDC ((px + 0.5) 2 / W - 1, ...):
// the pixel's ray from the camera meets the quad's plane at P; for a planar quad
// the perspective-correct interpolation of the vertices' view positions and
// UVs is View P and ((P - p).x / R, -(P - p).y / R).  depth.frag: discard when
// l2 = |UV|^2 > 1, else pView = View P - R (0, 0, cos(pi/2 sqrt(l2))) and the
// depth is (Projection pView).z / .w.  Fragments whose plane depth lies
// outside [0, 1] are clipped, written depths are clamped to [0, 1], and a
// particle with a quad corner behind the camera (w <= 0) is not drawn.  The
// minimum over all fragments of a pixel is kept (atomicMin on the bits of
// non-negative floats: the order of the particles does not matter), with an
// early depth test.
//
// At 1080p the dam break's 1M sprites put ~600 fragments on each drawn pixel,
// nearly all behind others.  Where that pays (kCullParticles), one particle of
// every kSampleStride, spread over the cloud, is drawn first; the largest depth of every 8x8 pixel tile of that
// image then bounds what a later sprite can still change, and a sprite whose
// nearest possible depth is not below it in any tile of its footprint is left
// out (sp_near).  The image is the same minimum.  1080p dam break: 952 us (one
// thread per sprite, 221 M pixel tests, the image's coherent traffic) -> 84 us
// for the sample + 6 for the tiles + 168 for the rest (16 M tests).  A sample of
// every 8th or 32nd particle: 269 and 300 us; a second sample in between
// (64, 8): 330 us.
// cos(pi/2 s) is the Taylor polynomial through s^12 (error < 7e-9 on [0, 1]).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "pm_internal.h"

namespace pm {

// glm mat4 * vec4 (x, y, z, 1), column-major M: (m0 x + m1 y) + (m2 z + m3).
__device__ __forceinline__ void sp_xform(const float *M, float x, float y, float z, float o[4])
{
#pragma unroll
    for (int r = 0; r < 4; r++) o[r] = (M[r] * x + M[4 + r] * y) + (M[8 + r] * z + M[12 + r] * 1.0f);
}

__device__ __forceinline__ float sp_cos_half_pi(float s)
{
    const float t = 1.57079632679f * s, z = t * t;
    float c = 1.0f / 479001600.0f;
    c = c * z + -1.0f / 3628800.0f;
    c = c * z + 1.0f / 40320.0f;
    c = c * z + -1.0f / 720.0f;
    c = c * z + 1.0f / 24.0f;
    c = c * z + -0.5f;
    return c * z + 1.0f;
}

// A sprite's screen footprint and the plane of its quad.
struct SpriteBox {
    int x0, x1, y0, y1;          // pixel range, clamped to the image; empty when x0 > x1 or y0 > y1
    float ax, ay, az, bx, by, bz;  // rows 0 and 1 of View: the quad's x and y
    float pn;                    // (p - eye) . (x cross y)
    float nx, ny, nz;            // x cross y
};

// A lower bound of the depth of every fragment of the sprite at q.  With an
// orthonormal View and a projection whose depth grows with view z alone
// (S.cull, sp_cull), the quad lies in the plane of its centre's view z and a
// fragment moves at most R towards the eye; the margins cover the rounding of
// the fragments' points (relative to all coordinates that enter) and of their
// depths (values up to 1).
__device__ __forceinline__ float sp_near(const SpriteLaunch &S, const float4 q)
{
    const float *V = S.view, *P = S.proj;
    const float zc = (V[2] * q.x + V[6] * q.y) + (V[10] * q.z + V[14]);
    const float all = ((fabsf(q.x) + fabsf(q.y)) + (fabsf(q.z) + fabsf(V[14]))) +
                      ((fabsf(S.cam[0]) + fabsf(S.cam[1])) + (fabsf(S.cam[2]) + fabsf(zc)));
    const float z = zc - 1.001f * S.radius - 1e-5f * (all + S.radius);
    const float w = P[11] * z + P[15];
    return w > 0.0f ? (P[10] * z + P[14]) / w - 1e-6f : -1.0f;
}

// The tiles of the footprint in which some pixel may still be lowered by a depth
// of at least zn, as bits in row order: tmax holds the largest depth of each 8x8
// tile at some time before (null: all tiles).  The footprint covers at most 32
// tiles.
__device__ __forceinline__ uint32_t sp_open(const SpriteBox &B, float zn, const uint32_t *__restrict__ tmax, uint32_t tiles_x)
{
    const uint32_t tx0 = (uint32_t)B.x0 >> 3, ty0 = (uint32_t)B.y0 >> 3;
    const uint32_t tw = ((uint32_t)B.x1 >> 3) - tx0 + 1, th = ((uint32_t)B.y1 >> 3) - ty0 + 1;
    uint32_t open = 0, bit = 0;
    for (uint32_t ty = 0; ty < th; ty++)
        for (uint32_t tx = 0; tx < tw; tx++, bit++)
            if (!tmax || zn < __uint_as_float(tmax[(ty0 + ty) * tiles_x + tx0 + tx])) open |= 1u << bit;
    return open;
}

// The axes and the normal of every quad.
__device__ __forceinline__ void sp_plane(const SpriteLaunch &S, SpriteBox &B)
{
    const float *V = S.view;
    B.ax = V[0]; B.ay = V[4]; B.az = V[8];      // row 0 of View: the quad's x
    B.bx = V[1]; B.by = V[5]; B.bz = V[9];      // row 1: its y
    // plane of the quad: normal x cross y
    B.nx = B.ay * B.bz - B.az * B.by; B.ny = B.az * B.bx - B.ax * B.bz; B.nz = B.ax * B.by - B.ay * B.bx;
}

// False when the particle draws nothing (a quad corner behind the eye, or a
// footprint outside the image).
__device__ __forceinline__ bool sp_box(const SpriteLaunch &S, const float4 q, SpriteBox &B)
{
    const float R = S.radius;
    const float *V = S.view, *P = S.proj;
    sp_plane(S, B);
    float lo_x = 3.0e38f, hi_x = -3.0e38f, lo_y = 3.0e38f, hi_y = -3.0e38f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const float sx = (k & 1) ? 1.0f : -1.0f, sy = (k & 2) ? 1.0f : -1.0f;
        const float cx = q.x + R * (sx * B.ax + sy * B.bx), cy = q.y + R * (sx * B.ay + sy * B.by),
                    cz = q.z + R * (sx * B.az + sy * B.bz);
        float v[4], c[4];
        sp_xform(V, cx, cy, cz, v);
        sp_xform(P, v[0], v[1], v[2], c);
        if (!(c[3] > 0.0f)) return false;
        const float fx = (c[0] / c[3] + 1.0f) * 0.5f * (float)S.W, fy = (c[1] / c[3] + 1.0f) * 0.5f * (float)S.H;
        lo_x = fminf(lo_x, fx); hi_x = fmaxf(hi_x, fx);
        lo_y = fminf(lo_y, fy); hi_y = fmaxf(hi_y, fy);
    }
    // pixel centres px + 0.5 inside [lo, hi], clamped to the image
    const float x0f = fmaxf(ceilf(lo_x - 0.5f), 0.0f), x1f = fminf(floorf(hi_x - 0.5f), (float)S.W - 1.0f);
    const float y0f = fmaxf(ceilf(lo_y - 0.5f), 0.0f), y1f = fminf(floorf(hi_y - 0.5f), (float)S.H - 1.0f);
    if (!(x0f <= x1f && y0f <= y1f)) return false;
    B.x0 = (int)x0f; B.x1 = (int)x1f; B.y0 = (int)y0f; B.y1 = (int)y1f;
    B.pn = ((q.x - S.cam[0]) * B.nx + (q.y - S.cam[1]) * B.ny) + (q.z - S.cam[2]) * B.nz;
    return true;
}

// The fragment of sprite q at pixel (px, py), if any, into the depth image.
__device__ __forceinline__ void sp_fragment(const SpriteLaunch &S, const float4 q, const SpriteBox &B, int px, int py,
                                            uint32_t *depth)
{
    const float R = S.radius, invR = 1.0f / R;
    const float *V = S.view, *P = S.proj;
    const float o0 = S.cam[0], o1 = S.cam[1], o2 = S.cam[2];
    const float ndx = ((float)px + 0.5f) * (2.0f / (float)S.W) - 1.0f;
    const float ndy = ((float)py + 0.5f) * (2.0f / (float)S.H) - 1.0f;
    float w[4];
    sp_xform(S.inv_pv, ndx, ndy, 1.0f, w);
    // the ray direction scaled by w (no division): t d is unchanged; the
    // far point of a perspective projection has w = 1 / far > 0
    if (!(w[3] > 0.0f)) return;
    const float d0 = w[0] - o0 * w[3], d1 = w[1] - o1 * w[3], d2 = w[2] - o2 * w[3];
    const float den = (d0 * B.nx + d1 * B.ny) + d2 * B.nz;
    if (den == 0.0f) return;
    const float t = B.pn / den;
    if (!(t > 0.0f)) return;
    const float X = o0 + t * d0, Y = o1 + t * d1, Z = o2 + t * d2;
    const float rx = X - q.x, ry = Y - q.y, rz = Z - q.z;
    const float u = ((rx * B.ax + ry * B.ay) + rz * B.az) * invR;
    const float v = -(((rx * B.bx + ry * B.by) + rz * B.bz) * invR);
    const float l2 = u * u + v * v;
    if (l2 > 1.0f) return;                                     // depth.frag: discard
    float vp[4], cp[4], cs[4];
    sp_xform(V, X, Y, Z, vp);
    sp_xform(P, vp[0], vp[1], vp[2], cp);
    const float zp = cp[2] / cp[3];
    if (!(zp >= 0.0f && zp <= 1.0f)) return;                   // clipped
    const float off = sp_cos_half_pi(sqrtf(l2));
    sp_xform(P, vp[0], vp[1], vp[2] - R * off, cs);
    float z = cs[2] / cs[3];
    if (z != z) return;
    z = z <= 0.0f ? 0.0f : (z > 1.0f ? 1.0f : z);           // -0 -> +0: the bits order as the values
    // early depth test: only a nearer fragment pays for the atomic (a stale
    // read costs an atomic that changes nothing, never a wrong result)
    uint32_t *dst = &depth[(size_t)py * S.W + (size_t)px];
    const uint32_t zb = __float_as_uint(z);
    if (zb < __atomic_load_n(dst, __ATOMIC_RELAXED)) atomicMin(dst, zb);
}

// Footprints larger than this many pixels (a particle close to the eye: one
// just past the near plane covers the whole image), or than 32 tiles, are drawn by
// the whole wave.
constexpr uint32_t kSpriteBigPixels = 1024;

// When the sample is drawn first (whole passes, without -> with it, launches and
// all; an estimate of what the particles draw comes from their bounding box):
// - for many particles: the few of a small sample last as long as they hide
//   (8,192 footprints of 2,300 pixels 119 -> 172 us, 54,000 of 1,480 419 -> 185);
// - where footprints lie on each other, kCullOver or more over a pixel (11 over
//   each: 98 -> 114 us, 15: 68 -> 113, 68: 115 -> 85, 615: 1257 -> 350);
// - for a pass of some length, kCullPixels or more in all footprints (0.18 M: 44 ->
//   50 us, 0.56 M: 64 -> 55, 0.63 M: 107 -> 70).
// A pass has at least kSpriteWaves waves, a particle each if need be: 8,192 of
// 2,300 pixels 138 us with 4,096 waves, 117 with 8,192; 1,000 of 63 pixels 23 us, 174
// sixty-four to a wave.  Up to kSampleLanes64 sample sprites of more than 32 pixels
// are drawn by 64 lanes each (eight lanes: 54,000 of 657 223 us, now 108).
constexpr uint32_t kCullParticles = 16384;
constexpr double kCullOver = 30.0, kCullPixels = 5e5;
constexpr uint32_t kSampleLanes64 = 16384, kSpriteWaves = 8192, kOwnPixels = 64;

// The particle of block t (of kSampleStride consecutive ones) that is drawn
// first; hashed, so the sample has no period of a lattice's.
constexpr uint32_t kSampleStride = 16;
__device__ __forceinline__ uint32_t sp_sample(uint32_t t)
{
    uint32_t x = t * 0x9e3779b1u;
    x ^= x >> 15;
    return t * kSampleStride + ((x * 0x85ebca77u >> 16) & (kSampleStride - 1));
}
static_assert((kSampleStride & (kSampleStride - 1)) == 0, "sp_sample takes bits of the hash");

// The footprint of one sprite by `lanes` lanes (j: this one), pixels in row order.
__device__ __forceinline__ void sp_draw(const SpriteLaunch &S, const float4 q, const SpriteBox &B, uint32_t j, uint32_t lanes,
                                        uint32_t *depth)
{
    const int bw = B.x1 - B.x0 + 1;
    int px = B.x0 + (int)j, py = B.y0;
    while (true) {
        while (px > B.x1) { px -= bw; py++; }
        if (py > B.y1) break;
        sp_fragment(S, q, B, px, py, depth);
        px += (int)lanes;
    }
}

__device__ __forceinline__ uint32_t sp_area(const SpriteBox &B)
{
    return (uint32_t)(B.x1 - B.x0 + 1) * (uint32_t)(B.y1 - B.y0 + 1);
}

__device__ __forceinline__ bool sp_is_big(const SpriteBox &B)
{
    const uint32_t tiles = (uint32_t)((B.x1 >> 3) - (B.x0 >> 3) + 1) * (uint32_t)((B.y1 >> 3) - (B.y0 >> 3) + 1);
    return sp_area(B) > kSpriteBigPixels || tiles > 32u;
}

// The sample: `lanes` lanes (8 or 64) per sprite, so its few sprites fill the chip.
// Sprites of more than 256 pixels a lane are left to the second pass.
__global__ __launch_bounds__(256) void k_sprites_sample(SpriteLaunch S, const float4 *__restrict__ pts, uint32_t n,
                                                        uint32_t lanes, uint32_t *depth)
{
    const uint64_t g = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    const uint32_t t = (uint32_t)(g / lanes), j = (uint32_t)g & (lanes - 1u);
    const uint32_t i = sp_sample(t);
    if (i >= n) return;
    const float4 q = pts[i];
    SpriteBox B;
    if (!sp_box(S, q, B)) return;
    if (sp_area(B) > 256u * lanes) return;
    sp_draw(S, q, B, j, lanes, depth);
}

// All particles, or with tmax what of them is not hidden.  A lane tests one
// particle against its footprint's tiles and draws a footprint of at most `own`
// pixels itself (up to as many as the wave has particles: a lane each then beats
// eight lanes for one after the other; 1 M of 1.4 pixels 112 -> 68 us); the wave then
// draws the open (particle, tile) pairs of the others, eight lanes per pair and a
// row of the tile at a time, and the large ones in turn, all lanes on one.  (1 M
// dam break at 1080p, 168 us: drawn whole by the testing lane 740 us; whole by eight
// lanes each 314; with a depth test per pixel ahead of the arithmetic 450, a chain
// of loads.)
// A wave takes `per` particles: with tmax from all over the cloud (scattered), so
// every wave gets its share of the visible ones (64 neighbours each: 427 against
// 168 us); else neighbours, read in order.
struct SpriteItem {
    float4 q;
    int x0, x1, y0, y1;
    float pn;
};
constexpr uint32_t kSpritePairs = 256;

__global__ __launch_bounds__(256) void k_depth_sprites(SpriteLaunch S, const float4 *__restrict__ pts, uint32_t n,
                                                       uint32_t nw, uint32_t per, uint32_t own, uint32_t *depth,
                                                       const uint32_t *__restrict__ tmax)
{
    __shared__ SpriteItem item[4][64];
    __shared__ uint16_t pair[4][kSpritePairs + 64];          // lane | bit << 6
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, tiles_x = (S.W + 7) / 8;
    const uint32_t w = blockIdx.x * 4u + wave;
    const uint64_t i = tmax ? (uint64_t)lane * nw + w : (uint64_t)w * per + lane;
    uint32_t open = 0;
    bool big = false;
    if (w < nw && lane < per && i < n) {
        const float4 q = pts[i];
        SpriteBox B;
        if (sp_box(S, q, B)) {
            big = sp_is_big(B);
            if (!big) open = sp_open(B, tmax ? sp_near(S, q) : -1.0f, tmax, tiles_x);
            if (big || sp_area(B) > own) {
                item[wave][lane] = SpriteItem{ q, B.x0, B.x1, B.y0, B.y1, B.pn };
            } else if (open) {
                sp_draw(S, q, B, 0u, 1u, depth);
                open = 0;
            }
        }
    }
    const uint32_t g = lane / 8u, j = lane % 8u;
    uint32_t count = 0;
    while (true) {
        const unsigned long long m = __ballot(open != 0);
        if (m) {                                             // one more pair of every lane that has one
            if (open) {
                const uint32_t bit = (uint32_t)__ffs(open) - 1u;
                open &= open - 1u;
                pair[wave][count + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)(lane | bit << 6);
            }
            count += (uint32_t)__popcll(m);
            if (count <= kSpritePairs) continue;
        }
        wave_lds_sync();
        for (uint32_t k = g; k < count; k += 8u) {
            const uint32_t p = pair[wave][k], bit = p >> 6;
            const SpriteItem it = item[wave][p & 63u];
            SpriteBox B;
            sp_plane(S, B);
            B.pn = it.pn;
            const uint32_t tw = ((uint32_t)it.x1 >> 3) - ((uint32_t)it.x0 >> 3) + 1;
            const int tx = (it.x0 >> 3) + (int)(bit % tw), ty = (it.y0 >> 3) + (int)(bit / tw);
            const int px = 8 * tx + (int)j;
            const int ya = max(it.y0, 8 * ty), yb = min(it.y1, 8 * ty + 7);
            if (px >= it.x0 && px <= it.x1)
                for (int py = ya; py <= yb; py++) sp_fragment(S, it.q, B, px, py, depth);
        }
        if (!m) break;
        wave_lds_sync();
        count = 0;
    }
    // large ones: whole rows where most tiles are open, else tile by tile
    for (unsigned long long todo = __ballot(big); todo != 0; todo &= todo - 1ull) {
        const SpriteItem it = item[wave][(uint32_t)__ffsll((long long)todo) - 1u];
        SpriteBox B;
        sp_plane(S, B);
        B.x0 = it.x0; B.x1 = it.x1; B.y0 = it.y0; B.y1 = it.y1;
        B.pn = it.pn;
        const uint32_t tx0 = (uint32_t)B.x0 >> 3, ty0 = (uint32_t)B.y0 >> 3;
        const uint32_t tw = ((uint32_t)B.x1 >> 3) - tx0 + 1, T = tw * (((uint32_t)B.y1 >> 3) - ty0 + 1);
        uint32_t nopen = T;
        const float zn = tmax ? sp_near(S, it.q) : -1.0f;
        auto is_open = [&](uint32_t t) { return zn < __uint_as_float(tmax[(ty0 + t / tw) * tiles_x + tx0 + t % tw]); };
        if (tmax) {
            nopen = 0;
            for (uint32_t t0 = 0; t0 < T; t0 += 64u)
                nopen += (uint32_t)__popcll(__ballot(t0 + lane < T && is_open(min(t0 + lane, T - 1))));
        }
        if (2 * nopen > T) {
            sp_draw(S, it.q, B, lane, 64u, depth);
            continue;
        }
        for (uint32_t t0 = 0; t0 < T && nopen != 0; t0 += 64u) {
            unsigned long long tiles = __ballot(t0 + lane < T && is_open(min(t0 + lane, T - 1)));
            for (; tiles != 0; tiles &= tiles - 1ull) {
                const uint32_t k = t0 + (uint32_t)__ffsll((long long)tiles) - 1u;
                const int px = (int)((tx0 + k % tw) * 8u + (lane & 7u)), py = (int)((ty0 + k / tw) * 8u + (lane >> 3));
                if (px >= B.x0 && px <= B.x1 && py >= B.y0 && py <= B.y1) sp_fragment(S, it.q, B, px, py, depth);
            }
        }
    }
}

// Largest depth of every 8x8 tile, one wave each.
__global__ __launch_bounds__(256) void k_tile_max(const uint32_t *__restrict__ depth, uint32_t W, uint32_t H,
                                                  uint32_t *__restrict__ tmax, uint32_t T)
{
    const uint32_t t = blockIdx.x * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (t >= T) return;   // whole wave
    const uint32_t tiles_x = (W + 7) / 8;
    const uint32_t px = (t % tiles_x) * 8 + (lane & 7u), py = (t / tiles_x) * 8 + (lane >> 3);
    uint32_t v = px < W && py < H ? depth[(size_t)py * W + px] : 0u;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const uint32_t o = __shfl_xor(v, off, 64);
        v = v > o ? v : o;
    }
    if (lane == 0) tmax[t] = v;
}

__global__ __launch_bounds__(256) void k_clear_sprites(uint32_t *depth, uint64_t n)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i < n) depth[i] = 0x3f800000u;                             // 1.0f: the depth clear value
}

// Whether sp_near bounds the fragments' depths: the rows of View orthonormal,
// and a projection whose z and w come from view z alone, with
// z / w = (a z + b) / (c z + d) growing where w > 0 (a d - b c > 0).
static bool sp_cull(const SpriteLaunch &S)
{
    const float *V = S.view, *P = S.proj;
    for (int a = 0; a < 3; a++)
        for (int b = a; b < 3; b++) {
            const float dot = V[a] * V[b] + V[4 + a] * V[4 + b] + V[8 + a] * V[8 + b];
            if (!(fabsf(dot - (a == b ? 1.0f : 0.0f)) < 1e-4f)) return false;
        }
    if (V[3] != 0.0f || V[7] != 0.0f || V[11] != 0.0f || V[15] != 1.0f) return false;
    return P[2] == 0.0f && P[6] == 0.0f && P[3] == 0.0f && P[7] == 0.0f && P[11] >= 0.0f &&
           P[10] * P[15] - P[14] * P[11] > 0.0f;
}

// What the particles draw, from their bounding box: the pixels of a footprint at
// its centre, and the footprints over a pixel of its rectangle on the screen.
struct SpriteEstimate {
    double area, over;
};
static SpriteEstimate sp_estimate(const SpriteLaunch &S, uint32_t n)
{
    const float *V = S.view, *P = S.proj;
    auto clip = [&](const double x[3], double c[4]) {
        double v[4];
        for (int r = 0; r < 4; r++) v[r] = V[r] * x[0] + V[4 + r] * x[1] + V[8 + r] * x[2] + V[12 + r];
        for (int r = 0; r < 4; r++) c[r] = P[r] * v[0] + P[4 + r] * v[1] + P[8 + r] * v[2] + P[12 + r];
    };
    const double px = (double)S.W * S.H;
    double mid[3], c[4], lo[2] = { 1.0, 1.0 }, hi[2] = { -1.0, -1.0 };
    bool inside = false;
    for (int k = 0; k < 8; k++) {
        const double x[3] = { k & 1 ? S.hi[0] : S.lo[0], k & 2 ? S.hi[1] : S.lo[1], k & 4 ? S.hi[2] : S.lo[2] };
        clip(x, c);
        inside = inside || !(c[3] > 0.0);
        for (int a = 0; a < 2; a++) {
            lo[a] = fmin(lo[a], fmax(c[a] / c[3], -1.0));
            hi[a] = fmax(hi[a], fmin(c[a] / c[3], 1.0));
        }
    }
    for (int a = 0; a < 3; a++) mid[a] = 0.5 * ((double)S.lo[a] + S.hi[a]);
    clip(mid, c);
    const double w = fmax(c[3], 1e-3 * fabs(S.radius)), rect = inside ? 1.0 : fmax((hi[0] - lo[0]) * (hi[1] - lo[1]) / 4.0, 0.0);
    SpriteEstimate e;
    e.area = fmin((double)S.radius * S.radius * fabs((double)P[0] * P[5]) * px / (w * w), px);
    e.over = n * e.area / fmax(rect * px, 1.0);
    return e;
}

hipError_t launch_depth_sprites(const SpriteLaunch &S, const float4 *pts, uint32_t n, uint32_t *depth, uint32_t *tmax,
                                hipStream_t st)
{
    const uint64_t npx = (uint64_t)S.W * S.H;
    hipLaunchKernelGGL(k_clear_sprites, dim3((unsigned)((npx + 255) / 256)), dim3(256), 0, st, depth, npx);
    if (!n) return hipGetLastError();
    const uint32_t T = ((S.W + 7) / 8) * ((S.H + 7) / 8);
    const uint32_t *bound = nullptr;
    const SpriteEstimate e = sp_estimate(S, n);
    if (n >= kCullParticles && sp_cull(S) && e.over >= kCullOver && n * e.area >= kCullPixels) {
        const uint32_t ns = (n + kSampleStride - 1) / kSampleStride;
        const uint32_t lanes = ns < (1u << 24) && e.area > (ns <= kSampleLanes64 ? 32.0 : 256.0) ? 64u : 8u;
        hipLaunchKernelGGL(k_sprites_sample, dim3((uint32_t)(((uint64_t)ns * lanes + 255) / 256)), dim3(256), 0, st, S, pts, n,
                           lanes, depth);
        hipLaunchKernelGGL(k_tile_max, dim3((T + 3) / 4), dim3(256), 0, st, (const uint32_t *)depth, S.W, S.H, tmax, T);
        bound = tmax;
    }
    // few particles: fewer to a wave, so they fill the chip
    const uint32_t waves = std::max((n + 63u) / 64u, std::min(n, kSpriteWaves)), per = (n + waves - 1) / waves;
    const uint32_t nw = (n + per - 1) / per, own = bound ? 0u : std::min(per, kOwnPixels);
    hipLaunchKernelGGL(k_depth_sprites, dim3((nw + 3) / 4), dim3(256), 0, st, S, pts, n, nw, per, own, depth, bound);
    return hipGetLastError();
}

}  // namespace pm
