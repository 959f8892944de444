// pm_tiles.h -- the configured march of a wave, shared by the isotropic and the
// anisotropic kernels: a ray's steps, lane groups, and the split of a launch's
// active tiles over waves.
#pragma once

#include "pm_internal.h"
#include "pm_ray.h"

namespace pm {

// The first sample k at or above iso is known and the ray's march ends: its
// record (at the pixel) holds the bracket [t_{k-1}, t_k] of the bisection, or
// t itself (the ray starts inside the surface, or no bisection is asked for).
// Record: (1 | bracket << 1, lo, hi, 0); a miss leaves zeros.
// lead: this lane writes (the others of a lane group share the ray).
__device__ __forceinline__ void emit_hit(const MarchLaunch &L, RayState &r, bool lead = true)
{
    const pm_settings &s = L.s;
    float lo = r.tn, hi = r.tn;
    bool bracket = false;
    if (r.k != 0) {
        lo = r.tn + (float)(r.k - 1) * s.step;
        hi = r.tn + (float)r.k * s.step;
        bracket = s.bisect_iters > 0;
        if (!bracket) lo = hi = (lo + hi) * 0.5f;
    }
    if (lead) L.hit_rec[r.idx] = make_uint4(bracket ? 3u : 1u, __float_as_uint(lo), __float_as_uint(hi), 0u);
    r.phase = PH_DONE;
}

// First half of one step: the sample point of the lane's next FP32 density
// evaluation, after the skips of the march phase; false when the lane takes
// no sample this step (the ray ended, or it used up its HOPS skips).  Past an
// exactly skipped stretch the learned march may ask for proposals again.
template <int HOPS>
__device__ __forceinline__ bool ray_prepare(const MarchLaunch &L, RayState &r, float &qx, float &qy, float &qz)
{
    const pm_settings &s = L.s;
    const GridDev &g = L.g;
    const float o0 = L.cam[0], o1 = L.cam[1], o2 = L.cam[2];

    // at most HOPS skips per step: a lane crossing much skippable space
    // then idles for a step instead of holding the whole wave in this loop
    // (a skip costs a few dozen instructions, a step a density walk)
    for (int hop = 0;; hop++) {
        float t = r.tn + (float)r.k * s.step;
        if (t > r.tf || (s.max_steps > 0 && r.k >= s.max_steps)) {
            march_miss(L, r.idx);
            r.phase = PH_DONE;
            return false;
        }
        qx = o0 + t * r.d0; qy = o1 + t * r.d1; qz = o2 + t * r.d2;
        int kn;
        if (s.skip_mode == PM_SKIP_BOUND) kn = pm_skip_bound(g, o0, o1, o2, r, qx, qy, qz, L.inv_step);
        else if (s.skip_mode == PM_SKIP_EMPTY) kn = pm_skip_empty(g, o0, o1, o2, r, qx, qy, qz, s.step);
        else return true;
        if (kn == r.k) return true;
        r.k = kn;
        r.lrn = s.learned;
        if (hop == HOPS - 1) return false;
    }
}

// The counts of one FP32 density evaluation at q (instrumented launches also
// count its own stencil and its 27 search cells).
template <bool INSTR>
__device__ __forceinline__ void count_sample(const GridDev &g, float qx, float qy, float qz, uint32_t cand, bool march,
                                             Counts &cn)
{
    cn.samples++;
    cn.cand += cand;
    if (march) {
        cn.march++;
        cn.mcand += cand;
    }
    if (INSTR) {
        cn.cst += cand;
        cn.c27 += pm_cand27(g, qx, qy, qz);
    }
}

// Second half: the sample's density rho (and its stencil candidate count)
// ends the march, asks for a proposal or moves to the next sample.
template <bool INSTR>
__device__ __forceinline__ void ray_finish(const MarchLaunch &L, RayState &r, float rho, uint32_t cand, float qx,
                                           float qy, float qz, Counts &cn)
{
    count_sample<INSTR>(L.g, qx, qy, qz, cand, true, cn);
    if (rho >= L.s.iso) {
        emit_hit(L, r);
        cn.in_aabb += kTileHit;
    } else if (r.lrn && rho < L.mlp_gate_rho) {
        r.rho = rho;
        r.phase = PH_PROPOSE;
    } else {
        r.k++;
    }
}

// One march sample of this ray and the transition it implies.  Dens(q, cand) is
// the FP32 density.  HOPS: skips per step before a lane idles.
template <bool INSTR, int HOPS, class Dens>
__device__ __forceinline__ void ray_step(const MarchLaunch &L, RayState &r, Dens dens, Counts &cn)
{
    float qx, qy, qz;
    if (!ray_prepare<HOPS>(L, r, qx, qy, qz)) return;
    uint32_t cand = 0;
    float rho = dens(qx, qy, qz, cand);
    ray_finish<INSTR>(L, r, rho, cand, qx, qy, qz, cn);
}

// ---- lane groups ----
// As a tile's rays end, its remaining ones are spread over the wave's idle lanes:
// G lanes (a power of two) per ray, every lane of a group holding the same
// RayState.  A step then evaluates the G lattice samples k .. k+G-1 at once and
// takes the first at or above iso.  Each sample is computed as the one-lane
// march computes it, and a sample the skip would pass has its density below
// iso, so the first crossing, the bracket and the image are those of the
// one-lane march.  Counters count what the one-lane march evaluates: the
// samples the skip keeps, up to the crossing.

// The ray's state to LDS and back (region: 64 floats per field).
__device__ __forceinline__ void state_put(float *region, uint32_t slot, const RayState &r)
{
    float *p = region + slot;
    p[0 * 64] = r.d0; p[1 * 64] = r.d1; p[2 * 64] = r.d2; p[3 * 64] = r.tn; p[4 * 64] = r.tf;
    p[5 * 64] = __int_as_float(r.k); p[6 * 64] = __int_as_float(r.phase); p[7 * 64] = __uint_as_float(r.idx);
    p[8 * 64] = r.id0; p[9 * 64] = r.id1; p[10 * 64] = r.id2;
}

__device__ __forceinline__ void state_get(const float *region, uint32_t slot, RayState &r)
{
    const float *p = region + slot;
    r.d0 = p[0 * 64]; r.d1 = p[1 * 64]; r.d2 = p[2 * 64]; r.tn = p[3 * 64]; r.tf = p[4 * 64];
    r.k = __float_as_int(p[5 * 64]); r.phase = __float_as_int(p[6 * 64]); r.idx = __float_as_uint(p[7 * 64]);
    r.id0 = p[8 * 64]; r.id1 = p[9 * 64]; r.id2 = p[10 * 64];
    r.lrn = 0;
    if (r.phase == PH_PROPOSE) { r.phase = PH_MARCH; r.k++; }   // below iso, and no proposals in groups
}

// Widens the groups when the busy rays fit in fewer lanes: G becomes the
// largest power of two with (busy rays) x G <= 64.  Called by all 64 lanes.
template <class State>
__device__ __forceinline__ void regroup(State &r, int &G, float *region)
{
    const uint32_t lane = threadIdx.x & 63;
    const unsigned long long lead = __ballot(r.phase != PH_DONE && (lane & (uint32_t)(G - 1)) == 0);
    const int nb = __popcll(lead);
    int Gn = 1;
    while (Gn < 64 && nb * Gn * 2 <= 64) Gn *= 2;
    if (Gn <= G || nb == 0) return;
    if ((lead >> lane) & 1ull) state_put(region, (uint32_t)__popcll(lead & ((1ull << lane) - 1ull)), r);
    wave_lds_sync();
    if ((int)(lane / (uint32_t)Gn) < nb) state_get(region, lane / (uint32_t)Gn, r);
    else r.phase = PH_DONE;
    wave_lds_sync();
    G = Gn;
}

// Lane j of its group: its sample of this step; false when it takes none.
// nonskip: the sample is one the one-lane march would evaluate.
__device__ __forceinline__ bool group_prepare(const MarchLaunch &L, RayState &r, int G, int j, float &qx, float &qy,
                                              float &qz, bool &nonskip)
{
    const pm_settings &s = L.s;
    const GridDev &g = L.g;
    const float o0 = L.cam[0], o1 = L.cam[1], o2 = L.cam[2];
    nonskip = false;
    // the group's first sample, as ray_prepare finds it; the wave has few
    // rays left, so a group may take 8 G skips in one step
    const int hop_cap = 8 * G - 1;
    for (int hop = 0;; hop++) {
        float t = r.tn + (float)r.k * s.step;
        if (t > r.tf || (s.max_steps > 0 && r.k >= s.max_steps)) {
            if (j == 0) march_miss(L, r.idx);
            r.phase = PH_DONE;
            return false;
        }
        qx = o0 + t * r.d0; qy = o1 + t * r.d1; qz = o2 + t * r.d2;
        int kn = r.k;
        if (s.skip_mode == PM_SKIP_BOUND) kn = pm_skip_bound(g, o0, o1, o2, r, qx, qy, qz, L.inv_step);
        else if (s.skip_mode == PM_SKIP_EMPTY) kn = pm_skip_empty(g, o0, o1, o2, r, qx, qy, qz, s.step);
        if (kn == r.k) break;
        r.k = kn;
        if (hop == hop_cap) return false;
    }
    if (j == 0) { nonskip = true; return true; }
    const int kj = r.k + j;
    const float t = r.tn + (float)kj * s.step;
    if (t > r.tf || (s.max_steps > 0 && kj >= s.max_steps)) return false;
    qx = o0 + t * r.d0; qy = o1 + t * r.d1; qz = o2 + t * r.d2;
    // (a skip returns a later sample than r.k exactly where q may be skipped)
    nonskip = s.skip_mode == PM_SKIP_BOUND   ? pm_skip_bound(g, o0, o1, o2, r, qx, qy, qz, L.inv_step) == r.k
              : s.skip_mode == PM_SKIP_EMPTY ? pm_skip_empty(g, o0, o1, o2, r, qx, qy, qz, s.step) == r.k
                                             : true;
    return true;
}

// The group's transition from its lanes' densities.  Called by all 64 lanes.
template <bool INSTR>
__device__ __forceinline__ void group_finish(const MarchLaunch &L, RayState &r, int G, int j, bool want, bool nonskip,
                                             float rho, uint32_t cand, float qx, float qy, float qz, Counts &cn)
{
    const uint32_t lane = threadIdx.x & 63, gbase = lane & ~(uint32_t)(G - 1);
    const unsigned long long gmask = G == 64 ? ~0ull : ((1ull << G) - 1ull);
    const unsigned long long cross = (__ballot(want && rho >= L.s.iso) >> gbase) & gmask;
    const unsigned long long wants = (__ballot(want) >> gbase) & gmask;
    if (r.phase != PH_MARCH || !(wants & 1ull)) return;
    const int jc = cross ? __ffsll((long long)cross) - 1 : G;
    if (want && nonskip && j <= jc) count_sample<INSTR>(L.g, qx, qy, qz, cand, true, cn);
    if (cross) {
        r.k += jc;
        emit_hit(L, r, j == 0);
        if (j == 0) cn.in_aabb += kTileHit;
    } else {
        r.k += G;
    }
}

// One step of the wave's groups (all 64 lanes).
template <bool INSTR, class Dens>
__device__ __forceinline__ void group_step(const MarchLaunch &L, RayState &r, int G, Dens dens, Counts &cn)
{
    const int j = (int)(threadIdx.x & (uint32_t)(G - 1));
    float qx = 0.f, qy = 0.f, qz = 0.f, rho = 0.f;
    bool nonskip = false, want = false;
    uint32_t cand = 0;
    if (r.phase != PH_DONE) want = group_prepare(L, r, G, j, qx, qy, qz, nonskip);
    if (want) rho = dens(qx, qy, qz, cand);
    group_finish<INSTR>(L, r, G, j, want, nonskip, rho, cand, qx, qy, qz, cn);
}

// Active tile i of a launch's list for wave `w` of the grid (one-wave
// workgroups, dispatched to the 8 XCDs round-robin): runs of kXcdRun
// consecutive tiles go to the XCDs in turn, so neighbouring tiles share an L2
// and every XCD gets its share of a dense region.
static constexpr uint32_t kXcdRun = 32;
__device__ __forceinline__ uint32_t xcd_tile(uint32_t w)
{
    const uint32_t local = w >> 3;
    return ((local / kXcdRun) * 8 + (w & 7u)) * kXcdRun + local % kXcdRun;
}

// Workgroups for T tiles (all of them may be active): a multiple of a full
// round of runs; beyond kMaxWaves each wave takes several tiles (16,384 waves
// left some with two tiles of the 4K pool: 4.9 against 3.6 ms in the finish).
static constexpr uint32_t kMaxWaves = 65536;
__host__ __device__ __forceinline__ uint32_t tile_waves_of(uint32_t T)
{
    return (T + 8 * kXcdRun - 1) / (8 * kXcdRun) * (8 * kXcdRun);
}

// Waves per tile of the march, as a power of two, for TA active tiles.  The
// chip holds about 4,096 of its waves: with fewer tiles a launch lasts as long
// as its longest tile (a ray along a face takes a hundred samples), so each tile
// is split over four waves whose rays start with four lanes each; the samples
// evaluated past a crossing cost less than the idle SIMDs.  March kernel for
// one / two / four / eight waves per tile: 640x480 lattice cube (3,200 tiles)
// 493 / 354 / 268 / 354 us, 96x64 213 / 156 / 130 / 152 us, 1080p dam break
// (4,300) 331 / 297 / 318 / 448 us, 4K pool (19,000) 2,490 / 2,578 / 2,899 /
// 5,184 us.
static constexpr uint32_t kResidentWaves = 4096, kMaxSplit = 2;
__host__ __device__ __forceinline__ uint32_t tile_split(uint32_t TA)
{
    return TA < kResidentWaves ? 2u : (TA < 2 * kResidentWaves ? 1u : 0u);
}

// The same for the finish of the hits: four lanes per hit where the tiles fill
// less than half of the chip (two would not shorten the bisection).
__device__ __forceinline__ uint32_t finish_split(uint32_t TA) { return TA < kResidentWaves / 2 ? 2u : 0u; }

// Pixel of ray rr of part i mod 2^sub of a tile (the whole tile for sub = 0).
__device__ __forceinline__ void part_pixel(uint32_t tile, uint32_t tiles_x, uint32_t i, uint32_t sub, uint32_t rr,
                                           uint32_t &px, uint32_t &py)
{
    const uint32_t part = i & ((1u << sub) - 1u);
    const uint32_t lw = sub >= 2 ? 2u : 3u, np = 3u - lw;   // a part is 2^lw pixels wide, 2^np in a row
    px = (tile % tiles_x) * 8 + (part & ((1u << np) - 1u)) * (1u << lw) + (rr & ((1u << lw) - 1u));
    py = (tile / tiles_x) * 8 + (part >> np) * (64u >> sub >> lw) + (rr >> lw);
}

// ---- finishing a hit with G lanes ----
// The n32 FP32 bisection steps of one hit per group of G lanes: a round
// evaluates the 2^lv - 1 midpoints of the next lv = floor(log2(G + 1)) levels
// at once and descends through them; every midpoint is the one the one-lane
// bisection computes, and only those on its path are counted.  Called by all 64
// lanes; want: the group has a bracket [lo, hi].
template <class Dens>
__device__ __forceinline__ void group_bisect(const MarchLaunch &L, const float d[3], float &lo, float &hi, int n32, bool want,
                                             int G, Dens dens, Counts &cn)
{
    const uint32_t lane = threadIdx.x & 63, gbase = lane & ~(uint32_t)(G - 1);
    const int j = (int)(lane & (uint32_t)(G - 1));
    const int lvg = 31 - __clz(G + 1);
    for (int it = 0; it < n32;) {
        const int lv = min(lvg, n32 - it);
        const int node = j + 1, depth = 31 - __clz(node);   // heap order: 1 = the next midpoint
        float rho = 0.0f;
        uint32_t cand = 0;
        if (want && node < (1 << lv)) {
            float l = lo, h = hi;
            for (int b = depth - 1; b >= 0; b--) {      // left child: the crossing lies below the midpoint
                const float tm = (l + h) * 0.5f;
                if ((node >> b) & 1) l = tm; else h = tm;
            }
            const float tm = (l + h) * 0.5f;
            rho = dens(L.cam[0] + tm * d[0], L.cam[1] + tm * d[1], L.cam[2] + tm * d[2], cand);
        }
        int at = 1;
        for (int l = 0; l < lv; l++) {
            const float rn = __shfl(rho, (int)gbase + at - 1, 64);
            if (want && j == at - 1) { cn.samples++; cn.cand += cand; }
            const float tm = (lo + hi) * 0.5f;
            if (rn >= L.s.iso) { hi = tm; at = 2 * at; } else { lo = tm; at = 2 * at + 1; }
        }
        it += lv;
    }
}

// The central differences of the density at p, one sample per lane of the
// group at a time.  Called by all 64 lanes; want as above.
template <class Dens>
__device__ __forceinline__ void group_cdiff(const float p[3], float eps, bool want, int G, Dens dens, float gv[3],
                                            Counts &cn)
{
    const uint32_t lane = threadIdx.x & 63, gbase = lane & ~(uint32_t)(G - 1);
    const int j = (int)(lane & (uint32_t)(G - 1));
    float rp[3] = { 0.f, 0.f, 0.f }, rm[3] = { 0.f, 0.f, 0.f };
    for (int k0 = 0; k0 < 6; k0 += G) {
        const int k = k0 + j;                           // +x, -x, +y, -y, +z, -z
        float rho = 0.0f;
        if (want && k < 6) {
            const float q0 = k == 0 ? p[0] + eps : (k == 1 ? p[0] - eps : p[0]);
            const float q1 = k == 2 ? p[1] + eps : (k == 3 ? p[1] - eps : p[1]);
            const float q2 = k == 4 ? p[2] + eps : (k == 5 ? p[2] - eps : p[2]);
            uint32_t cand = 0;
            rho = dens(q0, q1, q2, cand);
            cn.samples++;
            cn.cand += cand;
        }
#pragma unroll
        for (int m = 0; m < 6; m++) {
            const float v = __shfl(rho, (int)gbase + (m - k0 >= 0 && m - k0 < G ? m - k0 : 0), 64);
            if (m >= k0 && m < k0 + G) {
                if (m & 1) rm[m >> 1] = v; else rp[m >> 1] = v;
            }
        }
    }
#pragma unroll
    for (int a = 0; a < 3; a++) gv[a] = rp[a] - rm[a];
}

// normalize(-grad rho), zero where the gradient is.
__device__ __forceinline__ void cdiff_normal(const float gv[3], float &nx, float &ny, float &nz)
{
    const float dd = (gv[0] * gv[0] + gv[1] * gv[1]) + gv[2] * gv[2];
    nx = ny = nz = 0.0f;
    if (dd > 0.0f) {
        const float inv = 1.0f / sqrtf(dd);
        nx = -gv[0] * inv; ny = -gv[1] * inv; nz = -gv[2] * inv;
    }
}

// ---- the reference march of a wave ----
// PerPixel_Isotropic / PerPixel_Anisotropic (RayMarcher.cpp:256-423) over one
// part of an active tile: start on the depth-buffer surface, p += step for at
// most MaxSteps samples, the DensityGrid's cleared nodes skipped, the first
// sample with rho >= iso.  Rays that leave their lanes idle widen the others'
// groups, as in the configured march: lane j of a group takes j + 1 of the
// ray's steps (p += step and the skips, in the same order) and evaluates the
// sample it arrives at; the group takes the first crossing, or goes on from the
// last lane's point.  Hits wait in LDS until every ray of the part has ended, so
// their normals are computed by all lanes at once (inside the loop, each of a
// tile's hit steps cost the wave a normal).
struct RefState {
    float p0, p1, p2, s0, s1, s2;   // point, step vector
    int i, phase;                   // samples taken
    uint32_t slot;                  // ray of the part
};

__device__ __forceinline__ void state_put(float *region, uint32_t slot, const RefState &r)
{
    float *q = region + slot;
    q[0 * 64] = r.p0; q[1 * 64] = r.p1; q[2 * 64] = r.p2; q[3 * 64] = r.s0; q[4 * 64] = r.s1; q[5 * 64] = r.s2;
    q[6 * 64] = __int_as_float(r.i); q[7 * 64] = __int_as_float(r.phase); q[8 * 64] = __uint_as_float(r.slot);
}

__device__ __forceinline__ void state_get(const float *region, uint32_t slot, RefState &r)
{
    const float *q = region + slot;
    r.p0 = q[0 * 64]; r.p1 = q[1 * 64]; r.p2 = q[2 * 64]; r.s0 = q[3 * 64]; r.s1 = q[4 * 64]; r.s2 = q[5 * 64];
    r.i = __float_as_int(q[6 * 64]); r.phase = __float_as_int(q[7 * 64]); r.slot = __float_as_uint(q[8 * 64]);
}

// region: the lanes' lists (and the groups' hand-over); hits: 64 float4 in LDS.
template <class Dens, class Normal>
__device__ __forceinline__ void ref_part(const MarchLaunch &L, uint32_t tile, uint32_t tiles_x, uint32_t part, uint32_t sub,
                                         float *region, float4 *hits, Dens dens, Normal normal, Counts &cn)
{
    const GridDev &g = L.g;
    const pm_settings &s = L.s;
    const uint32_t lane = threadIdx.x & 63;
    const bool dg = s.skip_mode == PM_SKIP_DG_BOX || s.skip_mode == PM_SKIP_DG_CONS;
    int G = 1 << sub;
    RefState r{};
    r.phase = PH_DONE;
    r.slot = lane >> sub;
    uint32_t px, py;
    part_pixel(tile, tiles_x, part, sub, r.slot, px, py);
    if (px < L.W && py < L.H) {
        const bool lead = (lane & (uint32_t)(G - 1)) == 0;
        if (lead) cn.rays++;
        const float z = L.depth[py * L.W + px];
        if (z != 1.0f) {
            if (lead) cn.in_aabb++;
            const float cx = (float)px * (2.0f / (float)L.W) - 1.0f;
            const float cy = (float)py * (2.0f / (float)L.H) - 1.0f;
            float d0, d1, d2;
            pm_unproject(L.M, cx, cy, z, r.p0, r.p1, r.p2);
            pm_normalize(r.p0 - L.cam[0], r.p1 - L.cam[1], r.p2 - L.cam[2], d0, d1, d2);
            r.s0 = s.step * d0; r.s1 = s.step * d1; r.s2 = s.step * d2;
            if (s.max_steps > 0) r.phase = PH_MARCH;
        }
    }
    hits[lane] = make_float4(0.f, 0.f, 0.f, 0.f);
    wave_lds_sync();
    while (__ballot(r.phase != PH_DONE) != 0) {
        regroup(r, G, region);
        const int j = (int)(lane & (uint32_t)(G - 1));
        const uint32_t gbase = lane & ~(uint32_t)(G - 1);
        const unsigned long long gmask = G == 64 ? ~0ull : ((1ull << G) - 1ull);
        const bool want = r.phase != PH_DONE && r.i + j < s.max_steps;
        float p0 = r.p0, p1 = r.p1, p2 = r.p2, rho = 0.0f;
        uint32_t cand = 0;
        if (want) {
            for (int t = 0; t <= j; t++) {
                p0 += r.s0; p1 += r.s1; p2 += r.s2;
                if (dg) {                                            // RayMarcher.cpp:284-304
                    float nmin[3], nmax[3];
                    while (pm_dg_query(g, p0, p1, p2, nmin, nmax)) {
                        const float pin[3] = { p0, p1, p2 }, st[3] = { r.s0, r.s1, r.s2 };
                        float q[3];
                        pm_intersect_aabb(pin, st, nmin, nmax, q);
                        p0 = q[0] + r.s0; p1 = q[1] + r.s1; p2 = q[2] + r.s2;
                    }
                }
            }
            rho = dens(p0, p1, p2, cand);
        }
        const unsigned long long cross = (__ballot(want && rho >= s.iso) >> gbase) & gmask;
        const float l0 = __shfl(p0, (int)gbase + G - 1, 64), l1 = __shfl(p1, (int)gbase + G - 1, 64),
                    l2 = __shfl(p2, (int)gbase + G - 1, 64);
        if (r.phase == PH_DONE) continue;
        const int jc = cross ? __ffsll((long long)cross) - 1 : G;
        if (want && j <= jc) { cn.samples++; cn.march++; cn.cand += cand; }
        if (cross) {
            if (j == jc) hits[r.slot] = make_float4(p0, p1, p2, 1.0f);
            r.phase = PH_DONE;
        } else {
            r.p0 = l0; r.p1 = l1; r.p2 = l2;
            r.i += G;
            if (r.i >= s.max_steps) r.phase = PH_DONE;
        }
    }
    wave_lds_sync();
    if (lane < (64u >> sub)) {
        part_pixel(tile, tiles_x, part, sub, lane, px, py);
        if (px < L.W && py < L.H) {
            const uint32_t idx = py * L.W + px;
            const float4 P = hits[lane];
            float4 N = make_float4(0.f, 0.f, 0.f, 0.f);
            float t = -1.0f;
            if (P.w != 0.0f) {
                const float p[3] = { P.x, P.y, P.z };
                normal(p, N.x, N.y, N.z);
                N.w = 1.0f;
                const float v0 = P.x - L.cam[0], v1 = P.y - L.cam[1], v2 = P.z - L.cam[2];
                t = sqrtf((v0 * v0 + v1 * v1) + v2 * v2);
                cn.hits++;
            }
            L.pos[idx] = P;
            L.nrm[idx] = N;
            if (L.t) L.t[idx] = t;
        }
    }
    wave_lds_sync();
}

}  // namespace pm
