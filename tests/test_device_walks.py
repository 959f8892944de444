"""The march-grid walks of csrc/pm_device.h compiled for the CPU, one lane as a
wave of its own and every buffer checked (AddressSanitizer), so reads beyond the
cell table show without a GPU."""
import pathlib
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]

# What pm_device.h needs of the HIP headers, for a wave of one lane.
STUB = r"""
#pragma once
#include <cmath>
#include <cstdint>
#include <cstdlib>
#define __device__
#define __forceinline__ inline
#define __ballot(p) ((p) ? 1ull : 0ull)
#define __builtin_amdgcn_rsqf(x) (1.0f / std::sqrt(x))
using std::fabs; using std::sqrt;
struct float4 { float x, y, z, w; };
"""

# A frame's march grid as the build lays it out (cells of h/2, four cells of
# margin, cell-major, by input index inside a cell).
COMMON = r"""
#include "pm_device.h"
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

struct Frame {
    std::vector<float4> sorted;
    std::vector<uint32_t> start;
    GridDev g{};
    float pmin[3], pmax[3];
    Frame(const std::vector<float4> &p, float h)
    {
        g.h = h; g.inv_h = 1.0f / h; g.h2 = h * h; g.inv_hf = 2.0f * g.inv_h;
        g.sig = 8.0f / (PM_PI_F * h * h * h);
        g.h_d = h; g.h2_d = g.h_d * g.h_d; g.hinv_d = 1.0 / g.h_d; g.sig_d = 8.0 / (PM_PI_D * g.h_d * g.h_d * g.h_d);
        for (int a = 0; a < 3; a++) { pmin[a] = 3e38f; pmax[a] = -3e38f; }
        for (const float4 &v : p) {
            const float x[3] = { v.x, v.y, v.z };
            for (int a = 0; a < 3; a++) { pmin[a] = fminf(pmin[a], x[a]); pmax[a] = fmaxf(pmax[a], x[a]); }
        }
        int32_t fo[3], fn[3];
        for (int a = 0; a < 3; a++) {
            fo[a] = pm_key(pmin[a], g.inv_hf) - 4;
            fn[a] = pm_key(pmax[a], g.inv_hf) + 5 - fo[a];
        }
        g.fox = fo[0]; g.foy = fo[1]; g.foz = fo[2];
        g.fnx = fn[0]; g.fny = fn[1]; g.fnz = fn[2];
        const size_t nc = (size_t)fn[0] * fn[1] * fn[2];
        std::vector<std::vector<float4>> cell(nc);
        for (const float4 &v : p)
            cell[(size_t)(pm_key(v.x, g.inv_hf) - fo[0]) +
                 fn[0] * ((size_t)(pm_key(v.y, g.inv_hf) - fo[1]) + fn[1] * (size_t)(pm_key(v.z, g.inv_hf) - fo[2]))]
                .push_back(v);
        start.resize(nc + 1);
        for (size_t c = 0; c < nc; c++) {
            start[c] = (uint32_t)sorted.size();
            sorted.insert(sorted.end(), cell[c].begin(), cell[c].end());
        }
        start[nc] = (uint32_t)sorted.size();
        start.shrink_to_fit();
        sorted.shrink_to_fit();
        g.fcell_start = start.data();
        g.fsorted = sorted.data();
    }
};

static constexpr int kCap = 56;
static uint32_t lst[(kCap + kListPad) * 64];

// A jittered lattice of n[0] x n[1] x n[2] particles from `lo`.
static std::vector<float4> lattice(const int n[3], float spacing, const float lo[3], unsigned seed)
{
    std::mt19937 rng(seed);
    std::uniform_real_distribution<float> u(-0.1f * spacing, 0.1f * spacing);
    std::vector<float4> p;
    for (int z = 0; z < n[2]; z++)
        for (int y = 0; y < n[1]; y++)
            for (int x = 0; x < n[0]; x++)
                p.push_back({ lo[0] + x * spacing + u(rng), lo[1] + y * spacing + u(rng), lo[2] + z * spacing + u(rng), 0.0f });
    return p;
}
"""


def run(tmp_path, main):
    # -O0: every load of the source is made, also one whose value is dropped
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(COMMON + main)
    subprocess.run(["g++", "-std=c++17", "-O0", "-g", "-ffp-contract=off", "-w", "-fsanitize=address",
                    "-I" + str(tmp_path), "-I" + str(ROOT / "bachelor-thesis_amd" / "csrc"), str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, (out.stdout + out.stderr)[-3000:]
    return out.stdout


SEGMENT_EDGE = r"""
int main()
{
    const int n[3] = { 9, 7, 8 };
    const float lo[3] = { -0.13f, 0.21f, 0.4f }, h = 0.1f, eps = h / 32, step = h / 8;
    Frame f(lattice(n, 0.05f, lo, 1), h);
    std::mt19937 rng(2);
    std::uniform_real_distribution<float> u(-1.0f, 1.0f);
    long listed = 0, last = 0;
    for (int corner = 0; corner < 8; corner++)
        for (int i = 0; i < 20000; i++) {
            float a[3], b[3], len = 0.0f, d[3];
            for (int k = 0; k < 3; k++) { d[k] = u(rng); len += d[k] * d[k]; }
            for (int k = 0; k < 3; k++) {
                a[k] = ((corner >> k) & 1 ? f.pmax[k] : f.pmin[k]) + 1.1f * h * u(rng);
                b[k] = a[k] + step * d[k] / sqrtf(len);
            }
            int m = 0;
            for (int k = 0; k < 3; k++) d[k] = b[k] - a[k];
            if (!pm_list_segment<kCap>(f.g, a, d, 0.0f, 1.0f, eps, lst, m)) continue;
            listed++;
            BoxWalk w;
            const float l[3] = { fminf(a[0], b[0]) - eps, fminf(a[1], b[1]) - eps, fminf(a[2], b[2]) - eps };
            const float r[3] = { fmaxf(a[0], b[0]) + eps, fmaxf(a[1], b[1]) + eps, fmaxf(a[2], b[2]) + eps };
            pm_box_begin(f.g, l, r, w);
            last += (int)w.kh[1] + 2 - f.g.foy == f.g.fny - 1 && (int)w.kh[2] + 2 - f.g.foz == f.g.fnz - 1;
        }
    std::printf("%ld %ld\n", listed, last);
}
"""


def test_segment_list_at_the_grid_edge(tmp_path):
    """Segments around every corner of the particles' box, up to the last cells
    a 5-cell stencil fits in: no row bound is read beyond the cell table."""
    listed, last = map(int, run(tmp_path, SEGMENT_EDGE).split())
    assert listed > 10000 and last > 100


BOX_ENDS = r"""
int main()
{
    const int n[3] = { 9, 7, 8 };
    const float lo[3] = { -0.2f, -0.17f, -0.23f }, h = 0.1f;
    Frame f(lattice(n, 0.05f, lo, 1), h);
    const float offsets[] = { NAN, INFINITY, -INFINITY, 3e38f, -3e38f, 1e9f, -1e9f };
    static float buf[96 * 64];
    const float a[3] = { 0.0f, 0.0f, 0.0f }, d[3] = { 1.0f, 0.0f, 0.0f };
    int bad = 0, m = 0;
    for (float e : offsets) {
        bad += pm_list_segment<kCap>(f.g, a, d, 0.0f, 0.01f, fabsf(e), lst, m);
        bad += pm_box_cand(f.g, a, e) != 0xffffffffu;
        bad += pm_cdiff6_lds<96>(f.g, 0.0f, 0.0f, 0.0f, e, buf, true).cand != 0xffffffffu;
    }
    std::printf("%d %d\n", bad, (int)pm_list_segment<kCap>(f.g, a, d, 0.0f, 0.01f, h / 32, lst, m));
}
"""


def test_box_without_keys(tmp_path):
    """An offset that is not a number, infinite or beyond any grid has no box: no
    fused walk, no list (a NaN offset would otherwise list nothing)."""
    assert run(tmp_path, BOX_ENDS).split() == ["0", "1"]


BOX_CAND = r"""
int main()
{
    const int n[3] = { 16, 15, 14 };
    const float lo[3] = { -0.3f, -0.17f, 0.23f }, h = 0.1f;
    Frame f(lattice(n, 0.05f, lo, 1), h);
    static float buf[96 * 64];
    std::mt19937 rng(3);
    std::uniform_real_distribution<float> u(0.0f, 1.0f);
    long differ = 0, most = 0, seven = 0;
    const float offsets[] = { 0.0f, h / 32, -h / 32, 0.02f, 0.026f, 0.03f, -0.03f, 0.06f, 0.1f };
    for (float eps : offsets)
        for (int i = 0; i < 400; i++) {
            float x[3];
            for (int a = 0; a < 3; a++) x[a] = f.pmin[a] + (f.pmax[a] - f.pmin[a]) * u(rng);
            const Cdiff6 o = pm_cdiff6_lds<96>(f.g, x[0], x[1], x[2], eps, buf, true);
            const uint32_t c = pm_box_cand(f.g, x, eps);
            differ += c != o.cand;
            seven += fabsf(eps) >= 0.026f && o.cand != 0xffffffffu;
            if (o.cand != 0xffffffffu && (long)o.cand > most) most = o.cand;
        }
    std::printf("%ld %ld %ld\n", differ, most, seven);
}
"""


def test_box_candidates(tmp_path):
    """The count without a walk is the six-sample walk's, also where the box
    spans seven rows or more (offsets beyond h / 4)."""
    differ, most, seven = map(int, run(tmp_path, BOX_CAND).split())
    assert differ == 0 and most > 100 and seven > 500


FAR_EYE = r"""
int main()
{
    const int n[3] = { 12, 12, 12 };
    const float lo3[3] = { 0.2f, 0.2f, 0.2f }, h = 0.1f, eps = h / 32;
    Frame f(lattice(n, 0.05f, lo3, 1), h);
    std::mt19937 rng(5);
    std::uniform_real_distribution<float> u(-1.0f, 1.0f);
    long listed = 0, missing = 0, within = 0;
    const float dist[] = { 2.0f, 2e2f, 2e3f, 2e4f, 2e5f };
    for (float D : dist)
        for (int i = 0; i < 4000; i++) {
            float d[3], o[3], s = 0.0f;
            for (int k = 0; k < 3; k++) { d[k] = u(rng); s += d[k] * d[k]; }
            for (int k = 0; k < 3; k++) {
                d[k] /= sqrtf(s);
                o[k] = (0.475f + 0.3f * u(rng)) - D * d[k];
            }
            const float lo = D, hi = lo + h / 8;
            int m = 0;
            if (!pm_list_segment<kCap>(f.g, o, d, lo, hi, eps, lst, m)) continue;
            listed++;
            for (int j = 0; j < 10; j++) {
                // bracket ends and midpoints; the FP64 sample; the central differences of its point
                const float t = j == 0 ? lo : j == 1 ? hi : fminf(fmaxf(lo + (hi - lo) * (0.5f + 0.5f * u(rng)), lo), hi);
                const double td = ((double)lo + (double)t) * 0.5;
                double q[3], h2 = f.g.h2_d;
                for (int k = 0; k < 3; k++) {
                    q[k] = (double)o[k] + td * (double)d[k];
                    if (j < 4) q[k] = o[k] + t * d[k];
                    if (j > 5) q[k] = (float)q[k];
                }
                if (j > 6) q[j - 7] = (float)q[j - 7] + (j & 1 ? eps : -eps);
                for (size_t p = 0; p < f.sorted.size(); p++) {
                    const double rx = f.sorted[p].x - q[0], ry = f.sorted[p].y - q[1], rz = f.sorted[p].z - q[2];
                    if (!((rx * rx + ry * ry) + rz * rz < h2 * (j == 4 || j == 5 ? 1.0 : 0.999999))) continue;
                    within++;
                    bool found = false;
                    for (int k = 0; k < m; k++) found = found || lst[k * 64] == p;
                    missing += !found;
                }
            }
        }
    std::printf("%ld %ld %ld\n", listed, within, missing);
}
"""


def test_segment_list_of_a_far_eye(tmp_path):
    """Every particle within h of any of a hit's samples is in its list, from
    20 h to 2,000,000 h away (where the coordinates' rounding outgrows h and no
    list is made)."""
    listed, within, missing = map(int, run(tmp_path, FAR_EYE).split())
    assert listed > 12000 and within > 10 ** 6 and missing == 0
