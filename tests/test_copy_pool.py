"""The shared host copy (csrc/pm_copy.h) on the CPU: ranges around a piece and
around the size from which the workers share, many in a row, from two pools in
two threads at once."""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include "pm_copy.h"
#include <cstdio>
#include <vector>
using pm::CopyPool;

static bool many(unsigned seed)
{
    CopyPool pool;
    const size_t P = pm::kCopyPiece, S = pm::kCopyShared;
    const size_t sizes[] = { 0, 1, P - 1, P, P + 1, S - 1, S, S + 1, 3 * S + 17 };
    for (int rep = 0; rep < 30; rep++) {
        std::vector<std::vector<unsigned char>> src(3), dst(3);
        CopyPool::Range r[3];
        for (int k = 0; k < 3; k++) {
            seed = seed * 1664525u + 1013904223u;
            const size_t n = sizes[(seed >> 8) % 9];
            src[k].resize(n + 1);
            dst[k].assign(n + 1, 7);
            for (size_t i = 0; i < n; i++) src[k][i] = (unsigned char)(i * 31 + rep + k);
            src[k][n] = 9;
            r[k] = { dst[k].data(), src[k].data(), n };
        }
        pool.copy(r, 3);
        for (int k = 0; k < 3; k++) {
            const size_t n = r[k].bytes;
            if (memcmp(dst[k].data(), src[k].data(), n) != 0 || dst[k][n] != 7) return false;
        }
    }
    return true;
}

int main()
{
    bool a = false, b = false;
    std::thread t([&] { a = many(1); });
    b = many(2);
    t.join();
    CopyPool unused;
    std::puts(a && b ? "ok" : "differs");
    return a && b ? 0 : 1;
}
"""


def test_shared_copy(tmp_path):
    src, exe = tmp_path / "copy.cpp", tmp_path / "copy"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-I" + str(ROOT / "bachelor-thesis_amd" / "csrc"), str(src), "-pthread", "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
