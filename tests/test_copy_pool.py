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


NO_MEMORY = r"""
#include "pm_copy.h"
#include <cstdio>
#include <cstdlib>
#include <new>

// The next allocations of the copying thread that fail; -1: none do.
static thread_local int left = -1;
void *operator new(size_t n)
{
    if (left == 0) throw std::bad_alloc();
    if (left > 0) left--;
    if (void *p = malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

int main()
{
    const size_t n = 3 * pm::kCopyShared + 17;
    char *a = (char *)malloc(n), *b = (char *)malloc(n);
    for (int allowed = 0; allowed < 4; allowed++) {
        pm::CopyPool pool;
        for (int rep = 0; rep < 3; rep++) {
            memset(a, 17 * rep + allowed + 1, n);
            memset(b, 0, n);
            const pm::CopyPool::Range r = { b, a, n };
            left = allowed;
            pool.copy(&r, 1);
            left = -1;
            if (memcmp(a, b, n) != 0) return 1;
        }
    }
    std::puts("ok");
    return 0;
}
"""


def test_copy_without_memory_for_workers(tmp_path):
    """No memory for the first, second or third worker: the copy is made by those
    there are, and nothing is thrown."""
    src, exe = tmp_path / "copy.cpp", tmp_path / "copy"
    src.write_text(NO_MEMORY)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-I" + str(ROOT / "bachelor-thesis_amd" / "csrc"), str(src),
                    "-pthread", "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
