"""The root of the kernel weights, on which the bit equality of every density
rests: equal to sqrtf for every float from 2^-96 to 2^64, and exact weights below
(tests/sqrt_check.hip, built with the library)."""
import pathlib
import subprocess

import pytest

pytestmark = pytest.mark.gpu

EXE = pathlib.Path(__file__).resolve().parents[1] / "bachelor-thesis_amd" / "sqrt_check"


def test_root_equals_sqrtf():
    assert EXE.exists(), "not built (run __graft_entry__.build())"
    print("root against sqrtf, all floats from 2^-96 to 2^64", flush=True)
    out = subprocess.run([str(EXE)], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.split() == ["0", "0"]
