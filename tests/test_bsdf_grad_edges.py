"""The adjoint's BSDF derivatives at clamped roughness and grazing directions, against 64-bit
ones and the dual numbers: in the mean and in the worst case.

Compiles tests/native/bsdf_grad_edges_check.cpp with the oracle's flags (no contraction) and
runs it.
"""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parents[1]


def test_bsdf_grad_edges(tmp_path):
    exe = tmp_path / "bsdf_grad_edges_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fno-fast-math", "-I",
                    str(ROOT / "trayracer_amd" / "csrc"), str(ROOT / "tests" / "native" / "bsdf_grad_edges_check.cpp"),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.rstrip().endswith("ok"), out.stdout + out.stderr
