"""Address limits of the denoiser's kernels (host code): what forward takes, backward takes.

Compiles tests/native/dn_limits_check.cpp with g++ and runs it.
"""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parents[1]


def test_limits(tmp_path):
    exe = tmp_path / "dn_limits_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", str(ROOT / "trayracer_amd" / "csrc"),
                    str(ROOT / "tests" / "native" / "dn_limits_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr
    assert int(out.stdout.split()[1]) >= 8064
