"""Packing 32-byte nodes where threads run out.

Compiles tests/native/node32_threads_check.cpp against trayracer_amd/csrc/bvh_build.cpp with g++
and runs it.
"""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parents[1]


def test_no_more_threads(tmp_path):
    exe = tmp_path / "node32_threads_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", str(ROOT / "trayracer_amd" / "csrc"),
                    str(ROOT / "tests" / "native" / "node32_threads_check.cpp"),
                    str(ROOT / "trayracer_amd" / "csrc" / "bvh_build.cpp"), "-o", str(exe), "-ldl"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr
