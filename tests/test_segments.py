"""Blocks of any grid share the segments of a list without gaps, repeats or endless loops.

Compiles tests/native/segments_check.cpp with g++ and runs it.
"""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parents[1]


def test_segments(tmp_path):
    exe = tmp_path / "segments_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", str(ROOT / "trayracer_amd" / "csrc"),
                    str(ROOT / "tests" / "native" / "segments_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr
