"""32-byte device nodes of finely divided axis-aligned surfaces (host packing): thin, or refused.

Compiles tests/native/node32_planes_check.cpp against trayracer_amd/csrc/bvh_build.cpp with g++
(no contraction, as the kernels are built) and runs it.
"""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parents[1]


def test_node32_planes(tmp_path):
    exe = tmp_path / "node32_planes_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-ffp-contract=off", "-I", str(ROOT / "trayracer_amd" / "csrc"),
                    str(ROOT / "tests" / "native" / "node32_planes_check.cpp"),
                    str(ROOT / "trayracer_amd" / "csrc" / "bvh_build.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr
