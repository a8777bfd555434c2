"""Contexts without pinned host memory: tests/native/no_pinned_check.cpp, a C++ program in which
hipHostMalloc fails, renders, reads and traces as one in which it does not."""
import pathlib
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
SCENE = ROOT / "tests" / "golden" / "scenes" / "box_scene.json"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp("no_pinned") / "no_pinned_check"
    lib = ROOT / "trayracer_amd"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", str(ROOT / "include"),
                    str(ROOT / "tests" / "native" / "no_pinned_check.cpp"), "-L", str(lib), "-ltrt", "-ldl",
                    f"-Wl,-rpath,{lib}", "-o", str(exe)], check=True)
    return exe


def test_program_builds(program):
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is present: covered by the GPU test")
    out = subprocess.run([str(program), str(SCENE)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 2 and out.stdout == "no device\n", out.stdout + out.stderr


@pytest.mark.gpu
def test_everything_works_without_pinned_memory(program):
    out = subprocess.run([str(program), str(SCENE)], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr
    refused, rays = map(int, out.stdout.split()[1:])
    assert refused >= 4 and rays > 500_000  # frame, read and small-query blocks, the frame's again
