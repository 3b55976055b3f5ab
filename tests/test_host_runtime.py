"""CPU checks of the library's host code over a stand-in for the HIP runtime
(tests/host_runtime.h): what it does at memory limits and which kernels it
launches."""
from __future__ import annotations

import os
import shutil
import subprocess
from pathlib import Path

import pytest

from polytope_amd.build import LIB

ROOT = Path(__file__).resolve().parents[1]


def run_check(tmp_path, name: str) -> str:
    """Builds tests/<name>.cpp against the library and returns what it prints."""
    rocm = Path("/opt/rocm")
    cxx = shutil.which("g++")
    if not cxx or not (rocm / "include" / "hip").exists():
        pytest.skip("no g++ or HIP headers")
    exe = tmp_path / name
    subprocess.run([cxx, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{rocm / 'include'}",
                    f"-I{ROOT / 'include'}", str(ROOT / "tests" / f"{name}.cpp"), str(LIB), "-o", str(exe),
                    f"-Wl,-rpath,{LIB.parent}", f"-Wl,-rpath-link,{rocm / 'lib'}", "-lpthread"],
                   check=True, capture_output=True, timeout=300)
    env = dict(os.environ, LD_LIBRARY_PATH=f"{rocm / 'lib'}:{os.environ.get('LD_LIBRARY_PATH', '')}")
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300, env=env)
    assert out.returncode == 0, out.stdout + out.stderr
    return out.stdout


def test_scene_creation_at_every_memory_limit(tmp_path):
    assert "\n0 failures" in run_check(tmp_path, "scene_memory_check")


def test_tuning_that_was_got_can_be_set_back(tmp_path):
    assert run_check(tmp_path, "tuning_check") == "0 failures\n"


def test_render_at_memory_limits(tmp_path):
    assert " 0 failures" in run_check(tmp_path, "render_memory_check")


def test_stack_spill_at_memory_limits(tmp_path):
    assert " 0 failures" in run_check(tmp_path, "spill_memory_check")
