"""Launches of any length: the host build of the kernels' tile deal (ox_xcd.hpp)
takes every tile once and stays below HIP's 2^32 work items in a dimension, at
lengths around its chunk, its line for few workgroups and its fold."""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_launch_grid_and_deal(tmp_path):
    exe = tmp_path / "launch_grid"
    cmd = ["g++", "-std=c++17", "-O2", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__", "-x", "c++",
           str(ROOT / "tests" / "cpp" / "launch_grid.cpp"), "-o", str(exe)]
    subprocess.run(cmd, check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert "launch grids ok" in r.stdout
