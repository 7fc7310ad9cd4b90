"""Every access of the 3-D sweeps stays in its array: a host build of the kernels'
bodies under AddressSanitizer, over ragged grids, segment lengths, runs and walls
(tests/cpp/sweep_bounds.cpp).  LDS starts as NaN, so that a value read before it is
written shows in the result, and integer overflow ends the run."""
import os
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_sweeps_stay_in_their_arrays(tmp_path):
    exe = tmp_path / "sweep_bounds"
    cmd = ["g++", "-std=c++17", "-O0", "-w", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
           "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__", f"-I{ROOT / 'ouxsbli_amd' / 'csrc'}", f"-I{ROOT / 'include'}",
           "-x", "c++", str(ROOT / "tests" / "cpp" / "sweep_bounds.cpp"), "-o", str(exe)]
    subprocess.run(cmd, check=True, capture_output=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_stack_use_after_return=0:detect_leaks=0")
    r = subprocess.run([str(exe), "quick"], capture_output=True, text=True, env=env)
    print(r.stdout[-2000:], r.stderr[-4000:])
    assert r.returncode == 0
    assert "bad=0" in r.stdout
