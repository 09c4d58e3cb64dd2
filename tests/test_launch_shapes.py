"""The host-side arithmetic that launchers and runner share (kernels.h), over its whole range, compiled by g++."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_launch_shapes_hold_over_their_range(tmp_path):
    exe = str(tmp_path / "launch_shapes")
    built = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
                            "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", os.path.join(HERE, "..", "treebeard_amd", "csrc"),
                            os.path.join(HERE, "native", "launch_shapes.cpp"), "-o", exe], capture_output=True, text=True)
    if built.returncode != 0 and ("sanitize" in built.stderr or "hip/hip_runtime" in built.stderr):
        pytest.skip("this g++ has no sanitizer runtime, or the HIP headers are missing")
    assert built.returncode == 0, built.stderr[-3000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and run.stdout.strip().endswith("ok"), (run.stdout + run.stderr)[-4000:]
