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


KERNELS = os.path.join(HERE, "..", "treebeard_amd", "build", "kernels.o")


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists(KERNELS), reason="needs g++ and the built kernels")
def test_launchers_refuse_what_no_kernel_is_built_for(tmp_path):
    exe = str(tmp_path / "launch_refusals")
    built = subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
                            os.path.join(HERE, "..", "treebeard_amd", "csrc"), os.path.join(HERE, "native", "launch_refusals.cpp"), KERNELS,
                            "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-o", exe], capture_output=True, text=True)
    assert built.returncode == 0, built.stderr[-3000:]
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1")        # (nothing of this is meant to reach a device)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60, env=env)
    assert run.returncode == 0 and run.stdout.strip().endswith("ok"), (run.stdout + run.stderr)[-4000:]
