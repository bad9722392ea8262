"""Plans that the library makes on the host, asked without a GPU (the planners then take 256 compute units)."""
import os
import shutil
import subprocess

import pytest

from llm_metal_amd import lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_plans_of_value_and_residual_rows(tmp_path):
    """Every plan for the large-M kernel, on F16 tiles or on the F16 image of Q8_0 tiles, has the steps and planes that its launch asks for."""
    lib.load()
    exe = tmp_path / "plan_probe"
    r = subprocess.run([HIPCC, "--cuda-host-only", "-std=c++17", "-O1", "-w", "-I", os.path.join(ROOT, "llm_metal_amd", "csrc"),
                        os.path.join(ROOT, "tests", "plan_probe.hip"), "-L" + os.path.dirname(lib.LIB_PATH), "-lllm_metal_hip",
                        "-Wl,-rpath," + os.path.dirname(lib.LIB_PATH), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout[-3000:]
