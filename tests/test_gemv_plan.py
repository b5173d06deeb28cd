"""The run-time slicing of the decode GEMV for any K (host code): compiled by
itself and run over problems."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_any_plan(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    exe = tmp_path / "gemv_plan"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", os.path.join(ROOT, "cuda-llm-inference-engine_amd", "csrc"),
                    os.path.join(ROOT, "tests", "gemv_plan.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
