"""Batched plans when a launch or an allocation fails, and what outlives them, on the CPU: cuszp_batch.cpp
built with a HIP runtime and launches of host memory (tests/host/batch_plan.cpp)."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "cuszp_amd"))

import build as B  # noqa: E402


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not os.path.exists(B.HIPCC) or not shutil.which("g++"):
        pytest.skip("no compiler")
    d = tmp_path_factory.mktemp("host")
    obj, exe = str(d / "batch_plan.o"), str(d / "batch_plan")
    src = os.path.join(ROOT, "tests", "host", "batch_plan.cpp")
    subprocess.run([B.HIPCC, "-x", "hip", f"--offload-arch={B.ARCH}", "--cuda-host-only", "-std=c++17", "-O1", "-fPIC", "-w", "-c", src, "-o", obj],
                   check=True)
    subprocess.run(["g++", obj, "-o", exe, "-lpthread"], check=True)   # without the HIP runtime
    return exe


@pytest.mark.parametrize("case", ["epoch", "words", "tune", "tune graph", "tune-lost", "tune-lost graph"])
def test_plan(program, case):
    r = subprocess.run([program, *case.split()], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
