"""The library's device-memory pool against a stand-in of a device: reuse, its bounds,
what it gives back and when, and several threads at once (tests/pool_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pool_reuse_bounds_and_returns(tmp_path):
    hip = "/opt/rocm/include"
    if not shutil.which("g++") or not os.path.isdir(hip):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path / "pool_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + hip, "-o", exe,
                    os.path.join(ROOT, "tests", "pool_check.cpp"),
                    os.path.join(ROOT, "edrixs_amd", "csrc", "runtime.cpp"), "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "pool ok" in r.stdout, r.stderr


def test_outputs_are_allocated_again_after_a_trim(monkeypatch):
    import torch
    from edrixs_amd import core
    calls, trims = [], []
    zeros = torch.zeros

    def scarce(*a, **k):
        calls.append(a)
        if not trims:
            raise torch.cuda.OutOfMemoryError("no room")
        return zeros(*a, **k)
    monkeypatch.setattr(torch, "zeros", scarce)
    monkeypatch.setattr(core, "mem_trim", lambda: trims.append(1))
    y = core._zeros((2, 3), "cpu")
    assert len(calls) == 2 and len(trims) == 1
    assert y.shape == (2, 3) and y.dtype == torch.complex128
