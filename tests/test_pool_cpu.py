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


def test_serving_counts_and_returns_kept_blocks(monkeypatch):
    """Blocks the library keeps count against the budget; they go back when they alone keep
    a request out, or when what is held exceeds the budget, and stay otherwise."""
    from edrixs_amd import core, serving
    eng = serving.Engine(budget_gb=10.0, max_wait_s=5.0)
    req = serving.make_requests(1, rate=1.0, sizes=(16,), seed=1)
    need = eng.need_bytes(req[0])
    state = {"idle": 0.0, "live": 0.0, "trims": 0}

    def trim():
        state["idle"] = 0.0
        state["trims"] += 1
    monkeypatch.setattr(core, "mem_trim", trim)
    eng.device_bytes = lambda: state["live"]
    eng.idle_bytes = lambda: state["idle"]

    def decide(live, idle, queue=req, running=1):
        state.update(live=live, idle=idle, trims=0)
        return eng.next_request(queue, running, now=0.0), state["trims"]
    assert decide(0.0, 1e9) == (req[0], 0)                    # both fit
    assert decide(9e9 - need, 2e9) == (req[0], 1)             # only without the kept blocks
    assert decide(10e9 - 0.5 * need, 1e8) == (None, 1)        # not even then
    assert decide(10e9 - 0.5 * need, 0.0) == (None, 0)
    assert decide(9.5e9, 1e9, queue=[]) == (None, 1)          # nobody waits, but too much is held
    assert decide(5e9, 1e9, queue=[]) == (None, 0)
    assert decide(9.9e9, 1e9, running=0) == (req[0], 1)       # alone: admitted, kept blocks back
