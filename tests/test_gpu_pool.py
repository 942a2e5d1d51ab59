"""Device blocks kept for reuse, on the device: what is reported, given back, and reused by
another thread on its own stream."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


def _build(core, m):
    b = core.Basis.combinations(m.norb, m.nocc + 1)
    return core.build_ham_n(b, m.norb, m.ncore, m.hop_n, m.coul_n)


def test_kept_blocks_are_reported_and_given_back():
    import torch
    from edrixs_amd import core
    held = core.Basis.combinations(10, 5)        # something stays alive
    m = H.small_siam(nbath=8, seed=4)
    core.mem_trim()
    assert core.mem_reserved()[1] == 0
    free0 = torch.cuda.mem_get_info()[0]
    A = _build(core, m)
    n = A.nnz
    live, _ = core.mem_reserved()
    assert live >= core.mem_in_use() >= 20 * n
    del A
    live1, idle = core.mem_reserved()
    assert live1 < live and idle >= 20 * n        # kept, and said so
    core.mem_trim()
    assert core.mem_reserved() == (live1, 0)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] >= free0 - (64 << 20)
    assert len(held) == 252


def test_blocks_freed_by_one_thread_serve_another_on_its_own_stream():
    """Builds, products and frees in three threads, each on its own stream: every product is
    the one of a thread alone, bit for bit."""
    import threading
    import torch
    from edrixs_amd import core
    models = [H.small_siam(nbath=4, seed=s) for s in (1, 2, 3)]
    x = torch.randn(6 * H.ncomb(14, models[0].nocc + 1), dtype=torch.complex128, device="cuda")
    ref = [_build(core, m).matvec(x).cpu().numpy() for m in models]
    torch.cuda.synchronize()
    bad = []

    def work(k):
        s = torch.cuda.Stream()
        core.set_stream(s)
        try:
            with torch.cuda.stream(s):
                for i in range(12):
                    q = (k + i) % 3
                    y = _build(core, models[q]).matvec(x).cpu().numpy()
                    if not np.array_equal(y, ref[q]):
                        bad.append((k, i))
        finally:
            core.set_stream(None)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
