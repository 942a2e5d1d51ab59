"""The no-allocation Krylov entry point against edx_build_krylov.

edx_build_krylov_noalloc runs the same recurrence with its device memory in
the library's static scratch array, so on a prepared matrix it must return
the same (alpha, beta, norm) bit for bit.  Two calls in a row, the second on
a smaller input (the array keeps the first call's contents), then a request
beyond the array's size, which must fail with a clear error.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _krylov(core, entry, H, precision, v0, maxn):
    alpha = np.zeros(maxn)
    beta = np.zeros(maxn)
    neff = ctypes.c_int()
    norm = ctypes.c_double()
    core._lib.call(entry, H._h, core._prec(precision), core._dptr(v0), maxn, ctypes.byref(neff),
                   core._ptr(alpha), core._ptr(beta), ctypes.byref(norm))
    n = neff.value
    return alpha[:n], beta[:n], norm.value


def test_noalloc_krylov_equals_allocating_entry_point():
    import torch
    from edrixs_amd import core, siam
    from tests import helpers as H
    cases = [(6, "c128i", 300), (4, "c128", 120)]     # norb 16 then norb 14: smaller
    for nbath, precision, maxn in cases:
        m = H.small_siam(nbath=nbath, seed=5)
        bn = core.Basis.combinations(m.norb, m.nocc + 1)
        Hn = core.build_ham_n(bn, m.norb, m.ncore, m.hop_n, m.coul_n, layout="interleaved")
        Hn.prepare(precision)
        g = torch.Generator(device="cuda").manual_seed(nbath)
        v0 = torch.randn(Hn.n, dtype=torch.complex128, device="cuda", generator=g)
        used = core.mem_in_use()
        a1, b1, n1 = _krylov(core, "edx_build_krylov_noalloc", Hn, precision, v0, maxn)
        assert core.mem_in_use() == used          # no device allocation by the library
        a2, b2, n2 = _krylov(core, "edx_build_krylov", Hn, precision, v0, maxn)
        assert len(a1) == len(a2) == maxn
        assert np.array_equal(a1, a2) and np.array_equal(b1, b2) and n1 == n2
    # an unprepared form is refused (preparing it would allocate)
    m = H.small_siam(nbath=2, seed=5)
    bn = core.Basis.combinations(m.norb, m.nocc + 1)
    Hn = core.build_ham_n(bn, m.norb, m.ncore, m.hop_n, m.coul_n)
    v0 = torch.ones(Hn.n, dtype=torch.complex128, device="cuda")
    with pytest.raises(Exception, match="not prepared"):
        _krylov(core, "edx_build_krylov_noalloc", Hn, "c64d", v0, 10)
    # more than the static array holds: a clear error, nothing run
    with pytest.raises(Exception, match="bytes of scratch"):
        _krylov(core, "edx_build_krylov_noalloc", Hn, "c128", v0, 1 << 23)


def test_noalloc_krylov_up_to_the_size_of_its_scratch():
    """64 MB of vectors, partials, state, history and flags run; 256 bytes more are refused.
    The bytes a run needs are read from the message of a refused one; the step tails'
    counters in it (33 of 128 bytes) come on top of the 64 MB."""
    import re
    import torch
    from edrixs_amd import core
    from tests import helpers as H
    hop = [[i, i % 6 + 1, 0.5, 0.0] for i in range(1, 7)] + [[i % 6 + 1, i, 0.5, 0.0] for i in range(1, 7)]
    A = core.build_ham_i(core.Basis.combinations(6, 3), hop, None)
    v0 = torch.ones(A.n, dtype=torch.complex128, device="cuda")
    counters = 33 * 128 + 128

    def need(maxn):
        with pytest.raises(Exception, match="bytes of scratch") as err:
            _krylov(core, "edx_build_krylov_noalloc", A, "c128", v0, maxn)
        return int(re.search(r"needs (\d+) bytes", str(err.value)).group(1)) - counters
    lo, hi = 1, 1 << 22
    assert need(hi) > 64 << 20
    fixed = need(hi) - (-(-(2 * hi + 2) * 8 // 256) * 256 + -(-(hi + 2) * 4 // 256) * 256)
    def size(maxn):
        return fixed + -(-(2 * maxn + 2) * 8 // 256) * 256 + -(-(maxn + 2) * 4 // 256) * 256
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if size(mid) <= 64 << 20 else (lo, mid)
    assert size(lo) <= 64 << 20 < size(lo + 1)
    assert need(lo + 1) == size(lo + 1)
    a, b, nrm = _krylov(core, "edx_build_krylov_noalloc", A, "c128", v0, lo)
    a2, b2, nrm2 = _krylov(core, "edx_build_krylov", A, "c128", v0, 64)
    k = len(a2)
    assert len(a) >= k > 0 and nrm == nrm2
    assert np.array_equal(a[:k], a2) and np.array_equal(b[:k], b2)
