"""Products of blocks of vectors larger than the last-level cache, which walk the
rows in parts: a batched recurrence against one vector at a time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("space,norb,nocc,K", [("n", 23, 11, 3), ("i", 22, 11, 24), ("i", 23, 9, 21)])
def test_large_block_recurrence_is_the_single_one(space, norb, nocc, K):
    """alpha and beta are sums over n rows of products summed over a row: two
    orders differ by a few sqrt(n) eps of |H| at most, and a second step carries
    that on once."""
    import torch
    from edrixs_amd import core, siam
    m = siam.SiamModel(nbath=norb - 10, nocc=nocc, seed=4)
    if space == "i":
        b = core.Basis.combinations(norb, nocc)
        H = core.build_ham_i(b, m.hop_i, m.coul_i)
    else:
        b = core.Basis.combinations(norb, nocc + 1)
        H = core.build_ham_n(b, m.norb, m.ncore, m.hop_n, m.coul_n, layout="interleaved")
    H.prepare("c128i")
    assert H.n * K * 16 > 256 << 20
    g = torch.Generator(device="cuda").manual_seed(7)
    V = torch.randn((K, H.n), dtype=torch.complex128, device="cuda", generator=g)
    kb = core.KrylovBatch(H, V, "c128i", capacity=2)
    kb.advance(2)
    a, be, nrm = kb.coefficients()
    kb.close()
    for k in (0, 1, K // 2, K - 1):
        a1, b1, n1 = core.build_krylov(H, V[k].contiguous(), 2, "c128")
        scale = max(np.abs(a1).max(), np.abs(b1).max())
        tol = 50 * np.sqrt(H.n) * 2.3e-16 * scale
        assert np.abs(np.asarray(a[k]) - a1).max() <= tol
        assert np.abs(np.asarray(be[k])[:1] - b1[:1]).max() <= tol
