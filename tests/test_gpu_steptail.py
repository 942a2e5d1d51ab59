"""Krylov steps whose scalars are computed by the last workgroup of a pass, over
the widths of launch where that is done and where it is not: one workgroup,
fewer than the arrival counters, more, and too many for a tail."""
import numpy as np
import pytest

from oracle import oracle as o
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbits,nocc", [(6, 1), (10, 5), (13, 6), (15, 7), (16, 8), (17, 8)])
@pytest.mark.parametrize("K", [1, 2, 5, 17])
@pytest.mark.parametrize("precision", ["c128", "c128i"])
def test_recurrences_match_the_oracle_and_repeat(nbits, nocc, K, precision):
    """alpha and beta against the oracle's recurrence for the first steps (a step
    adds a few eps of |H|; 6 steps of a random vector stay far from any
    breakdown), and bit for bit the same on a second run."""
    import torch
    from edrixs_amd import core, siam
    rng = np.random.default_rng(nbits * 100 + K)
    ht = siam.emat_terms(H.random_hermitian_emat(nbits, rng))
    ut = siam.umat_terms(np.round(H.random_hermitian_umat(nbits, rng, nnz=12).real, 1) + 0j)
    fock = H.fock_words(nbits, nocc)
    A = core.build_ham_i(core.Basis.combinations(nbits, nocc), ht, ut).prepare(precision)
    R = o.build_ham_i(fock, ht, ut)
    n, steps = R.m, 6 if R.m > 50 else 3
    V = rng.normal(size=(K, n)) + 1j * rng.normal(size=(K, n))
    Vd = torch.from_numpy(V).cuda()
    al, be, nr = core.build_krylov_batch(A, Vd, steps, precision)
    al2, be2, _ = core.build_krylov_batch(A, Vd, steps, precision)
    scale = np.abs(R.vals).sum() / n
    for k in range(K):
        assert np.array_equal(al[k], al2[k]) and np.array_equal(be[k], be2[k])
    for k in {0, K - 1}:
        ra, rb, rn = o.build_krylov(R, V[k], steps)
        tol = 1e4 * 2.3e-16 * scale
        assert np.abs(al[k] - ra).max() <= tol and np.abs(be[k] - rb).max() <= tol
        assert abs(nr[k] - rn) <= 1e-13 * rn
        a1, b1, _ = core.build_krylov(A, Vd[k].contiguous(), steps, precision)
        assert np.abs(a1 - ra).max() <= tol and np.abs(b1 - rb).max() <= tol


@pytest.mark.parametrize("nbits,nocc", [(10, 5), (13, 6), (14, 7), (15, 7), (16, 8)])
@pytest.mark.parametrize("K", [3, 4, 8, 12, 16])
def test_blocks_around_the_widths_of_the_tails(nbits, nocc, K):
    """Four vectors at 640 partials, twelve and sixteen at 900, and more, of the product and
    of the update."""
    test_recurrences_match_the_oracle_and_repeat(nbits, nocc, K, "c128")


@pytest.mark.parametrize("nbath,N", [(1, 5), (4, 7), (5, 8)])
@pytest.mark.parametrize("K", [2, 3, 4])
def test_small_blocks_over_corehole_matrices(nbath, N, K):
    """2,772, 20,592 and 38,610 rows: below and above those the factored product takes."""
    import torch
    from edrixs_amd import core, siam
    m = siam.SiamModel(nbath=nbath, nocc=N - 1, seed=2)
    fn, bn = H.fock_words(m.norb, N), core.Basis.combinations(m.norb, N)
    A = core.build_ham_n(bn, m.norb, m.ncore, m.hop_n, m.coul_n, layout="interleaved").prepare("c128i")
    R = o.build_ham_n(fn, m.norb, m.ncore, m.hop_n, m.coul_n)
    perm = core.corehole_permutation(len(fn), m.ncore)
    rng = np.random.default_rng(nbath + K)
    V = rng.normal(size=(K, R.m)) + 1j * rng.normal(size=(K, R.m))
    al, be, nr = core.build_krylov_batch(A, torch.from_numpy(V[:, perm].copy()).cuda(), 6, "c128i")
    scale = np.abs(R.vals).sum() / R.m
    for k in range(K):
        ra, rb, rn = o.build_krylov(R, V[k], 6)
        tol = 1e4 * 2.3e-16 * scale
        assert np.abs(al[k] - ra).max() <= tol and np.abs(be[k] - rb).max() <= tol
        assert abs(nr[k] - rn) <= 1e-13 * rn
