"""CSR builds over the term plan at the edges of its range, against the oracle
(values equal, not close): workgroup remainders, 32- and 64-bit words, both core-hole layouts,
columns that ignore the core word, and the calls that keep the term-by-term
build (incomplete bases, rows longer than the plan's lists, many terms)."""
import numpy as np
import pytest

from edrixs_amd import siam
from oracle import oracle as o
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def core():
    from edrixs_amd import core as c
    return c


def _same(A, R, perm_rows=None, perm_cols=None):
    """Row pointers, columns and values of A equal the oracle's (rows and
    columns permuted by perm: new index i holds old index perm[i])."""
    rp, cols, vals = A.download()
    ref_rp, ref_c, ref_v = (np.asarray(x) for x in (R.rowptr, R.cols, R.vals))
    if perm_rows is not None or perm_cols is not None:
        pr = np.arange(len(ref_rp) - 1) if perm_rows is None else perm_rows
        inv = None
        if perm_cols is not None:
            inv = np.empty(len(perm_cols), dtype=np.int64)
            inv[perm_cols] = np.arange(len(perm_cols))
        oc, ov, orp = [], [], [0]
        for r in pr:
            c, v = ref_c[ref_rp[r]:ref_rp[r + 1]], ref_v[ref_rp[r]:ref_rp[r + 1]]
            if inv is not None:
                c = inv[c]
                k = np.argsort(c, kind="stable")
                c, v = c[k], v[k]
            oc.append(c)
            ov.append(v)
            orp.append(orp[-1] + len(c))
        ref_rp, ref_c, ref_v = np.array(orp), np.concatenate(oc), np.concatenate(ov)
    assert np.array_equal(rp, ref_rp)
    assert np.array_equal(cols, ref_c)
    assert np.array_equal(vals, ref_v)


def _terms(n, seed, nnz_u, density=0.5):
    rng = np.random.default_rng(seed)
    return (siam.emat_terms(H.random_hermitian_emat(n, rng, density=density)),
            siam.umat_terms(H.random_hermitian_umat(n, rng, nnz=nnz_u)))


@pytest.mark.parametrize("nbits,nocc", [(1, 0), (1, 1), (5, 5), (6, 1), (8, 4), (12, 6), (31, 2),
                                        (32, 2), (33, 2), (40, 1), (62, 1),
                                        (11, 5), (15, 12), (31, 3), (32, 3), (33, 3)])
def test_plain_builds_at_word_and_workgroup_edges(core, nbits, nocc):
    ht, ut = _terms(min(nbits, 14), nbits, 60)
    if nbits > 14:       # spread the orbitals over the whole word
        step = (nbits - 1) // 13
        for f in ("ind1", "ind2"):
            ht[f] = 1 + (ht[f] - 1) * step
        for f in ("ind1", "ind2", "ind3", "ind4"):
            ut[f] = 1 + (ut[f] - 1) * step
    fock = H.fock_words(nbits, nocc)
    b = core.Basis.combinations(nbits, nocc)
    for omega, sign in ((0j, 1.0), (-0.75 + 0.25j, -1.0)):
        _same(core.build_ham_i(b, ht, ut, omega=omega, ham_sign=sign),
              o.build_ham_i(fock, ht, ut, omega=omega, ham_sign=sign))


@pytest.mark.parametrize("nv,nc,nocc", [(7, 6, 3), (10, 2, 5), (26, 6, 2), (28, 6, 1)])
def test_corehole_operators_in_both_layouts(core, nv, nc, nocc):
    """H_n, absorption and emission operators of random terms over valence and
    core orbitals, core-core ones among them (absorption columns ignore the
    core word, so such terms meet in one column)."""
    ntot = nv + nc
    rng = np.random.default_rng(nv)
    ht, ut = _terms(ntot, 5, 200, density=0.4)
    tr = siam.emat_terms(rng.normal(size=(ntot, ntot)) * (rng.random((ntot, ntot)) < 0.3))
    fi, fn = H.fock_words(nv, nocc), H.fock_words(nv, nocc + 1)
    bi, bn = core.Basis.combinations(nv, nocc), core.Basis.combinations(nv, nocc + 1)
    perm = core.corehole_permutation(len(fn), nc)
    for lay, p in (("reference", None), ("interleaved", perm)):
        for omega, sign in ((0j, 1.0), (1.5 + 0.5j, -1.0)):
            A = core.build_ham_n(bn, nv, nc, ht, ut, omega=omega, ham_sign=sign, layout=lay)
            _same(A, o.build_ham_n(fn, nv, nc, ht, ut, omega=omega, ham_sign=sign), p, p)
        _same(core.build_transop_i(bn, bi, nv, nc, tr, layout=lay),
              o.build_transop_i(fn, fi, nv, nc, tr), p, None)
        _same(core.build_transop_f(bi, bn, nv, nc, tr, layout=lay),
              o.build_transop_f(fi, fn, nv, nc, tr), None, p)


def test_terms_outside_the_words_and_impossible_terms(core):
    """Orbitals no row has, an orbital taken out or put in twice, spectators, and
    duplicates that cancel to an explicit zero."""
    fock = H.fock_words(6, 3)
    b = core.Basis.combinations(6, 3)
    hop = [[1, 9, 1.0, 0.0], [9, 9, 2.0, 0.0], [2, 2, -0.0, 0.0], [1, 2, 0.5, 1.0],
           [1, 2, -0.5, -1.0], [40, 1, 3.0, 0.0]]
    coul = [[1, 1, 2, 3, 1.0, 0.0], [1, 2, 4, 4, 1.0, 0.0], [1, 2, 2, 1, 0.25, 0.0],
            [1, 2, 1, 2, 0.25, -0.0], [3, 1, 1, 5, 0.75, 0.1], [1, 3, 5, 1, 0.75, 0.1],
            [2, 33, 33, 2, 1.0, 0.0]]
    for sign in (1.0, -1.0):
        _same(core.build_ham_i(b, hop, coul, omega=0.5j, ham_sign=sign),
              o.build_ham_i(fock, hop, coul, omega=0.5j, ham_sign=sign))
    _same(core.build_ham_i(b, None, None), o.build_ham_i(fock, None, None))


@pytest.mark.parametrize("case", ["incomplete", "long_rows", "many_terms"])
def test_builds_that_keep_the_term_by_term_kernel(core, case):
    if case == "long_rows":       # more than 255 entries in a row
        n, N = 16, 8
        ht, ut = _terms(n, 3, 2000, density=1.0)
        assert len(ht) + len(ut) <= 4096
    elif case == "many_terms":    # more than 4096 terms, fewer than 4096 survivors
        n, N = 10, 2
        ht, ut = _terms(n, 4, 4200, density=1.0)
        ut = np.concatenate([ut, ut])
    else:
        n, N = 9, 4
        ht, ut = _terms(n, 5, 80)
    fock = H.fock_words(n, N)
    if case == "incomplete":
        fock = fock[1::2].copy()
    R = o.build_ham_i(fock, ht, ut)
    if case == "long_rows":
        assert np.diff(R.rowptr).max() > 255
    if case == "many_terms":
        assert len(ht) + len(ut) > 4096
    _same(core.build_ham_i(core.Basis.from_words(fock, n), ht, ut), R)


@pytest.mark.parametrize("space,nv,nocc", [("i", 6, 1), ("i", 8, 4), ("i", 33, 2), ("i", 16, 8),
                                           ("i", 18, 9), ("n", 7, 3), ("n", 28, 1), ("n", 13, 6),
                                           ("n", 15, 7)])
def test_matrix_free_apply_at_word_and_workgroup_edges(core, space, nv, nocc):
    """y += H x from the term plan against the oracle's product.  Both add the
    same products in another order (the plan also adds equal terms' values
    first): each row of n entries of T terms in all differs by at most
    (n + T) eps times the sum of |value| |x|, bounded here through the longest
    row and the largest term."""
    import torch
    nc = 6 if space == "n" else 0
    rng = np.random.default_rng(nv)
    ht, ut = _terms(min(nv + nc, 16), 7, 250)
    if nv + nc > 16:
        step = (nv + nc - 1) // 15
        for t, fs in ((ht, ("ind1", "ind2")), (ut, ("ind1", "ind2", "ind3", "ind4"))):
            for f in fs:
                t[f] = 1 + (t[f] - 1) * step
    fock = H.fock_words(nv, nocc)
    b = core.Basis.combinations(nv, nocc)
    for omega, sign in ((0j, 1.0), (0.5 - 0.25j, -1.0)):
        if space == "i":
            op = core.mf_ham_i(b, ht, ut, omega=omega, ham_sign=sign)
            R = o.build_ham_i(fock, ht, ut, omega=omega, ham_sign=sign)
        else:
            op = core.mf_ham_n(b, nv, nc, ht, ut, omega=omega, ham_sign=sign)
            R = o.build_ham_n(fock, nv, nc, ht, ut, omega=omega, ham_sign=sign)
        x = rng.normal(size=R.m) + 1j * rng.normal(size=R.m)
        y0 = rng.normal(size=R.m) + 1j * rng.normal(size=R.m)
        dev = [torch.from_numpy(v).cuda() for v in (x, y0)]
        y = op.apply(*dev).cpu().numpy()
        ref = o.matvec(R, x, y0)
        T = len(ht) + len(ut) + 1
        big = max(np.abs(ht["re"] + 1j * ht["im"]).max(), np.abs(ut["re"] + 1j * ut["im"]).max(),
                  abs(omega), 1.0)
        assert np.abs(y - ref).max() <= 2 * T * 2.3e-16 * T * big * np.abs(x).max()
        again = op.apply(dev[0], torch.from_numpy(y0).cuda()).cpu().numpy()
        assert np.array_equal(y, again)


@pytest.mark.parametrize("nbits,nocc,sets,sign", [(7, 3, 40, 1.0), (10, 5, 90, -1.0),
                                                  (12, 6, 700, 1.0), (12, 6, 700, -1.0)])
def test_merged_terms_keep_every_bit(core, nbits, nocc, sets, sign):
    """Terms in all orders of their operators, with equal, opposite, unrelated and
    zero values: the entries are the oracle's sums in term order, signs of zeros
    included.  700 sets make rows of more than 64 entries and more than 256 groups."""
    rng = np.random.default_rng(nbits + sets)
    u = np.zeros((nbits,) * 4, dtype=np.complex128)
    for q in range(sets):
        i, j, k, l = rng.integers(0, nbits, size=4)
        if i == j or k == l:
            continue
        v = [0.5, -1.25, rng.normal(), 1j * rng.normal(), rng.normal() + 1j * rng.normal()][q % 5]
        orders = [(i, j, k, l), (j, i, k, l), (i, j, l, k), (j, i, l, k)]
        rel = [(1, -1, -1, 1), (1, 1, 1, 1), (1, -1, 1, -1), (1, 0, 0, 1), (1, 0.3, -0.7, 1)][q % 4 + (q % 7 == 0)]
        for o4, r in zip(orders, rel):
            u[o4] += r * v
            u[o4[::-1]] += r * np.conj(v)
    ht, ut = siam.emat_terms(H.random_hermitian_emat(nbits, rng, density=0.5)), siam.umat_terms(u)
    ut["re"][::9] *= 0.0
    ut["im"][::4] = -0.0
    A = core.build_ham_i(core.Basis.combinations(nbits, nocc), ht, ut, omega=-0.0 + 0.5j, ham_sign=sign)
    R = o.build_ham_i(H.fock_words(nbits, nocc), ht, ut, omega=-0.0 + 0.5j, ham_sign=sign)
    if sets == 700:
        assert 64 < np.diff(R.rowptr).max() <= 255
    rp, cols, vals = A.download()
    assert np.array_equal(rp, np.asarray(R.rowptr)) and np.array_equal(cols, np.asarray(R.cols))
    ref = np.ascontiguousarray(R.vals).view(np.float64)
    got = np.ascontiguousarray(vals).view(np.float64)
    assert np.array_equal(got, ref) and np.array_equal(np.signbit(got), np.signbit(ref))


def _few_terms(n, seed, most=56):
    """At most `most` terms over n orbitals spread from the first to the last: hoppings, densities,
    two-body terms and their conjugates."""
    rng = np.random.default_rng(seed)
    k = min(n, 9)
    orb = np.unique(np.linspace(0, n - 1, k).round().astype(int))
    hop = [[i + 1, j + 1, *rng.normal(size=2)] for i in orb for j in orb if rng.random() < 0.3]
    coul = []
    for _ in range(most):
        i, j, p, q = rng.choice(orb, size=4)
        if i == j or p == q:
            continue
        re, im = rng.normal(size=2)
        coul += [[i + 1, j + 1, p + 1, q + 1, re, im], [q + 1, p + 1, j + 1, i + 1, re, -im]]
    hop = hop[:most // 2]
    return hop, coul[:most - len(hop)]


def _rule(source, pattern):
    """The numbers of a rule of the library, read from its source: a test that means one
    route fails when the line moves past its sizes."""
    import os
    import re
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src = open(os.path.join(root, "edrixs_amd", "csrc", source)).read()
    return [float(x) for x in re.search(pattern, src).groups()]


def _build_max_groups(M, T):
    a, r, t, u, g = _rule("csr_build.hip", r"const double g = \(([\d.e-]+) \+ M \* \(([\d.e-]+) \+ ([\d.e-]+) \* T\)"
                                           r" - ([\d.e-]+) \* T\) / ([\d.e-]+);")
    most = (a + M * (r + t * T) - u * T) / g
    return most if 16 * most >= T else -1


def _mf_max_groups(M, T):
    r, t, u, a, g = _rule("mf.hip", r"const double g = \(M \* \(([\d.e-]+) \+ ([\d.e-]+) \* T\) \+ ([\d.e-]+) \* T"
                                    r" - ([\d.e-]+)\) / ([\d.e-]+);")
    most = (M * (r + t * T) + u * T - a) / g
    return most if 16 * most >= T else -1


def _groups_and_mean_row(n, N, ht, ut):
    """Groups of the terms, and the rule's measure of a mean row: the largest share of the
    C(n, N) rows that a term of each group survives on."""
    from math import comb
    share = {}
    for t in list(ht) + list(ut):
        ops = [int(t[f]) - 1 for f in ("ind1", "ind2", "ind3", "ind4") if f in t.dtype.names]
        out, into = ops[:len(ops) // 2], ops[len(ops) // 2:]
        if len(set(out)) < len(out) or len(set(into)) < len(into):
            continue
        full, empty = len(out), len(set(into) - set(out))
        key = sum(1 << q for q in set(out) ^ set(into))
        share[key] = max(share.get(key, 0.0), comb(n - full - empty, N - full) / comb(n, N))
    return len(share), sum(share.values())


def test_calls_of_few_terms_take_the_plan_on_any_number_of_rows():
    """The sizes below count on it."""
    assert _build_max_groups(0, 56) >= 56          # 56 terms in 56 groups, no rows


@pytest.mark.parametrize("nbits,nocc", [(1, 0), (1, 1), (5, 5), (6, 1), (8, 4), (11, 5), (15, 12),
                                        (31, 2), (32, 2), (33, 2), (40, 1), (62, 1), (62, 2)])
def test_few_terms_at_word_and_workgroup_edges(core, nbits, nocc):
    ht, ut = _few_terms(nbits, nbits + nocc)
    b, fock = core.Basis.combinations(nbits, nocc), H.fock_words(nbits, nocc)
    for omega, sign in ((0j, 1.0), (-0.75 + 0.25j, -1.0)):
        _same(core.build_ham_i(b, ht, ut, omega=omega, ham_sign=sign),
              o.build_ham_i(fock, ht, ut, omega=omega, ham_sign=sign))


@pytest.mark.parametrize("nv,nc,nocc", [(1, 1, 0), (7, 6, 3), (10, 2, 5), (26, 6, 2), (27, 6, 1), (40, 6, 1)])
def test_few_corehole_terms_in_both_layouts(core, nv, nc, nocc):
    ht, ut = _few_terms(nv + nc, nv)
    tr = _few_terms(nv + nc, nv + 1)[0]
    fi, fn = H.fock_words(nv, nocc), H.fock_words(nv, nocc + 1)
    bi, bn = core.Basis.combinations(nv, nocc), core.Basis.combinations(nv, nocc + 1)
    perm = core.corehole_permutation(len(fn), nc)
    for lay, p in (("reference", None), ("interleaved", perm)):
        for omega, sign in ((0j, 1.0), (1.5 + 0.5j, -1.0)):
            _same(core.build_ham_n(bn, nv, nc, ht, ut, omega=omega, ham_sign=sign, layout=lay),
                  o.build_ham_n(fn, nv, nc, ht, ut, omega=omega, ham_sign=sign), p, p)
        _same(core.build_transop_i(bn, bi, nv, nc, tr, layout=lay),
              o.build_transop_i(fn, fi, nv, nc, tr), p, None)
        _same(core.build_transop_f(bi, bn, nv, nc, tr, layout=lay),
              o.build_transop_f(fi, fn, nv, nc, tr), None, p)


def test_few_terms_on_incomplete_bases(core):
    """Words left out, at the end, at the front and inside: columns are found by search."""
    ht, ut = _few_terms(12, 3)
    fock = H.fock_words(12, 6)
    for part in (fock[:-1], fock[1:], fock[::3], np.delete(fock, 400)):
        part = part.copy()
        _same(core.build_ham_i(core.Basis.from_words(part, 12), ht, ut), o.build_ham_i(part, ht, ut))


def test_a_few_long_rows_among_short_ones(core):
    """Terms on 14 of 20 orbitals: rows with all six electrons there are longer than the
    plan's lists. By the largest share of rows that a term of each group survives on, the mean
    row has 61 entries, so the plan's count is what finds them."""
    ht, ut = _terms(14, 3, 4000, density=1.0)
    ut = ut[:4090 - len(ht)]
    fock = H.fock_words(20, 6)
    R = o.build_ham_i(fock, ht, ut)
    assert np.diff(R.rowptr).max() > 255
    groups, mean = _groups_and_mean_row(20, 6, ht, ut)
    assert _build_max_groups(R.m, len(ht) + len(ut)) >= groups
    assert mean <= _rule("csr_build.hip", r"BUILD_MEAN_ROW = ([\d.]+);")[0]
    _same(core.build_ham_i(core.Basis.combinations(20, 6), ht, ut), R)


@pytest.mark.parametrize("space,nv,nocc", [("i", 33, 4), ("i", 40, 3), ("i", 24, 4), ("n", 26, 2), ("n", 36, 2)])
def test_matrix_free_apply_of_few_terms_on_many_rows(core, space, nv, nocc):
    """Hoppings and densities of one sign, so no sum cancels: row by row within
    (entries + terms on the diagonal + 4) eps of sum |value| |x|, in 32- and 64-bit
    words, by four and by sixteen waves."""
    import torch
    nc = 6 if space == "n" else 0
    rng = np.random.default_rng(nv)
    k = nv + nc
    orb = np.unique(np.linspace(0, k - 1, 7).round().astype(int))
    ht = [[i + 1, j + 1, *rng.normal(size=2)] for i in orb for j in orb if i < j]
    ht += [[j, i, re, -im] for i, j, re, im in ht]
    ut = [[i + 1, j + 1, j + 1, i + 1, -rng.uniform(0.5, 2.0), 0.0] for i in orb for j in orb if i < j][:14]
    N = nocc + (space == "n")
    fock, b = H.fock_words(nv, N), core.Basis.combinations(nv, N)
    if space == "i":
        op, R = core.mf_ham_i(b, ht, ut), o.build_ham_i(fock, ht, ut)
    else:
        op, R = core.mf_ham_n(b, nv, nc, ht, ut), o.build_ham_n(fock, nv, nc, ht, ut)
    assert _mf_max_groups(R.m, len(ht) + len(ut)) >= 43      # 42 hoppings and the diagonal
    x = rng.normal(size=R.m) + 1j * rng.normal(size=R.m)
    y0 = rng.normal(size=R.m) + 1j * rng.normal(size=R.m)
    y = op.apply(torch.from_numpy(x).cuda(), torch.from_numpy(y0).cuda()).cpu().numpy()
    rp, c, v = (np.asarray(q) for q in (R.rowptr, R.cols, R.vals))
    size = np.zeros(R.m)
    rows = np.repeat(np.arange(R.m), np.diff(rp))
    np.add.at(size, rows, 2.0 * np.abs(v) * np.abs(x[c]))
    size += np.abs(y0)
    eps = np.finfo(float).eps
    assert np.all(np.abs(y - o.matvec(R, x, y0)) <= (np.diff(rp) + 14 + 4) * eps * size)


@pytest.mark.parametrize("im", [0.0, -0.0])
@pytest.mark.parametrize("order", [0, 1])
def test_rows_with_omega_alone_on_the_diagonal_keep_its_bits(core, im, order):
    """More than 24 density terms, none of which survives on rows without a pair of
    electrons among the first nine orbitals: there the entry is omega itself, signs of
    zeros included."""
    nbits, nocc = 16, 4
    pairs = [(i, j) for i in range(1, 10) for j in range(i + 1, 10)][:30]
    coul = [[i, j, j, i, 0.5, im] if order else [i, j, i, j, 0.5, im] for i, j in pairs]
    omega = complex(0.25, -0.0)
    A = core.build_ham_i(core.Basis.combinations(nbits, nocc), None, coul, omega=omega, ham_sign=-1.0)
    R = o.build_ham_i(H.fock_words(nbits, nocc), None, coul, omega=omega, ham_sign=-1.0)
    rp, cols, vals = A.download()
    ref, got = (np.ascontiguousarray(v).view(np.float64) for v in (R.vals, vals))
    assert np.array_equal(rp, np.asarray(R.rowptr)) and np.array_equal(cols, np.asarray(R.cols))
    assert np.sum(np.asarray(R.vals) == omega) > 20
    assert np.array_equal(got, ref) and np.array_equal(np.signbit(got), np.signbit(ref))


@pytest.mark.parametrize("nbits,nocc,sets,density,sign", [(16, 8, 300, 0.5, 1.0), (16, 8, 300, 0.5, -1.0),
                                                          (14, 7, 40, 0.1, -1.0), (14, 7, 40, 0.1, 1.0)])
def test_merged_terms_keep_every_bit_over_the_plan(core, nbits, nocc, sets, density, sign):
    """Terms in all orders of their operators, as above, on enough rows for the plan: with
    rows of more than 64 entries and more than 256 groups, and with short ones."""
    rng = np.random.default_rng(nbits + sets)
    u = np.zeros((nbits,) * 4, dtype=np.complex128)
    for q in range(sets):
        i, j, k, l = rng.integers(0, nbits, size=4)
        if i == j or k == l:
            continue
        v = [0.5, -1.25, rng.normal(), 1j * rng.normal(), rng.normal() + 1j * rng.normal()][q % 5]
        rel = [(1, -1, -1, 1), (1, 1, 1, 1), (1, -1, 1, -1), (1, 0, 0, 1), (1, 0.3, -0.7, 1)][q % 4 + (q % 7 == 0)]
        for o4, r in zip([(i, j, k, l), (j, i, k, l), (i, j, l, k), (j, i, l, k)], rel):
            u[o4] += r * v
            u[o4[::-1]] += r * np.conj(v)
    ht = siam.emat_terms(H.random_hermitian_emat(nbits, rng, density=density))
    ut = siam.umat_terms(u)
    ut["re"][::9] *= 0.0
    ut["im"][::4] = -0.0
    R = o.build_ham_i(H.fock_words(nbits, nocc), ht, ut, omega=-0.0 + 0.5j, ham_sign=sign)
    groups, mean = _groups_and_mean_row(nbits, nocc, ht, ut)
    assert _build_max_groups(R.m, len(ht) + len(ut)) >= groups + 1
    assert mean <= _rule("csr_build.hip", r"BUILD_MEAN_ROW = ([\d.]+);")[0]
    if sets == 300:
        assert 64 < np.diff(R.rowptr).max() <= 255 and groups > 256
    A = core.build_ham_i(core.Basis.combinations(nbits, nocc), ht, ut, omega=-0.0 + 0.5j, ham_sign=sign)
    rp, cols, vals = A.download()
    assert np.array_equal(rp, np.asarray(R.rowptr)) and np.array_equal(cols, np.asarray(R.cols))
    ref = np.ascontiguousarray(R.vals).view(np.float64)
    got = np.ascontiguousarray(vals).view(np.float64)
    assert np.array_equal(got, ref) and np.array_equal(np.signbit(got), np.signbit(ref))
