"""The division-free continued fraction against the nested one in extended
precision, at the edges of its blocks, stages and range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("neff", [1, 2, 7, 8, 9, 511, 512, 513, 521, 2500])
@pytest.mark.parametrize("nw,scale", [(1, 1.0), (65, 1.0), (130, 1e-12), (64, 1e12), (64, 1e20),
                                      (64, 1e-20)])
def test_fraction_matches_extended_precision(neff, nw, scale):
    """Rounding is that of coefficients off by a few eps: with T perturbed by dT,
    the fraction norm <1|(z - T)^-1|1> changes by at most norm |dT| / gamma^2,
    |dT| <= c eps (|z - a| + 2 b) with c = 8 for the operations of a step.
    Scales 1e20 and 1e-20 leave the recurrence's range."""
    from edrixs_amd import core
    rng = np.random.default_rng(neff + nw)
    a, b = rng.normal(20.0, 6.0, neff) * scale, np.abs(rng.normal(8.0, 2.0, neff)) * scale
    om, g = np.linspace(-30.0, 50.0, nw) * scale, np.full(nw, 0.4 * scale)
    norm, e, weight = 0.7, 3.0 * scale, 0.6
    start = rng.normal(size=nw) / scale
    got = core.cf_spectrum(a, b, norm, e, om, g, weight=weight, out=start.copy())
    al, bl = a.astype(np.longdouble), b.astype(np.longdouble)
    z = (om.astype(np.longdouble) + e) + 1j * g.astype(np.longdouble)
    t = np.zeros(nw, dtype=np.clongdouble)
    for j in range(neff - 1, 0, -1):
        t = bl[j - 1] ** 2 / (z - al[j] - t)
    ref = start - np.imag(1 / (z - al[0] - t)) * norm * weight / np.pi
    eps = np.finfo(float).eps
    width = np.abs(z[:, None] - al[None, :]).max() + 2 * bl.max()
    tol = weight * norm / np.pi * 8 * eps * width / g[0] ** 2 + 4 * eps * np.abs(ref).max()
    assert np.abs(got - ref).max() <= tol


def test_breakdown_and_zero_couplings():
    """A zero coupling ends the fraction there; the coefficients behind it do not matter."""
    from edrixs_amd import core
    om = np.linspace(-5.0, 5.0, 70)
    a, b = np.array([1.0, -2.0, 0.5, 9.0, 4.0]), np.array([0.8, 0.0, 3.0, 2.0, 1.0])
    s = core.cf_spectrum(a, b, 1.0, 0.0, om, 0.3)
    t = core.cf_spectrum(a[:2], b[:2], 1.0, 0.0, om, 0.3)
    np.testing.assert_allclose(s, t, rtol=1e-14)


@pytest.mark.parametrize("neff", [1, 8, 60, 300, 1000, 4000])
@pytest.mark.parametrize("gamma", [1.0, 0.1, 1e-3, 1e-8])
def test_fraction_keeps_its_digits_far_from_the_poles(neff, gamma):
    """Grid points far from the band, where the imaginary part is a small fraction of
    the real one, point by point.  With |z - a| >= 4 b each quotient of neighbours
    D_j / D_{j+1} = z - a - b^2 D_{j+2} / D_{j+1} carries a rounding of at most 5 eps
    (the error of the one before comes in with weight b^2 / |w|^2 < 1/12), so does
    P_j / |D_{j+1}|^2 = -gamma + b^2 P_{j+1} / |D_{j+1}|^2 with at most 6, and the final
    quotient and prefactors add 2 * 5 + 6: 22 eps, whatever the number of poles."""
    from edrixs_amd import core
    rng = np.random.default_rng(neff)
    a, b = rng.uniform(-4.0, 4.0, neff), rng.uniform(4.0, 8.0, neff)
    om = np.concatenate([np.linspace(-400.0, -36.0, 70), np.linspace(36.0, 120.0, 70),
                         np.geomspace(1e3, 1e8, 30)])
    got = core.cf_spectrum(a, b, 0.7, 0.0, om, gamma, weight=0.6)
    al, bl = a.astype(np.longdouble), b.astype(np.longdouble)
    z = om.astype(np.longdouble) + 1j * np.longdouble(gamma)
    t = np.zeros(len(om), dtype=np.clongdouble)
    for j in range(neff - 1, 0, -1):
        t = bl[j - 1] ** 2 / (z - al[j] - t)
    ref = -np.imag(1 / (z - al[0] - t)) * np.longdouble(0.7) * np.longdouble(0.6) / np.longdouble(np.pi)
    assert np.all(got > 0)
    assert np.max(np.abs(got - ref) / ref) <= 22 * np.finfo(float).eps


@pytest.mark.parametrize("tiny", [1e-14, 1e-16, 1e-30, 1e-39, 1e-60, 1e-120])
@pytest.mark.parametrize("neff", [2, 8, 9, 24])
def test_fraction_on_a_pole_with_tiny_broadening_and_couplings(tiny, neff):
    """Poles all at one place, seen from there with broadening and couplings far below
    it, beside ordinary points: every step shrinks the determinants by the
    broadening.  On the pole the fraction is i times b^2 / (gamma + b^2 / (gamma + ...)),
    positive throughout, so each step adds at most 4 eps."""
    from edrixs_amd import core
    a, b = np.full(neff, 10.0), np.full(neff, tiny) * np.linspace(0.5, 2.0, neff)
    om, g = np.array([10.0, 10.0, 12.0]), np.array([tiny, 3 * tiny, 0.5])
    got = core.cf_spectrum(a, b, 1.0, 0.0, om, g)
    al, bl = a.astype(np.longdouble), b.astype(np.longdouble)
    z = om.astype(np.longdouble) + 1j * g.astype(np.longdouble)
    t = np.zeros(3, dtype=np.clongdouble)
    for j in range(neff - 1, 0, -1):
        t = bl[j - 1] ** 2 / (z - al[j] - t)
    ref = -np.imag(1 / (z - al[0] - t)) / np.longdouble(np.pi)
    assert np.max(np.abs(got - ref) / ref) <= (4 * neff + 8) * np.finfo(float).eps


@pytest.mark.parametrize("nw", [32765, 32770, 100001])
def test_fraction_on_grids_beyond_the_staging_memory(nw):
    """Around and beyond 1 MB of inputs, with points in and out of the recurrence's range
    side by side; a quotient of three poles in the band adds at most
    8 eps (|z - a| + 2 b) / gamma^2 to a spectrum of order 1 / gamma, as above."""
    from edrixs_amd import core
    a, b = np.array([1.0, -2.0, 0.5]), np.array([0.8, 1.5])
    om, g = np.linspace(-6.0, 6.0, nw), np.full(nw, 0.3)
    g[::1000] = 1e-17
    om[::1000] = 1e3
    start = np.linspace(0.0, 1.0, nw)
    got = core.cf_spectrum(a, np.append(b, 7.0), 1.0, 0.25, om, g, out=start.copy())
    z = (om + 0.25).astype(np.longdouble) + 1j * g.astype(np.longdouble)
    t = b[1] ** 2 / (z - a[2])
    t = b[0] ** 2 / (z - a[1] - t)
    ref = -np.imag(1 / (z - a[0] - t)) / np.longdouble(np.pi)
    eps = np.finfo(float).eps
    assert np.abs(got - (start + ref)).max() <= 8 * eps * (9.0 + 3.0) / 0.3 ** 2 / np.pi + 2 * eps
    far = core.cf_spectrum(a, np.append(b, 7.0), 1.0, 0.25, om, g)[::1000]
    assert np.max(np.abs(far - ref[::1000]) / ref[::1000]) <= 32 * eps
