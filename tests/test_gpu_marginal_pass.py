"""GPU: the background integral of one channel at a time, about the rule that
accepts its first 61-point pass: windows from narrow to wide, bells whole and
clipped, fractional counts, one bin to more than a wavefront's, few counts to
many; against the incomplete gamma function (one bin, no star: the integrand
is B^D exp(-T B)) and against fixed quadrature in 64 bits
(xpsi/likelihoods/default_background_marginalisation.pyx:450-734)."""
import math

import numpy as np
import pytest
from scipy.special import gammainc, gammaln, roots_legendre

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _channel(T, star, data, sigmas, epsrel=1.0e-8):
    """lnL of one channel whose star counts come as the given background."""
    from xpsi_amd.likelihoods import default_background_marginalisation as G
    n = len(data)
    print("[gpu] marginal: %d bins, %.4g counts, %.3g deviations" % (n, data.sum(), sigmas), flush=True)
    grid = np.linspace(0.0, 1.0, 5)
    out = G.eval_marginal_likelihood(T, np.linspace(0.0, 1.0, n + 1), data[None], (np.zeros((1, 5)),), (grid,),
                                     np.zeros(1), np.zeros(1), np.array([[0.0, -1.0]]), 1000, 0.0, epsrel, 1.0e-3,
                                     sigmas, -1.0e90, slim=-1.0, background=star[None] / n)
    return out[0]


def _tolerance(T, star, data, B, rel):
    """rel of the integral, and the rounding of the exponent's terms
    d log c - c, which the reference's formula takes before their sum (an
    integral of them cannot be better): half an ulp each for c, its logarithm, the
    product and the difference, and the running sum's, two ulp of each term
    in all, and as much again in the normalisation."""
    c = T / len(data) * (star + B)
    return rel + 4.0 * EPS * np.sum(np.abs(data * np.log(c)) + c)


@pytest.mark.parametrize("epsrel", [1.0e-8, 1.0e-12])
@pytest.mark.parametrize("total,sigmas", [(4.6, 30.0), (5.2, 43.0), (6.3, 53.0), (11.5, 73.0), (17.3, 57.0), (4.3, 15.0),
                                          (4.3, 20.0), (27.3, 10.0), (27.3, 12.0), (27.3, 12.5), (3.7, 10.0),
                                          (400.5, 10.0), (400.5, 5.0)])
def test_one_bin_against_gamma(total, sigmas, epsrel):
    T, B = 2.0, total / 2.0
    got = _channel(T, np.zeros(1), np.array([total]), sigmas, epsrel)
    s = B / math.sqrt(total)
    lo, hi = T * max(B - sigmas * s, 0.0), T * (B + sigmas * s)
    ref = gammaln(total + 1.0) + math.log((gammainc(total + 1.0, hi) - gammainc(total + 1.0, lo)) / T)
    # scipy's functions: some 1e-15 of themselves
    assert abs(got - ref) < _tolerance(T, np.zeros(1), np.array([total]), B, min(epsrel, 1e-11)) + 1e-14 * (1.0 + abs(ref))


def _draw(bins, total, fraction, whole, seed):
    rng = np.random.default_rng(seed)
    data = rng.poisson(total / bins, bins).astype(float) if whole else total / bins * np.exp(rng.normal(0.0, 1.0, bins))
    data[0] += 0.0 if data.sum() > 0.0 else 1.0
    star = np.exp(rng.normal(0.0, 2.0, bins))
    return data, star * (fraction * data.sum() / star.sum())


def _reference(T, star, data, sigmas, epsilon=1.0e-3):
    """log of the integral over the kernel's window, as its logarithm form
    relative to the maximum: no terms cancel."""
    n = len(data)
    # counts per bin c = T / n (star + B)
    star = star * n / T
    B = max(data.sum() / T - star.mean(), 0.0)
    for _ in range(100):
        x = np.sum(data / (star + B) ** 2)
        dB = (np.sum(data / (star + B)) - T) / x
        if abs(dB) <= epsilon / math.sqrt(x):
            break
        B += dB
        if B < 0.0:
            B = 0.0
            break
    s = 1.0 / math.sqrt(np.sum(data / (star + B) ** 2))
    lo, hi = max(B - sigmas * s, 0.0), B + sigmas * s
    xk, wk = roots_legendre(40)
    edges = np.linspace(lo, hi, 41)
    b = edges[:-1, None] + np.diff(edges)[:, None] * 0.5 * (xk + 1.0)
    e = np.sum(data * np.log1p((b[..., None] - B) / (star + B)), axis=-1) - T * (b - B)
    c = T / n * (star + B)
    ref = math.log(np.sum(np.exp(e) * wk) * 0.5 * (hi - lo) / 40) + np.sum(data * np.log(c) - c)
    return ref, star, B


@pytest.mark.parametrize("whole", [True, False])
@pytest.mark.parametrize("sigmas", [6.0, 10.0, 11.9, 20.0])
@pytest.mark.parametrize("bins,total,fraction", [(1, 40.0, 0.5), (3, 9.0, 0.3), (32, 30.0, 0.7), (64, 2000.0, 0.9),
                                                 (65, 200.0, 0.05), (130, 3000.0, 0.6), (300, 40000.0, 0.5)])
def test_bins_against_quadrature(bins, total, fraction, sigmas, whole):
    T = 3.0
    data, star = _draw(bins, total, fraction, whole, seed=bins)
    ref, star, B = _reference(T, star, data, sigmas)
    got = _channel(T, star, data, sigmas)
    tol = _tolerance(T, star, data, B, 1e-11)
    print("lnL gpu %.12f reference %.12f: %.1e of %.1e" % (got, ref, abs(got - ref), tol))
    assert abs(got - ref) < tol
