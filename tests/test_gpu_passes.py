"""GPU: the small kernels ahead of and behind the fold, at the sizes where
their splits end: ray tables that settle in 31 points, in 61 and only
adaptively; parallels whose leaves are seen in part (the invisible-phase
padding), over more than 64 leaf steps; the background marginal with its bell
whole, clipped and with signals from LDS or memory; channel counts about 64;
energy grids beyond what LDS holds twice; and the response fold's last rows.
The references: xpsi/cellmesh/rays.pyx:61-390, xpsi/cellmesh/
integrator_for_azimuthal_invariance.pyx:343-549, xpsi/likelihoods/
default_background_marginalisation.pyx, xpsi/tools/energy_integrator.pyx,
xpsi/Instrument.py:163-197."""
import math
import sys

import numpy as np
import pytest

from oracle import oracle as O
from tests.bars import LNL_ATOL, SIG_RTOL, elem_relerr

pytestmark = pytest.mark.gpu


def say(msg):
    print("[gpu] " + msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("u", [0.05, 0.3, 0.54, 0.6, 0.64])
@pytest.mark.parametrize("n_rays", [3, 65, 200])
def test_rays_by_compactness(u, n_rays):
    from xpsi_amd.cellmesh.rays import compute_rays
    uu = np.array([u, u * (1 + 1e-3), u * (1 - 1e-3)])
    maxA = np.array([0.5 * math.pi, 0.5 * math.pi + 0.02, 0.5 * math.pi + 0.1])
    mg, mr = maxA.copy(), maxA.copy()
    say("rays: u %.3f, %d a parallel" % (u, n_rays))
    t, d, ca, lg, md = compute_rays(1, 3, 4.0e3, uu, mg, n_rays)
    tr, dr, car, lgr, mdr = O.compute_rays(4.0e3, uu, mr, n_rays)
    assert t == tr == 0
    # both are adaptive to 1e-12 of each integral, some of them differences of two;
    # cos_alpha = 1 - j inc passes through zero with the rounding of 200 inc
    for a, b in ((d, dr), (lg, lgr), (md, mdr)):
        assert elem_relerr(a, b) < 1e-11
    assert np.max(np.abs(ca - car)) < 200 * 2.3e-16


@pytest.mark.parametrize("colat", [0.3, 1.57, 2.2, 2.6])
@pytest.mark.parametrize("N_L", [7, 32, 33, 130, 131])
def test_leaves_seen_in_part(colat, N_L):
    from xpsi_amd import configs
    from xpsi_amd.cellmesh.integrator_for_azimuthal_invariance import integrate
    sp = configs.config1(np.zeros((100, 32)))["spacetime"]
    st = O.spacetime(sp["mass"], sp["radius"], sp["distance"], 0.3, sp["frequency"])
    hr = dict(super_colatitude=colat, super_radius=0.5, super_temperature=6.1, phase_shift=0.0, sqrt_num_cells=10,
              min_sqrt_num_cells=6, max_sqrt_num_cells=40, num_rays=60, num_leaves=N_L, is_antiphased=False)
    members, err = O.hot_region_embed(st, hr, sp["frequency"])
    assert err is None
    m = members[0]
    E, leaves, phases = np.logspace(-0.5, 1.0, 5), np.linspace(0, 2 * math.pi, N_L), 2 * math.pi * np.linspace(0, 1, 19)
    t, ref = O.integrate(st["Omega"], st["r_s"], st["i"], m["cellArea"], m["r"], m["r_s_over_r"], m["theta"], m["phi"],
                         m["params"], m["radiates"], m["deflection"], m["cos_alpha"], m["lag"], m["maxDeflection"],
                         m["cos_gamma"], E, leaves, phases, correction=None)
    say("leaves: colatitude %.2f, %d leaves" % (colat, N_L))
    status, flux = integrate(1, st["R"], st["Omega"], st["r_s"], st["i"], m["cellArea"], m["r"], m["r_s_over_r"],
                             m["theta"], m["phi"], m["params"], m["radiates"], None, m["deflection"].shape[1],
                             m["deflection"], m["cos_alpha"], m["lag"], m["maxDeflection"], m["cos_gamma"], E, leaves,
                             phases, (), (), 1, 1, 0)
    assert status == t
    if t == 0:
        err = elem_relerr(flux, ref)
        say("rel err %.2e" % err)
        assert err < SIG_RTOL


@pytest.mark.parametrize("mean", [0.2, 3.0, 900.0])
@pytest.mark.parametrize("channels,bins,n_phases,star", [(1, 8, 16, 0.5), (64, 32, 40, 0.02), (65, 33, 300, 0.9),
                                                         (129, 64, 700, 1.0)])
def test_marginal_passes(mean, channels, bins, n_phases, star):
    from xpsi_amd.likelihoods import default_background_marginalisation as G
    rng = np.random.default_rng(3)
    T = 2.0e4
    phases = np.linspace(0.0, 1.0, bins + 1)
    grid = np.linspace(0.0, 1.0, n_phases)
    comp = (star * mean * bins / T) * (1.0 + 0.5 * np.cos(2 * math.pi * grid))[None, :] * np.ones((channels, 1))
    counts = rng.poisson(mean, (channels, bins)).astype(np.float64)
    counts[:, 0] += 1.0     # a channel without counts is of the llzero class, a random draw on either side
    pre = O.precomputation(counts.astype(np.int32))
    sup = np.zeros((channels, 2))
    sup[:, 1] = -1.0
    if channels > 64:
        sup[::3, 1] = 0.8 * mean * bins / T     # a bound inside the bell
    say("marginal: %d channels, %d bins, %d phases, mean %.1f" % (channels, bins, n_phases, mean))
    args = (T, phases, counts, (comp, 0.3 * comp), (grid, grid), np.array([0.1, 0.4]), pre, sup)
    out = G.eval_marginal_likelihood(*args, 1000, 0.0, 1.0e-8, 1.0e-3, 10.0, -1.0e90, slim=-1.0)
    ref = O.eval_marginal_likelihood(*args, slim=-1.0)
    say("lnL gpu %.10f oracle %.10f" % (out[0], ref[0]))
    # each channel's integral is adaptive to 1e-11 on both sides; sums of counts
    # times logarithms are rounded to some 1e-16 of their total
    assert abs(out[0] - ref[0]) < max(LNL_ATOL, channels * (2e-11 + 1e-15 * mean * bins * 10))
    assert elem_relerr(out[1], ref[1]) < SIG_RTOL


@pytest.mark.parametrize("N_E", [5, 6, 40, 4096, 4097])
def test_energy_integral_grids(N_E):
    from xpsi_amd.tools.energy_integrator import energy_integrator
    rng = np.random.default_rng(N_E)
    x = np.linspace(-0.6, 1.1, N_E)
    sig = rng.uniform(0.5, 2.0, (N_E, 3))
    edges = np.linspace(-0.5, 1.0, 12)
    say("energy integral: %d energies" % N_E)
    got, ref = energy_integrator(1, sig, x, edges), O.energy_integrator(sig, x, edges)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert elem_relerr(np.nan_to_num(got), np.nan_to_num(ref)) < SIG_RTOL


@pytest.mark.parametrize("rows,inputs,phases", [(1, 1, 1), (16, 31, 33), (33, 32, 16), (40, 33, 32), (100, 129, 65)])
def test_response_fold_remainders(rows, inputs, phases):
    from xpsi_amd.instrument import Instrument
    rng = np.random.default_rng(rows)
    M, sig = rng.uniform(size=(rows, inputs)), rng.uniform(size=(inputs, phases))
    inst = Instrument(M, np.linspace(0.3, 10.0, inputs + 1), np.arange(rows))
    say("fold: %d x %d x %d" % (rows, inputs, phases))
    got = np.asarray(inst(sig, (0, inputs), (0, rows)))
    assert elem_relerr(got, M @ sig) < 1e-13
