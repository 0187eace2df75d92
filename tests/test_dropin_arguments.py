"""Arguments of the drop-ins as a caller may write them: tuples, lists, arrays
of other types and strides, as np.ascontiguousarray takes them (the reference's
typed memoryviews are arrays; its callers build phase shifts and grids as
sequences, xpsi/likelihoods/default_background_marginalisation.pyx:450-734)."""
import math

import numpy as np
import pytest

from oracle import oracle as O


class _HostTorch:
    """torch with its device and page-locked allocations in ordinary memory."""

    def __getattr__(self, name):
        import torch
        return getattr(torch, name)

    def empty(self, *size, dtype, device=None, pin_memory=False):
        import torch
        return torch.empty(*size, dtype=dtype)


@pytest.mark.parametrize("length", [1, 2, 3])
def test_call_takes_sequences(monkeypatch, length):
    from xpsi_amd import _device as D
    monkeypatch.setattr(D, "require_gpu", _HostTorch)
    want = np.linspace(0.1, 0.3, length)
    given = [tuple(want), list(want), want, np.repeat(want, 2)[::2]]
    call = D.Call(given, ((2,),))
    raw = call.buf.numpy()
    for p in call.inputs:
        assert np.array_equal(raw[p.off:p.off + 8 * length].view(np.float64), want)


def test_call_marks_types_and_absent_inputs(monkeypatch):
    from xpsi_amd import _device as D
    monkeypatch.setattr(D, "require_gpu", _HostTorch)
    call = D.Call([D.As((3, 1, 4), np.int32), D.As(None), D.As((0.5, 1.5))], ((2,),))
    raw, (n, absent, x) = call.buf.numpy(), call.inputs
    assert np.array_equal(raw[n.off:n.off + 12].view(np.int32), [3, 1, 4])
    assert absent is None and D.ptr(absent) is None
    assert np.array_equal(raw[x.off:x.off + 16].view(np.float64), [0.5, 1.5])


def _forms(a):
    """The same values as a tuple, a list and an array of another stride."""
    a = np.asarray(a)
    return tuple(a.tolist()), a.tolist(), np.repeat(a, 2, axis=0)[::2]


@pytest.mark.gpu
def test_marginal_sequences():
    from xpsi_amd.likelihoods import default_background_marginalisation as G
    rng = np.random.default_rng(5)
    phases, grid, shifts = np.linspace(0.0, 1.0, 9), np.linspace(0.0, 1.0, 17), np.array([0.1, 0.4])
    comp = 2.0 + np.cos(2 * math.pi * grid)[None, :] * np.ones((3, 1))
    counts = rng.poisson(9.0, (3, 8)).astype(np.float64)
    pre, sup = O.precomputation(counts.astype(np.int32)), np.tile([0.0, -1.0], (3, 1))

    def call(phases, shifts, counts, pre, sup, grid, **kw):
        print("[gpu] marginal: shifts as %s" % type(shifts).__name__, flush=True)
        return G.eval_marginal_likelihood(2.0, phases, counts, (comp, comp), (grid, grid), shifts, pre, sup, 1000, 0.0,
                                          1e-8, 1e-3, 10.0, -1e90, slim=-1.0, **kw)
    for kw in ({}, {"allow_negative": (True, False)}, {"background": np.full((3, 8), 0.5)}):
        ref = call(phases, shifts, counts, pre, sup, grid, **kw)
        for args in zip(*(_forms(a) for a in (phases, shifts, counts, pre, sup, grid))):
            got = call(*args, **kw)
            assert got[0] == ref[0]
            for a, b in zip(got[1:], ref[1:]):
                assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("stokes", [False, True])
def test_integrator_sequences(stokes):
    from tests.test_gpu_slabfold import _mesh
    from xpsi_amd.cellmesh import integrator_for_azimuthal_invariance as P, integratorIQU_for_azimuthal_invariance as Q
    st, m = _mesh()
    E, leaves, phases = np.logspace(-0.5, 1.0, 6), np.linspace(0.0, 2 * math.pi, 20), np.linspace(0.0, 6.0, 9)

    def call(E, leaves, phases, radial):
        print("[gpu] integrate: energies as %s" % type(E).__name__, flush=True)
        fn = Q.integrate if stokes else P.integrate
        return fn(1, st["R"], st["Omega"], st["r_s"], st["i"], m["cellArea"], radial, m["r_s_over_r"], m["theta"],
                  m["phi"], m["params"], m["radiates"], None, m["deflection"].shape[1], m["deflection"],
                  m["cos_alpha"], m["lag"], m["maxDeflection"], m["cos_gamma"], E, leaves, phases,
                  *((),) * (3 if stokes else 2), 1, 1, 0)
    ref = call(E, leaves, phases, m["r"])
    assert ref[0] == 0
    for args in zip(*(_forms(a) for a in (E, leaves, phases, m["r"]))):
        got = call(*args)
        assert got[0] == 0
        # blocks add to the flux in any order: a few roundings of sums of positive terms
        assert np.allclose(got[1], ref[1], rtol=1e-13, atol=0.0)


@pytest.mark.gpu
def test_ray_sequences():
    from xpsi_amd.cellmesh.rays import compute_rays
    u = np.array([0.3, 0.31])
    out = []
    for form in (u,) + _forms(u):
        print("[gpu] rays: compactness as %s" % type(form).__name__, flush=True)
        out.append(compute_rays(1, 2, 4.0e3, form, np.full(2, 0.5 * math.pi), 20))
    for got in out[1:]:
        assert got[0] == 0
        for a, b in zip(got[1:], out[0][1:]):
            assert np.array_equal(a, b)
