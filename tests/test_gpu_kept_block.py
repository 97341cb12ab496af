"""Calls on host arrays share the context's kept block and scratch.  After large
calls of every kind on one context (FP32 filter with moments, Newton filter with
three chemical potentials, moments, density, forces, noise), smaller calls of
each kind in both precisions give what a fresh context gives for that call
alone: sums in the same order, so the bounds are those of a reordered sum (FP64
1e-13, FP32 5e-6); anything left over from a larger call would show at order
one.  With projectors, on a system whose products ride in the plane stage's
launch and on one whose products run on the second stream."""
import numpy as np
import pytest

from sdft_amd import hip, systems

pytestmark = pytest.mark.gpu

A0 = 10.26


def _calls(ctx, s, nst, prec):
    """One call of every kind on `nst` orbitals: {name: results}."""
    chi = systems.noise_orbitals(s, nst, seed=nst)
    co = np.array([0.3, -0.7, 0.45, 0.2])
    z = np.array([1.9, -1.9, 0.1])
    nco = np.stack([co, 0.5 * co, -co], axis=1)
    scale, emean = 0.05, 8.0
    out = {
        "hpsi": [ctx.hpsi_raw(chi, prec)],
        "filter": list(ctx.cheby_filter(chi, co, scale, emean, prec, moments=True)),
        "newton": list(ctx.newton_filter(chi, nco, z, scale, emean, prec)),
        "moments": [ctx.cheby_moments(chi, 7, scale, emean, prec)],
        "bound": list(ctx.spectral_bound(chi[0], 0, conv=0.0, max_iter=3, prec=prec)[:2]),
    }
    if prec == hip.PREC_FP64:
        out.update(density=[ctx.density(chi, 2.0 / nst)], energies=list(ctx.energies(chi, 2.0, nst)),
                   forces=[ctx.nl_forces(chi, 2.0, nst)], noise=[ctx.noise(nst, 5)])
    return out


@pytest.mark.parametrize("n,natm", [(32, 8), (48, 60)])
def test_smaller_calls_after_larger_ones(n, natm):
    rng = np.random.default_rng(n)
    s = systems.build_system("k%d" % n, A0, 1, n, g2max=(0.19 * n * 2.0 * np.pi / A0) ** 2,
                             pos=rng.uniform(0, A0, (natm, 3)))
    ctx = hip.Context(s)
    for nst, prec in ((150, hip.PREC_FP32), (150, hip.PREC_FP64)):
        _calls(ctx, s, nst, prec)
    for nst in (1, 7, 34, 96):
        for prec, tol in ((hip.PREC_FP32, 5e-6), (hip.PREC_FP64, 1e-13)):
            got = _calls(ctx, s, nst, prec)
            fresh = hip.Context(s)
            want = _calls(fresh, s, nst, prec)
            fresh.close()
            for name in want:
                print("n", n, "states", nst, "prec", prec, name, flush=True)
                for g, w in zip(got[name], want[name]):
                    assert np.linalg.norm(np.asarray(g) - w) <= tol * np.linalg.norm(w)
    ctx.close()
