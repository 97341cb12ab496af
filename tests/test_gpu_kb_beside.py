"""Filter steps with the Kleinman-Bylander products on a second stream, on both
sides of the rules that choose the plane stage and whether the products are
queued ahead of it or behind: 128^3 at 16 and 17 pairs (FP64 with the largest
sphere whose planes fit LDS in the stage per wave, and the next), 64^3 FP32 and
48^3 FP64 one pair below and at 320 MiB of pair grids, 192^3.  Five Chebyshev
terms, so that steps follow each other on alternating streams: states from the
first, a middle and the last pair against the oracle at the parity tests' bounds
(FP64 1e-12, FP32 2e-5), and the whole block against another plane variant."""
import math

import numpy as np
import pytest

from oracle import sdft_oracle as O
from sdft_amd import hip, systems

pytestmark = pytest.mark.gpu

A0 = 10.26


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,K,natm,prec,states", [
    (128, 23, 20, hip.PREC_FP64, (32, 33)), (128, 24, 20, hip.PREC_FP64, (3, 34)),
    (128, 22, 20, hip.PREC_FP32, (32, 33)), (64, 12, 50, hip.PREC_FP32, (317, 319)),
    (48, 9, 60, hip.PREC_FP64, (377, 380)), (192, 24, 12, hip.PREC_FP64, (3,)),
    (192, 24, 12, hip.PREC_FP32, (4,))])
def test_filter_beside_products(n, K, natm, prec, states):
    rng = np.random.default_rng(n + natm)
    s = systems.build_system("b%d" % n, A0, 1, n, g2max=((K + 0.3) * 2.0 * math.pi / A0) ** 2,
                             pos=rng.uniform(0, A0, (natm, 3)), separable_sf=True)
    assert int(np.abs(s.k).max()) == K
    lo, hi = float(s.vks.min()) - 1.0, float(0.5 * s.ak2.max() + s.vks.max() + 4.0 * natm)
    co = np.array([0.3, -0.7, 0.45, 0.2, -0.15])
    scale, emean = 2.0 / (hi - lo), 0.5 * (hi + lo)
    tol = 1e-12 if prec == hip.PREC_FP64 else 2e-5
    ctx = hip.Context(s)
    for nst in states:
        print("n", n, "K", K, "projectors", s.nproj, "states", nst, "prec", prec, flush=True)
        C = systems.noise_orbitals(s, nst, seed=nst)
        ctx.set_config(0, 512)
        acc, last = ctx.cheby_filter(C, co, scale, emean, prec)
        pick = sorted({0, 1, nst // 2, nst - 2, nst - 1} & set(range(nst)))
        ref = O.filter_cheby(C[pick], co, s, scale, emean)
        assert _rel(acc[pick], ref[0]) < tol
        assert _rel(last[pick], ref[1]) < tol
        ctx.set_config(1, 512)
        acc1, last1 = ctx.cheby_filter(C, co, scale, emean, prec)
        assert _rel(acc, acc1) < tol and _rel(last, last1) < tol
    ctx.close()
