"""The a-plane stage per wave, whole and as its two halves around the grid:
every grid size, spheres from one wave vector per axis to the largest inside
n/4 and one beyond (where the workgroup-wide stage takes over), one orbital, an
odd count and several pairs, against the oracle at the parity tests' bounds
(FP64 1e-12, FP32 2e-5)."""
import math

import numpy as np
import pytest

from oracle import sdft_oracle as O
from sdft_amd import hip, systems

pytestmark = pytest.mark.gpu

A0 = 10.26
POS = np.array([[0.1, 0.2, 0.3], [4.0, 7.5, 1.3]])


def _system(n, K):
    g2 = ((K + 0.3) * 2.0 * math.pi / A0) ** 2
    return systems.build_system("w%d_%d" % (n, K), A0, 1, n, g2max=g2, pos=POS)


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n", [24, 32, 36, 48, 64, 96, 128])
def test_plane_stage_against_oracle(n):
    top = (n - 1) // 4
    for K, states in ((1, (1, 2)), (top // 2, (3,)), (top, (1, 6)), (top + 1, (2,))):
        s = _system(n, K)
        assert int(np.abs(s.k).max()) == K and (4 * K < n) == (K <= top)
        ctx = hip.Context(s)
        rs = systems.real_space_projectors(s, 2.0)
        for form in (None, rs):
            if form is not None:
                ctx.set_projectors_real(rs)
            for nst in states:
                print("n", n, "K", K, "states", nst, "real" if form else "table", flush=True)
                C = systems.noise_orbitals(s, nst, seed=7 * n + K)
                ref = O.hpsi_raw(C, s, nl_real=form)
                assert _rel(ctx.hpsi_raw(C), ref) < 1e-12
                assert _rel(ctx.hpsi_raw(C, hip.PREC_FP32), ref) < 2e-5
        ctx.close()
