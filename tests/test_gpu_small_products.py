"""Kleinman-Bylander products of small systems (projection in the plane stage's
launch, reduction in the force product's or in a launch of its own) against the
oracle at the parity tests' bounds (FP64 1e-12, FP32 2e-5) and against the
general path (another plane tile: its own launches on a second stream), whose
sums differ in order only (1e-13, 5e-6).  Projector counts below, at and above
a tile of 32; states of one, part of, one and several tiles; 64 projectors with
32 states are the largest fused tile, 65 projectors the next; so are 1024 with
one pair of orbitals, and with two."""
import numpy as np
import pytest

from oracle import sdft_oracle as O
from sdft_amd import hip, systems

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,natm,states", [(24, 1, (1, 31)), (24, 16, (2, 32, 65)),
                                           (32, 17, (33,)), (36, 27, (16, 18)),
                                           (48, 9, (1, 40)), (64, 50, (3, 12)),
                                           (24, 200, (1,)), (24, 256, (1, 3))])
def test_small_products(n, natm, states):
    rng = np.random.default_rng(n + natm)
    g2 = (0.2 * n * 2.0 * np.pi / 10.26) ** 2
    s = systems.build_system("p%d_%d" % (n, natm), 10.26, 1, n, g2max=g2,
                             pos=rng.uniform(0, 10.26, (natm, 3)))
    ctx = hip.Context(s)
    for nst in states:
        print("n", n, "projectors", s.nproj, "states", nst, flush=True)
        C = systems.noise_orbitals(s, nst, seed=nst)
        ref = O.hpsi_raw(C, s)
        for prec, tol, dif in ((hip.PREC_FP64, 1e-12, 1e-13), (hip.PREC_FP32, 2e-5, 5e-6)):
            ctx.set_config(0, 512)
            f = ctx.hpsi_raw(C, prec)
            ctx.set_config(1, 512)
            assert _rel(f, ref) < tol
            assert _rel(f, ctx.hpsi_raw(C, prec)) < dif
    ctx.close()
