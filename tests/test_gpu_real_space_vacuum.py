"""Real-space projectors in a cell that is mostly vacuum: tiles without a
projector's point get their potential on the way to the grid.  Grids of each
form of the plane stage (per wave, per workgroup, split), one orbital and an
odd count, one atom, and projector lists that are all empty, against the oracle
(FP64 1e-12, FP32 2e-5)."""
import dataclasses
import math

import numpy as np
import pytest

from oracle import sdft_oracle as O
from sdft_amd import hip, systems

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,K,states", [(32, 7, (1, 5)), (48, 11, (3,)), (64, 15, (3,)),
                                        (96, 23, (3,)), (128, 31, (2,)), (128, 33, (1,)),
                                        (192, 20, (1,)), (192, 34, (2,))])
def test_vacuum(n, K, states):
    g2 = ((K + 0.3) * 2.0 * math.pi / 10.26) ** 2
    s = systems.build_system("v%d_%d" % (n, K), 10.26, 1, n, g2max=g2, with_nl=False,
                             pos=np.array([[2.1, 8.2, 5.3]]))
    rs = systems.real_space_projectors(s, 1.6)
    ctx = hip.Context(s)
    ctx.set_projectors_real(rs)
    for nst in states:
        C = systems.noise_orbitals(s, nst, seed=n + nst)
        ref = O.hpsi_raw(C, s, nl_real=rs)
        for prec, tol in ((hip.PREC_FP64, 1e-12), (hip.PREC_FP32, 2e-5)):
            print("n", n, "K", K, "states", nst, "prec", prec, flush=True)
            assert _rel(ctx.hpsi_raw(C, prec), ref) < tol
    ctx.close()


def test_empty_lists():
    s = systems.build_system("v0", 10.26, 1, 32, with_nl=False)
    rs = systems.real_space_projectors(s, 1.6)
    rs = dataclasses.replace(rs, offsets=np.zeros_like(rs.offsets), index=rs.index[:0],
                             values=rs.values[:0])
    ctx = hip.Context(s)
    ctx.set_projectors_real(rs)
    C = systems.noise_orbitals(s, 3, seed=1)
    ref = O.hpsi_raw(C, s, with_nl=False)
    assert _rel(ctx.hpsi_raw(C), ref) < 1e-12
    assert _rel(ctx.hpsi_raw(C, hip.PREC_FP32), ref) < 2e-5
    ctx.close()
