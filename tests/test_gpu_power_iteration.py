"""The spectral bound's iterations are queued ahead of the host: the last one
that counts is the same as in a loop that looks at each (energy, vector and
number of iterations), with limits below, at and above the queue's depth and
with a convergence test that ends the loop."""
import numpy as np
import pytest

from oracle import sdft_oracle as O
from sdft_amd import hip, systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_iter,conv", [(1, 0.0), (2, 0.0), (3, 0.0), (4, 0.0), (7, 1e-9),
                                           (400, 1e-1), (400, 1e-2), (400, 1e6), (400, 1e8)])
@pytest.mark.parametrize("which", [0, 1])
def test_last_iteration(max_iter, conv, which):
    s = systems.build_system("pw", 10.26, 1, 32)
    ctx = hip.Context(s)
    v0 = systems.noise_orbitals(s, 1, seed=5)[0]
    e_r, v_r, it_r = O.gen_energy_bound(v0, s, which, emax=30.0, conv=conv, max_iter=max_iter)
    e, v, it = ctx.spectral_bound(v0, which, emax=30.0, conv=conv, max_iter=max_iter)
    assert it == it_r
    assert abs(e - e_r) <= 1e-9 * abs(e_r)
    assert np.linalg.norm(v - v_r) <= 1e-9 * np.linalg.norm(v_r)
    ctx.close()
