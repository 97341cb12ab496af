"""What a context keeps between calls on host arrays: no buffer above 256 MiB,
whatever the degree of a call.  The moment partials of a kept block grow with
the degree (24 bytes per chunk, pair and step), so the block is small here and
the degree high; device memory free after the call is compared with that after
the same call at a low degree (16 MiB for the runtime's own)."""
import numpy as np
import pytest
import torch

from sdft_amd import hip, systems

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("call", ["moments", "filter"])
def test_moment_partials_of_a_high_degree_are_given_back(call):
    s = systems.build_system("kept", 10.26, 1, 24, pos=np.array([[0.1, 0.2, 0.3]]))
    ctx = hip.Context(s)
    chi = systems.noise_orbitals(s, 256, seed=1)
    L = 72000 if call == "moments" else 36000  # 36000 steps: 105 MiB a chunk, four of them
    co = np.zeros(L)

    def run(n):
        if call == "moments":
            ctx.cheby_moments(chi, n, 1e-3, 0.0)
        else:
            ctx.cheby_filter(chi, co[:n], 1e-3, 0.0, moments=True)

    run(16)
    before = _free()
    run(L)
    kept = before - _free()
    print("call", call, "kept", kept / MIB, "MiB", flush=True)
    ctx.close()
    given_back = _free() - before
    assert kept <= 256 * MIB + 16 * MIB
    assert given_back >= 0
