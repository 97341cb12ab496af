"""The KB workgroup target that sdft_hip_tune keeps is a measured one.  With
variant 0 a small system's products do not use it (both targets run the same
launches), so it must be that of the fastest of the candidates that do: the
variants from 1 on.  Candidate order: variant, target (256, 1024), fused
expand."""
import numpy as np
import pytest

from sdft_amd import hip, systems

pytestmark = pytest.mark.gpu


def test_target_of_a_small_system_is_one_that_was_used():
    s = systems.build_system("tune", 10.26, 1, 32, pos=np.random.default_rng(2).uniform(
        0, 10.26, (20, 3)))
    ctx = hip.Context(s)
    small = 0
    for _ in range(8):
        (tile, kt, fu), ms = ctx.tune(32, hip.PREC_FP64, steps=4)
        assert len(ms) == 8
        best = int(np.argmin(ms))
        assert (tile, fu) == (best // 4, best % 2)
        if tile == 0:
            small += 1
            best = 4 + int(np.argmin(ms[4:]))
        assert kt == (256, 1024)[best // 2 % 2]
    assert small > 0
    ctx.close()
