"""Orbital transfers across the C ABI: separate re / im arrays and interleaved
complex arrays, through pinned memory (small), staging (larger) and several
staging passes, odd and even state counts.  A transfer moves numbers and
computes none, so every comparison is exact."""
import ctypes as C

import numpy as np
import pytest

from sdft_amd import hip, systems

pytestmark = pytest.mark.gpu


def _planar(a):
    return np.ascontiguousarray(a.real), np.ascontiguousarray(a.imag)


def _p(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


@pytest.fixture(scope="module")
def ctxs():
    out = {}

    def get(rep, n):
        if n not in out:
            out[n] = hip.Context(systems.build_system("t%d" % n, 10.26, rep, n, with_nl=False))
        return out[n]

    yield get
    for c in out.values():
        c.close()


# bytes per state: 5920 at 32^3, 48256 at 64^3.  44 / 45 and 88 / 89 states
# at 32^3 lie on either side of the pinned regions (256 KiB up, 512 KiB down);
# 1391 states at 64^3 take two passes of the 64 MiB staging buffer.
@pytest.mark.parametrize("rep,n,nstate", [(1, 32, 1), (1, 32, 2), (1, 32, 44), (1, 32, 45),
                                          (1, 32, 88), (1, 32, 89), (2, 64, 7), (2, 64, 1391)])
def test_round_trip_both_layouts(ctxs, rep, n, nstate):
    ctx = ctxs(rep, n)
    lib, nc = ctx.lib, ctx.sys.ncoef
    rng = np.random.default_rng(nstate)
    chi = rng.standard_normal((nstate, nc, 2)).view(np.complex128)[..., 0]
    blk = hip.Block(ctx, nstate)
    try:
        blk.set(chi)
        re, im = np.empty((nstate, nc)), np.empty((nstate, nc))
        assert lib.sdft_hip_block_get(blk.h, 1, _p(re), _p(im)) == 0
        assert np.array_equal(re, chi.real) and np.array_equal(im, chi.imag)
        pr, pi = _planar(2.0 * chi)
        assert lib.sdft_hip_block_set(blk.h, _p(pr), _p(pi)) == 0
        assert np.array_equal(blk.get(1), 2.0 * chi)
    finally:
        blk.close()


@pytest.mark.parametrize("nstate", [1, 5, 90])
def test_calls_take_both_layouts(ctxs, nstate):
    """One H application and one filter (in-place T_{L-1}, accumulator) from
    separate arrays equal those from interleaved ones, also when a smaller
    call follows a larger one on the context's kept block."""
    ctx = ctxs(1, 32)
    chi = systems.noise_orbitals(ctx.sys, nstate, seed=3)
    for prec in (hip.PREC_FP64, hip.PREC_FP32, hip.PREC_FP64):
        f = ctx.hpsi_raw(chi, prec)
        re, im = _planar(chi)
        fr, fi = np.empty_like(re), np.empty_like(im)
        assert ctx.lib.sdft_hip_hpsi(ctx.h, nstate, _p(re), _p(im), _p(fr), _p(fi), prec) == 0
        assert np.array_equal(fr, f.real) and np.array_equal(fi, f.imag)
        co = np.array([0.3, -0.2, 0.1, 0.05])
        acc, t, mom = ctx.cheby_filter(chi, co, 0.2, 4.0, prec, moments=True)
        m2 = np.zeros(4)
        ar, ai = np.empty_like(re), np.empty_like(im)
        assert ctx.lib.sdft_hip_cheby_filter(ctx.h, nstate, 4, _p(co), 0.2, 4.0, _p(re), _p(im),
                                             _p(ar), _p(ai), _p(m2), prec) == 0
        assert np.array_equal(ar, acc.real) and np.array_equal(ai, acc.imag)
        assert np.array_equal(re, t.real) and np.array_equal(im, t.imag)
        assert np.array_equal(m2, mom)
    small = ctx.hpsi_raw(chi[:1])
    assert np.array_equal(small, ctx.hpsi_raw(chi[:1]))
