"""Rounding where a small system's products ride in the plane stage's launch: the
error of H psi is no larger than that of the general path (another plane
variant: short chains per workgroup, their sums in FP64).  The FP32 form against
the FP64 form, the FP64 form against long double; the projector energies are ten
times the usual ones, so that the products' rounding is most of the error.  Bound
1.1: both errors are norms over 8 or more orbitals, whose spread between seeds is
2 %."""
import numpy as np
import pytest
import scipy.fft

from sdft_amd import hip, systems

pytestmark = pytest.mark.gpu

A0 = 10.26


def _system(n, natm):
    rng = np.random.default_rng(natm)
    return systems.build_system("e%d" % n, A0, 1, n, g2max=(0.19 * n * 2.0 * np.pi / A0) ** 2,
                                pos=rng.uniform(0, A0, (natm, 3)), h_kb=(20.0, 10.0))


def _errors(s, C, prec, ref=None):
    ctx = hip.Context(s)
    err = []
    for variant in (0, 1):
        ctx.set_config(variant, 512)
        r = ctx.hpsi_raw(C) if ref is None else ref
        d = abs(ctx.hpsi_raw(C, prec) - r)
        err.append(float(np.sqrt((d ** 2).sum() / (abs(r) ** 2).sum())))
    ctx.close()
    print("n", s.n[0], "projectors", s.nproj, "orbitals", len(C), "errors", err, flush=True)
    return err


@pytest.mark.parametrize("n,natm,nst", [(24, 16, 32), (32, 16, 64), (36, 27, 8), (48, 50, 8),
                                        (64, 64, 8), (64, 64, 64)])
def test_fp32_rounds_no_worse(n, natm, nst):
    s = _system(n, natm)
    small, general = _errors(s, systems.noise_orbitals(s, nst, seed=n), hip.PREC_FP32)
    assert small <= 1.1 * general


def _hpsi_long(C, s):
    """H psi as the library returns it (-4 H c, -2 H c at G = 0) in long double."""
    C = C.astype(np.clongdouble)
    v = s.vks.astype(np.longdouble).reshape(s.n)
    f = np.empty_like(C)
    for c, o in zip(C, f):
        g = np.zeros(s.ngrid, np.clongdouble)
        g[s.map[:-1]], g[s.map_conj[:-1]], g[0] = c[:-1], np.conj(c[:-1]), c[-1].real
        r = scipy.fft.ifftn(g.reshape(s.n), norm="forward")
        F = scipy.fft.fftn(r * v, norm="forward").ravel()
        o[:-1] = -4 * F[s.map[:-1]] - 2 * s.ak2[:-1].astype(np.longdouble) * c[:-1]
        o[-1] = -2 * F[0].real
    Q = s.proj.astype(np.clongdouble)
    Z = 2 * (C[:, :-1].real @ Q[:, :-1].real.T - C[:, :-1].imag @ Q[:, :-1].imag.T)
    Z = (Z + np.outer(C[:, -1].real, Q[:, -1].real)) * s.proj_energy
    f[:, :-1] -= 4 * (Z @ np.conj(Q[:, :-1]))
    f[:, -1] -= 2 * (Z @ Q[:, -1].real)
    return f


@pytest.mark.parametrize("n,natm", [(24, 16), (36, 27), (48, 50), (64, 64)])
def test_fp64_rounds_no_worse(n, natm):
    s = _system(n, natm)
    C = systems.noise_orbitals(s, 8, seed=n)
    small, general = _errors(s, C, hip.PREC_FP64, _hpsi_long(C, s))
    assert small <= 1.1 * general
