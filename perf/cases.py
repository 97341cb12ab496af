"""The work that programs have this library do, as cases that can be timed and checked.

A case is one pass through the public Python entry points (sdft_amd.hip) as a
stochastic-DFT program calls them.  `prepare` makes what such a program has in
hand before the call: the system's context (grid, plane-wave set, potential,
Kleinman-Bylander projectors), the orbitals, the polynomial.  `run` is the call.

The kinds of work, in the order of an SCF iteration:

  spectral   spectral range by power iteration on one orbital (the smallest
             latency-bound chain of H applications)
  hpsi       one H application to orbitals in host arrays
  moments    Chebyshev moments of a block in host arrays
  mu         chemical potential from the moments, and the expansion coefficients
  filter     the Chebyshev filter of a block in host arrays, with moments, as
             filterChebyPolyHerm is called
  block      the same filter on orbitals resident on the device
  newton     the Newton-form filter with several chemical potentials
  batch      the filter of many fragment systems together
  scf        what closes the iteration: density, Kohn-Sham potential, energies
             and forces
  density    the density alone

Results of the FP32 form carry single-precision accuracy, and a program that
asks for it keeps them in single precision.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "stochastic-density-functional-theory-piny_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from sdft_amd import hip, systems  # noqa: E402

A0 = 10.26          # diamond silicon, bohr
KB_CUTOFF = 4.0     # real-space projectors, bohr


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one orbital of the smallest fragment: what a caller with its own
        # iteration (a spectral estimate, a residual) asks for, latency only
        dict(name="hpsi_24_1", kind="hpsi", n=24, nstate=1, prec=0, nl="table"),
        # an H application to an odd block on a mid-size grid in the FP32 form
        dict(name="hpsi_96_65_fp32", kind="hpsi", n=96, nstate=65, prec=1, nl="table"),
        # the spectral range of a fragment: a chain of dependent H applications
        dict(name="spectral_36", kind="spectral", n=36, nstate=1, L=96, prec=0, nl="table"),
        # the chemical-potential search and the coefficients of one SCF iteration
        dict(name="mu_1024", kind="mu", n=32, L=1024),
        # Si8, 64 orbitals, degree 256: the whole filter call with its moments
        dict(name="filter_32_64", kind="filter", n=32, nstate=64, L=256, prec=0, nl="table"),
        # the moments pass of a fragment, an odd block
        dict(name="moments_48_93_fp32", kind="moments", n=48, nstate=93, L=257, prec=1,
             nl="table"),
        # Si64, 256 resident orbitals, the two precision forms
        dict(name="block_64_256_fp32", kind="block", n=64, nstate=256, L=512, prec=1,
             nl="table"),
        dict(name="block_64_256", kind="block", n=64, nstate=256, L=256, prec=0, nl="table"),
        # Si512 with real-space projectors, a block of orbitals in FP32
        dict(name="block_128_64_real_fp32", kind="block", n=128, nstate=64, L=64, prec=1,
             nl="real"),
        # a slab of Si288 in the 192^3 cell of Si1728, real-space projectors, FP64
        dict(name="block_192_32_real", kind="block", n=192, nstate=32, L=32, prec=0,
             nl="real"),
        # a batch of uneven fragments
        dict(name="batch_24_fp32", kind="batch", nfrag=24, L=128, prec=1),
        # the end of an SCF iteration of Si64: density, potential, energies, forces
        dict(name="scf_64_128", kind="scf", n=64, nstate=128, prec=0, nl="table"),
    ]


def draw(rng):
    """One more case: any kind, over the grids, block sizes, degrees, forms and
    projector kinds that the listed cases stand for."""
    kind = rng.choice(["hpsi", "hpsi", "spectral", "mu", "filter", "moments", "newton", "block",
                       "block", "batch", "scf", "density"])

    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    prec = rng.randrange(2)
    if kind == "mu":
        return dict(kind=kind, n=32, L=logint(100, 3000))
    if kind == "batch":
        return dict(kind=kind, nfrag=logint(3, 24), L=logint(16, 128), prec=prec)
    if kind == "spectral":
        n = rng.choice((24, 32, 36, 48, 64))
        return dict(kind=kind, n=n, nstate=1, L=logint(16, 96), prec=prec, nl="table")
    if kind in ("scf", "density"):
        n = rng.choice((32, 48, 64, 96, 128) if kind == "density" else (32, 64))
        top = max(2, min(128, 128 * 64 ** 3 // n ** 3))
        return dict(kind=kind, n=n, nstate=logint(1, top), prec=0,
                    nl="table" if kind == "scf" else "none")
    n = rng.choice((24, 32, 36, 48, 64, 96, 128, 192))
    nl = "real" if n >= 128 or (n > 24 and rng.random() < 0.3) else "table"
    top = max(2, min(256, 256 * 64 ** 3 // n ** 3))
    nstate = logint(1, top)
    if kind == "hpsi":
        return dict(kind=kind, n=n, nstate=nstate, prec=prec, nl=nl)
    most = max(16, int(256 * 64 ** 3 * 256 / (n ** 3 * max(nstate, 16))))
    return dict(kind=kind, n=n, nstate=nstate, L=logint(16, min(512, most)), prec=prec, nl=nl)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _wells(L, n, pos):
    """A potential of atomic wells on the grid, FFTW order (the depth and width
    of the screened silicon potential), from per-axis tables."""
    x = np.arange(n) * (L / n)
    e = []
    for d in range(3):
        u = x[:, None] - pos[None, :, d]
        u -= L * np.round(u / L)
        e.append(np.exp(-(u / 1.1) ** 2))
    jk = (e[1][:, None, :] * e[2][None, :, :]).reshape(n * n, -1)
    return np.ascontiguousarray((-1.6 * (e[0] @ jk.T)).ravel())


def _atoms(n, rng):
    """(cell side, positions) of the cell that goes with a grid."""
    if n in (24, 36, 48):
        natm = {24: 9, 36: 27, 48: 50}[n]
        _, p = systems.diamond_supercell(A0, 3)
        side = A0 * (natm / 8.0) ** (1.0 / 3.0)
        d = p - (1.5 * A0 + rng.uniform(-0.5, 0.5, 3) * A0)
        pos = np.mod(d[np.argsort(np.abs(d).max(axis=1), kind="stable")[:natm]] + 0.5 * side, side)
        return side, pos
    rep = n // 32
    side, pos = systems.diamond_supercell(A0, rep)
    if n in (96, 192):  # a slab: one layer of cells, the rest vacuum
        pos = pos[pos[:, 2] < 0.99 * A0]
    return side, pos + rng.normal(0.0, 0.05, size=pos.shape)


def _system(n, rng, nl="table"):
    """The system of a grid: cell, displaced atoms, plane waves, potential and
    projectors (the G-space table, the real-space lists, or none)."""
    side, pos = _atoms(n, rng)
    table = nl == "table"
    if n <= 64:
        s = systems.build_system("si%d" % len(pos), A0, 1, n, pos=pos, with_nl=table, cell=side,
                                 separable_sf=True)
    else:
        k = systems.half_sphere(side, 12.0)
        m, mc = systems.fftw_maps(k, (n, n, n))
        g = k * (2.0 * math.pi / side)
        if table:
            proj, pe, pa, pl, pm = systems.kb_table(side, pos, k, 0.8, (2.0, 1.0))
        else:
            proj, pe = np.zeros((0, len(k)), dtype=np.complex128), np.zeros(0)
            pa = pl = pm = np.zeros(0, dtype=np.int64)
        s = systems.System(name="si%d" % len(pos), L=side, n=(n, n, n), pos=pos, k=k, map=m,
                           map_conj=mc, ak2=(g * g).sum(axis=1), gvec=g,
                           vks=_wells(side, n, pos), proj=proj, proj_energy=pe, proj_atom=pa,
                           proj_l=pl, proj_m=pm)
    rs = systems.real_space_projectors(s, min(KB_CUTOFF, 0.45 * side)) if nl == "real" else None
    return s, rs


def _orbitals(nstate, ncoef, rng):
    """Stochastic orbitals: unit covariance on the coefficient set, G = 0 real."""
    c = rng.standard_normal((nstate, ncoef, 2)).view(np.complex128)[..., 0] * math.sqrt(0.5)
    c[:, -1] = rng.standard_normal(nstate)
    return c


def _range(s):
    """Bounds of the spectrum: potential, kinetic energy, and the projectors
    (energies 2 and 1 Ha, hardly overlapping)."""
    return float(s.vks.min()), float(0.5 * s.ak2.max() + s.vks.max() + 2.5)


def _fermi(x, mu, beta):
    with np.errstate(over="ignore"):
        return 1.0 / (1.0 + np.exp(beta * (x - mu)))


def _cheby(L, emin, emax, mu, beta):
    """Chebyshev coefficients of the root of the Fermi function."""
    M = 16 * L
    t = np.cos(2.0 * math.pi * np.arange(M) / M)
    f = np.sqrt(_fermi(0.5 * (emax - emin) * t + 0.5 * (emax + emin), mu, beta))
    c = 2.0 * np.fft.fft(f).real[:L] / M
    c[0] *= 0.5
    return np.ascontiguousarray(c)


def _leja(L):
    """L Leja points of [-2, 2]."""
    x = np.cos(math.pi * (np.arange(16 * L) + 0.5) / (16 * L)) * 2.0
    z = np.empty(L)
    z[0] = x[0]
    w = np.log(np.abs(x - z[0]) + 1e-300)
    for i in range(1, L):
        z[i] = x[np.argmax(w)]
        w += np.log(np.abs(x - z[i]) + 1e-300)
    return z


def _newton(L, emin, emax, mus, beta):
    """Newton-form coefficients (L, nmu) of the root of the Fermi function on
    L Leja points of the range mapped to [-2, 2], and the points."""
    z = _leja(L)
    e = 0.25 * (emax - emin) * z + 0.5 * (emax + emin)
    d = np.stack([np.sqrt(_fermi(e, mu, beta)) for mu in mus], axis=1)
    for j in range(1, L):
        d[j:] = (d[j:] - d[j - 1:-1]) / (z[j:] - z[:-j])[:, None]
    return np.ascontiguousarray(d), z


def _inputs(case, seed):
    """The host data of a case, from its seed alone."""
    rng = np.random.default_rng([11, seed])
    kind = case["kind"]
    if kind == "mu":
        L = case["L"]
        emin, emax = -1.0 + 0.1 * rng.random(), 9.0 + 0.1 * rng.random()
        # moments of a smooth density of states on 64 states per orbital
        y = np.clip(rng.normal(-0.1, 0.45, 4096), -0.999, 0.999)
        m = np.cos(np.arange(L + 1)[:, None] * np.arccos(y)[None, :]).sum(axis=1)
        nsto = 64.0
        x = 0.5 * (emax - emin) * y + 0.5 * (emax + emin)
        mu = float(np.quantile(x, 0.3 + 0.1 * rng.random()))
        ne = float(2.0 * _fermi(x, mu, 100.0).sum() / nsto)
        return dict(L=L, emin=emin, emax=emax, beta=100.0, moments=m, nsto=nsto, ne=ne,
                    mu0=mu + 0.1 * (rng.random() - 0.5), sys=_system(case["n"], rng)[0])
    if kind == "batch":
        specs = systems.fragment_specs(343, 3)
        frags = []
        for i in range(0, 14 * case["nfrag"], 14):
            specs[i].pos = specs[i].pos + rng.normal(0.0, 0.05, size=specs[i].pos.shape)
            s = systems.build_fragment(specs[i])
            emin, emax = _range(s)
            frags.append(dict(sys=s, chi=_orbitals(specs[i].nstate, s.ncoef, rng),
                              scale=2.0 / (emax - emin), emean=0.5 * (emin + emax),
                              coeffs=_cheby(case["L"], emin, emax, 0.2, 100.0)))
        return dict(frags=frags)
    s, rs = _system(case["n"], rng, case["nl"])
    emin, emax = _range(s)
    d = dict(sys=s, rs=rs, chi=_orbitals(case["nstate"], s.ncoef, rng), emin=emin, emax=emax,
             scale=2.0 / (emax - emin), emean=0.5 * (emin + emax))
    if kind in ("filter", "block"):
        d["coeffs"] = _cheby(case["L"], emin, emax, 0.2, 100.0)
    elif kind == "newton":
        d["scale"] = 4.0 / (emax - emin)
        d["coeffs"], z = _newton(case["L"], emin, emax, (0.15, 0.25), 20.0)
        d["points"] = np.ascontiguousarray(z[:-1])
    elif kind == "scf":
        d["dens"] = systems.density_sphere(s)
        d["vext"] = systems.vloc_density(s, d["dens"], separable=True)
        d["vloc"] = systems.vloc_form_factor(s, d["dens"])
    return d


def _context(s, rs):
    ctx = hip.Context(s, with_nl=rs is None)
    if rs is not None:
        ctx.set_projectors_real(rs)
    return ctx


def prepare(case, seed):
    d = _inputs(case, seed)
    st = dict(case=case)
    if case["kind"] == "batch":
        f = d["frags"]
        st["ctx"] = [_context(x["sys"], None) for x in f]
        st["blocks"] = [hip.Block(c, len(x["chi"]), case["prec"]) for c, x in zip(st["ctx"], f)]
        for b, x in zip(st["blocks"], f):
            b.set(x["chi"])
        st["batch"] = hip.Batch(st["blocks"])
        st["coeffs"] = np.stack([x["coeffs"] for x in f])
        st["scale"] = np.array([x["scale"] for x in f])
        st["emean"] = np.array([x["emean"] for x in f])
        return st
    d["ctx"] = _context(d["sys"], d.get("rs"))
    if case["kind"] == "block":
        d["block"] = hip.Block(d["ctx"], case["nstate"], case["prec"])
        d["block"].set(d["chi"])
    elif case["kind"] == "scf":
        d["ctx"].ks_init(d["dens"])
        d["types"] = np.zeros(d["sys"].natm, dtype=np.int32)
    st.update(d)
    return st


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _kept(case, *arrays):
    """Results as the program keeps them: FP32-form results in single precision."""
    if case.get("prec"):
        return [a.astype(np.complex64 if a.dtype.kind == "c" else np.float32) for a in arrays]
    return list(arrays)


def run(st):
    case = st["case"]
    kind = case["kind"]
    prec = case.get("prec", 0)
    if kind == "batch":
        st["batch"].filter(st["coeffs"], st["scale"], st["emean"])
        return _kept(case, *[b.get(0) for b in st["blocks"]])
    ctx = st["ctx"]
    if kind == "hpsi":
        return _kept(case, ctx.hpsi_raw(st["chi"], prec))
    if kind == "spectral":
        e, v, _ = ctx.spectral_bound(st["chi"][0], 0, conv=0.0, max_iter=case["L"], prec=prec)
        return _kept(case, np.array([e]), v)
    if kind == "mu":
        mu, ne = ctx.chem_pot(st["L"], st["emin"], st["emax"], st["beta"], st["moments"],
                              st["nsto"], st["ne"], st["mu0"], 0.1)
        c = ctx.cheby_coeffs(st["L"], st["emin"], st["emax"], st["mu0"], st["beta"])
        return [np.array([mu]), np.array([ne]), c]
    if kind == "filter":
        return _kept(case, *ctx.cheby_filter(st["chi"], st["coeffs"], st["scale"], st["emean"],
                                             prec, moments=True))
    if kind == "moments":
        return _kept(case, ctx.cheby_moments(st["chi"], case["L"], st["scale"], st["emean"], prec))
    if kind == "newton":
        return _kept(case, *ctx.newton_filter(st["chi"], st["coeffs"], st["points"], st["scale"],
                                              st["emean"], prec))
    if kind == "block":
        st["block"].filter(st["coeffs"], st["scale"], st["emean"])
        return _kept(case, st["block"].get(0))
    occ = 2.0 / case["nstate"]
    if kind == "density":
        return [ctx.density(st["chi"], occ, hip.RHO_GENERIC)]
    s = st["sys"]
    rho = ctx.density(st["chi"], occ, hip.RHO_GENERIC)
    vks, e = ctx.ks_potential(rho, st["vext"], s.volume, hip.XC_PZ_LDA, hip.RHO_GENERIC)
    eke, enl = ctx.energies(st["chi"], 2.0, case["nstate"])
    fnl = ctx.nl_forces(st["chi"], 2.0, case["nstate"])
    floc = ctx.local_forces(s.pos, st["types"], st["vloc"], st["dens"].gvec)
    return [rho, vks, np.array([e["eh"], e["eext"], e["exc"], eke, enl]), fnl, floc]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _sphere(n):
    """(coefficients, columns, projectors) of a grid's usual system."""
    K = {24: 5, 32: 5, 36: 8, 48: 10, 64: 11, 96: 16, 128: 22, 192: 33}[n]
    nat = {24: 9, 32: 8, 36: 27, 48: 50, 64: 64, 96: 72, 128: 512, 192: 288}[n]
    return int(2.0 / 3.0 * math.pi * K ** 3) + 1, int(math.pi * K * K), 4 * nat


def _step(n, nstate, nl):
    """(bytes, flops) of one H application with its recurrence on resident
    FP64 orbitals: T_k, T_k-1 and the accumulator read, T_k+1 and the
    accumulator written, the potential once; the transforms of the sphere's
    columns, rows and lines per orbital pair, and the projectors."""
    nc, ncol, P = _sphere(n)
    line = 5.0 * n * math.log2(n)
    rows = 2.0 * math.sqrt(ncol / math.pi) + 1.0
    fl = (nstate + 1) // 2 * 2.0 * line * (ncol + n * (rows + n))
    by = 80.0 * nc * nstate + 8.0 * n ** 3
    if nl == "none":
        return by, fl
    if nl == "real":
        pts = 4.0 / 3.0 * math.pi * (KB_CUTOFF * n / (A0 * n / 32.0)) ** 3
        return by + 9.0 * P * pts, fl + 8.0 * P * pts * nstate
    return by + 32.0 * nc * P, fl + 16.0 * nc * P * nstate


def work(case):
    kind = case["kind"]
    if kind == "mu":
        M = 32.0 * case["L"]
        return dict(bytes=16.0 * case["L"], flops=M * (2.0 * case["L"] + 40 * 20.0))
    if kind == "batch":
        by = fl = 0.0
        for n, share, ns in ((24, 0.03, 33), (32, 0.25, 40), (36, 0.17, 64), (48, 0.55, 95)):
            b, f = _step(n, ns, "table")
            by += share * case["nfrag"] * b
            fl += share * case["nfrag"] * f
        return dict(bytes=by * (case["L"] - 1), flops=fl * (case["L"] - 1))
    n, ns = case["n"], case["nstate"]
    by, fl = _step(n, ns, case["nl"])
    nc, ncol, P = _sphere(n)
    if kind == "hpsi":
        return dict(bytes=by, flops=fl)
    if kind in ("density", "scf"):
        b, f = 16.0 * nc * ns + 8.0 * n ** 3, 0.5 * fl
        if kind == "scf":
            b += 4 * 8.0 * n ** 3 + 3 * 16.0 * nc * ns + 16.0 * nc * P
            f += 4 * 8.0 * nc * P * ns + 8 * 5.0 * n ** 3 * math.log2(n)
        return dict(bytes=b, flops=f)
    steps = case["L"] // 2 if kind == "moments" else case["L"] - 1
    return dict(bytes=by * steps, flops=fl * steps)


# ---------------------------------------------------------------------------
# The same results in 64 bits
# ---------------------------------------------------------------------------

class _H:
    """H on complex orbitals (state, coefficient) in plain torch, 64 bits."""

    def __init__(self, s, rs, dev):
        t = lambda a, k=torch.float64: torch.as_tensor(np.ascontiguousarray(a), device=dev).to(k)  # noqa: E731
        self.dev, self.n, self.N = dev, s.n[0], s.ngrid
        self.map, self.mapc = t(s.map, torch.int64), t(s.map_conj, torch.int64)
        self.v, self.ak2 = t(s.vks), t(s.ak2)
        self.q, self.e = (t(s.proj, torch.complex128), t(s.proj_energy)) if s.nproj else (None, None)
        self.rs = None
        if rs is not None:
            # an atom's four channels share one point list
            cnt = np.diff(rs.offsets)[::4]
            top = int(cnt.max())
            idx = np.zeros((len(cnt), top), dtype=np.int64)
            val = np.zeros((len(cnt), 4, top))
            for a in range(len(cnt)):
                o = rs.offsets[4 * a:4 * a + 5]
                idx[a, :cnt[a]] = rs.index[o[0]:o[1]]
                val[a, :, :cnt[a]] = rs.values[o[0]:o[4]].reshape(4, -1)
            self.rs = (t(idx, torch.int64), t(val),
                       t(rs.energy.reshape(-1, 4) * rs.vol_elem))

    def grids(self, c):
        """Orbital pairs packed as psi1 + i psi2 on the grid."""
        if len(c) % 2:
            c = torch.cat([c, torch.zeros_like(c[:1])])
        a, b = c[0::2], c[1::2]
        z = torch.zeros(len(a), self.N, dtype=torch.complex128, device=self.dev)
        z[:, self.mapc] = a.conj() + 1j * b.conj()
        z[:, self.map] = a + 1j * b
        n = self.n
        return torch.fft.ifftn(z.view(-1, n, n, n), dim=(1, 2, 3), norm="forward").view(-1, self.N)

    def coefs(self, z, count):
        n = self.n
        F = torch.fft.fftn(z.view(-1, n, n, n), dim=(1, 2, 3), norm="forward").view(-1, self.N)
        p, m = F[:, self.map], F[:, self.mapc].conj()
        out = torch.stack([0.5 * (p + m), -0.5j * (p - m)], dim=1).flatten(0, 1)[:count]
        out[:, -1] = out[:, -1].real.to(out.dtype)
        return out

    def projections(self, c):
        return 2.0 * (c[:, :-1] @ self.q[:, :-1].T).real + c[:, -1:].real * self.q[:, -1].real

    def real_kb(self, z):
        idx, val, e = self.rs
        out = torch.zeros(z.shape[1], z.shape[0], dtype=torch.float64, device=self.dev)
        im = torch.zeros_like(out)
        zt = z.T.contiguous()
        for a in range(0, len(idx), 32):
            i, b, ee = idx[a:a + 32], val[a:a + 32], e[a:a + 32]
            for part, to in ((zt.real, out), (zt.imag, im)):
                g = part[i.reshape(-1)].view(i.shape[0], i.shape[1], -1)
                y = torch.matmul(b, g) * ee[:, :, None]
                to.index_add_(0, i.reshape(-1), torch.matmul(b.transpose(1, 2).contiguous(), y).flatten(0, 1))
        return torch.complex(out, im).T

    def __call__(self, c):
        z = self.grids(c)
        w = z * self.v
        if self.rs is not None:
            w = w + self.real_kb(z)
        h = self.coefs(w, len(c)) + 0.5 * self.ak2 * c
        if self.q is not None:
            y = (self.projections(c) * self.e).to(torch.complex128)
            h[:, :-1] += y @ self.q[:, :-1].conj()
            h[:, -1] += y @ self.q[:, -1].real.to(torch.complex128)
        h[:, -1] = h[:, -1].real.to(h.dtype)
        return h


def _dot(a, b):
    s = 2.0 * (a.real * b.real + a.imag * b.imag).sum(-1) - a[..., -1].real * b[..., -1].real
    return float(s.sum())


def _expand(h, chi, coeffs, scale, emean, count):
    """sum_k c_k T_k chi, the last T_k, and <chi|T_k chi> for k < count."""
    H = lambda c: scale * (h(c) - emean * c)  # noqa: E731
    acc, a, b = coeffs[0] * chi, chi, H(chi)
    mom = [_dot(chi, chi), _dot(chi, b)]
    acc = acc + coeffs[1] * b
    for k in range(2, count):
        a, b = b, 2.0 * H(b) - a
        acc += coeffs[k] * b
        mom.append(_dot(chi, b))
    return acc, b, np.array(mom[:count])


def exact(case, seed):
    kind = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if dev == "cpu" and work(case)["flops"] > 2e11:
        return None
    d = _inputs(case, seed)
    if kind == "mu":
        return _exact_mu(d)
    host = lambda x: x.cpu().numpy()  # noqa: E731
    if kind == "batch":
        out = []
        for f in d["frags"]:
            h = _H(f["sys"], None, dev)
            chi = torch.as_tensor(f["chi"], device=dev)
            out.append(host(_expand(h, chi, f["coeffs"], f["scale"], f["emean"], case["L"])[0]))
        return out
    s = d["sys"]
    h = _H(s, d["rs"], dev)
    chi = torch.as_tensor(d["chi"], device=dev)
    if kind == "hpsi":
        f = -4.0 * h(chi)
        f[:, -1] *= 0.5
        return [host(f)]
    if kind == "spectral":
        phi = chi[:1] / math.sqrt(_dot(chi[:1], chi[:1]))
        for _ in range(case["L"]):
            w = h(phi)
            e = _dot(w, phi)
            phi = w / math.sqrt(_dot(w, w))
        return [np.array([e]), host(phi)[0]]
    if kind in ("filter", "block"):
        acc, last, mom = _expand(h, chi, d["coeffs"], d["scale"], d["emean"], case["L"])
        return [host(acc)] if kind == "block" else [host(acc), host(last), mom]
    if kind == "moments":
        return [_exact_moments(h, chi, case["L"], d["scale"], d["emean"])]
    if kind == "newton":
        co, p = d["coeffs"], chi
        out = [c * chi for c in co[0]]
        for k in range(1, len(co)):
            p = d["scale"] * (h(p) - d["emean"] * p) - d["points"][k - 1] * p
            out = [o + c * p for o, c in zip(out, co[k])]
        return [host(torch.stack(out)), host(p)]
    z = h.grids(chi)
    n = s.n[0]
    rho = (z.real.square() + z.imag.square()).sum(0) * (2.0 / case["nstate"])
    generic = lambda x: host(x.view(n, n, n).permute(2, 1, 0).reshape(-1))  # noqa: E731
    if kind == "density":
        return [generic(rho)]
    return _exact_scf(case, d, s, h, chi, rho, generic, dev)


def _exact_moments(h, chi, L, scale, emean):
    """mu_0 .. mu_L from the first half and the product identities, as the
    moments of an even or odd degree are written (a direct mu_k wins)."""
    H = lambda c: scale * (h(c) - emean * c)  # noqa: E731
    top = L // 2 + 1 if L % 2 == 0 else (L + 1) // 2
    m = np.zeros(L + 1)
    a, b = chi, H(chi)
    m[0], m[1] = _dot(chi, chi), _dot(chi, b)
    for k in range(2, top):
        a, b = b, 2.0 * H(b) - a
        m[k] = _dot(chi, b)
        m[2 * k - 1] = 2.0 * _dot(b, a) - m[1]
        m[2 * k] = 2.0 * _dot(b, b) - m[0]
    return m


def _exact_mu(d):
    """The root of N(mu) = N_e, and the coefficients at the starting mu."""
    L, M = d["L"], _closest_23(32 * d["L"])
    j = np.arange(M)
    t = np.cos(2.0 * math.pi * j / M)
    x = 0.5 * (d["emax"] - d["emin"]) * t + 0.5 * (d["emax"] + d["emin"])
    m = np.zeros(M)
    m[:L] = 2.0 * d["moments"][:L]
    m[0] *= 0.5
    w = np.fft.fft(m).real * (2.0 / (d["nsto"] * M))
    lo, hi = d["mu0"] - 1.0, d["mu0"] + 1.0
    for _ in range(100):
        mid = 0.5 * (lo + hi)
        lo, hi = (mid, hi) if float(_fermi(x, mid, d["beta"]) @ w) < d["ne"] else (lo, mid)
    f = np.sqrt(_fermi(x, d["mu0"], d["beta"]))
    c = 2.0 * np.fft.fft(f).real[:L] / M
    c[0] *= 0.5
    return [np.array([0.5 * (lo + hi)]), np.array([d["ne"]]), c]


def _closest_23(n):
    """The 2^a 3^b nearest to n (the quadrature's point count)."""
    best = None
    for a in range(int(math.log2(n)) + 2):
        for b in range(int(math.log(n, 3)) + 2):
            v = 2 ** a * 3 ** b
            if best is None or abs(v - n) < abs(best - n):
                best = v
    return best


def _exact_scf(case, d, s, h, chi, rho, generic, dev):
    n, N, V, dens = s.n[0], s.ngrid, s.volume, d["dens"]
    t = lambda a, k=torch.float64: torch.as_tensor(np.ascontiguousarray(a), device=dev).to(k)  # noqa: E731
    mp, mc = t(dens.map, torch.int64), t(dens.map_conj, torch.int64)
    vext, g2, g = t(d["vext"], torch.complex128), t(dens.ak2), t(dens.gvec)
    q = torch.fft.fftn(rho.view(n, n, n), norm="forward").view(-1)[mp]
    hart = torch.zeros_like(vext)
    hart[:-1] = 4.0 * math.pi * q[:-1] / (g2[:-1] * V)
    vg = vext + hart
    z = torch.zeros(N, dtype=torch.complex128, device=dev)
    z[mc] = vg.conj()
    z[mp] = vg
    z[0] = vext[-1].real.to(z.dtype)
    vr = torch.fft.ifftn(z.view(n, n, n), norm="forward").view(-1).real
    # Perdew-Zunger LDA
    r = rho / V
    rs = (3.0 / (4.0 * math.pi * r)).pow(1.0 / 3.0)
    sq, lr = rs.sqrt(), rs.log()
    vx = -(3.0 * r / math.pi).pow(1.0 / 3.0)
    c1 = 1.0 + 1.0529 * sq + 0.3334 * rs
    c2 = 1.0 + 7.0 / 6.0 * 1.0529 * sq + 4.0 / 3.0 * 0.3334 * rs
    A, B, C, D = 0.0311, -0.048, 0.002, -0.0116
    far = rs >= 1.0
    ec = torch.where(far, -0.1423 / c1, A * lr + B + C * rs * lr + D * rs)
    mu = torch.where(far, -0.1423 * c2 / c1 ** 2, A * lr + (B - A / 3.0) + 2.0 / 3.0 * C * rs * lr
                     + (2.0 * D - C) / 3.0 * rs)
    eh = float((4.0 * math.pi * q[:-1].abs().square() / (g2[:-1] * V)).sum())
    ee = float(2.0 * (vext[:-1] * q[:-1].conj()).real.sum() + vext[-1].real * q[-1].real)
    ex = float(((0.75 * vx + ec) * r).sum()) * V / N
    ns = case["nstate"]
    eke = float((2.0 * h.ak2[:-1] * chi[:, :-1].abs().square()).sum()) / ns
    Z = h.projections(chi)
    enl = 2.0 * float((Z.square() * h.e).sum()) / ns
    gv = t(s.gvec)
    fnl = np.zeros((s.natm, 3))
    floc = np.zeros((s.natm, 3))
    pos, f = t(s.pos), t(d["vloc"])[0]
    for x in range(3):
        dZ = 2.0 * (chi[:, :-1] @ (1j * gv[:-1, x] * h.q[:, :-1]).T).real
        per = (-4.0 / ns * h.e * (Z * dZ).sum(0)).cpu().numpy()
        np.add.at(fnl[:, x], s.proj_atom, per)
    ph = g @ pos.T
    w = f[:, None] * (ph.cos() * q.imag[:, None] + ph.sin() * q.real[:, None])
    w[-1] = 0.0
    floc[:] = (2.0 * (w.T @ g)).cpu().numpy()
    return [generic(rho), generic(vr + vx + mu), np.array([eh, ee, ex, eke, enl]), fnl, floc]
