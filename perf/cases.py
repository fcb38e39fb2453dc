"""The work that programs have this framework do, as cases that can be timed.

Every case calls public entry points on device tensors, as a simulation
pipeline does: the FP64 transforms of ``glass_amd.healpix`` (the default
precision of every drop-in function), ``generate`` and ``from_convergence``
built on them, the batched FP32 engines ``LognormalShells`` and
``ShearShells``, multi-plane lensing, and the preparation of Gaussian spectra.

``exact`` restates each path in 64 bits with plain torch: Wigner-d recurrences
for whole blocks of m, float64 matrix products over l, and chirp-z transforms
along the rings.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import glass_amd
from glass_amd import healpix
from glass_amd.batch import LognormalShells, ShearShells, shell_spectra

# correlation of a shell with its neighbours, by the number of neighbours kept
# (a chain that ends after one neighbour admits at most 1/2)
RHO = ((), (0.45,), (0.6, 0.3), (0.6, 0.3, 0.1), (0.6, 0.3, 0.1))


def listed():
    return [
        # one low-resolution map, as tests and quick looks make it: launches and latency
        {"name": "alm2map-n32", "kind": "alm2map", "nside": 32, "lmax": 64},
        # one field at the resolution of a C_l study, synthesis ...
        {"name": "alm2map-n1024", "kind": "alm2map", "nside": 1024, "lmax": 2048},
        # ... and its analysis with healpy's three refinement passes
        {"name": "map2alm-n1024", "kind": "map2alm", "nside": 1024, "lmax": 2048, "iter": 3},
        # a spin-2 field at a resolution that is no power of two, E and B
        {"name": "spin-n300", "kind": "spin", "nside": 300, "lmax": 767, "spin": 2},
        # deflection and shear of a source plane, with the pixel weights and windows
        {"name": "convergence-n256", "kind": "convergence", "nside": 256, "lmax": 512},
        # the drop-in generator: ten correlated lognormal shells, one map at a time
        {"name": "generate-n128", "kind": "generate", "nside": 128, "lmax": 256, "shells": 10,
         "ncorr": 1},
        # the batch engine on the same small job, on a ragged one, and on the headline job
        {"name": "shells-n128", "kind": "shells", "nside": 128, "lmax": 256, "shells": 10,
         "ncorr": 1},
        {"name": "shells-n512", "kind": "shells", "nside": 512, "lmax": 1023, "shells": 33,
         "ncorr": 3},
        {"name": "shells-n2048", "kind": "shells", "nside": 2048, "lmax": 4096, "shells": 64,
         "ncorr": 3},
        # the shear of a whole stack of source planes
        {"name": "shear-n1024", "kind": "shear", "nside": 1024, "lmax": 2047, "shells": 64},
        # the convergence behind a handful of density shells, plane by plane
        {"name": "planes-n1024", "kind": "planes", "nside": 1024, "shells": 6, "bits": 32},
        # one Gaussian spectrum for a lognormal field (each pair of shells needs one)
        {"name": "solve-l2048", "kind": "solve", "lmax": 2048},
    ]


def _nside(rng, lo, hi):
    """log-uniform in [lo, hi]: most often a power of two, else any number."""
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return 2 ** round(math.log2(x)) if rng.random() < 0.6 else max(lo, int(x))


def draw(rng):
    kind = rng.choice(["alm2map", "alm2map", "map2alm", "map2alm", "spin", "convergence",
                       "generate", "shells", "shells", "shear", "planes", "solve"])
    if kind == "solve":
        return {"kind": kind, "lmax": int(math.exp(rng.uniform(math.log(100), math.log(4097))))}
    if kind == "planes":
        return {"kind": kind, "nside": _nside(rng, 32, 2048), "shells": rng.randint(2, 8),
                "bits": rng.choice([32, 64])}
    hi = {"alm2map": 2048, "map2alm": 1024, "spin": 1024, "convergence": 512, "generate": 512,
          "shells": 1024, "shear": 512}[kind]
    nside = _nside(rng, 16, hi)
    # band limits in use run from below 2 nside to healpy's 3 nside - 1
    lmax = min(rng.choice([2 * nside, 2 * nside - 1, rng.randint(nside, 3 * nside - 1)]), 4096)
    case = {"kind": kind, "nside": nside, "lmax": lmax}
    if kind == "map2alm":
        case["iter"] = rng.choice([0, 1, 3])
    if kind == "spin":
        case["spin"] = rng.choice([1, 2])
    if kind in ("generate", "shells", "shear"):
        room = int(2e8 / (12 * nside * nside))
        top = max(2, min({"generate": 12, "shells": 80, "shear": 24}[kind], room))
        case["shells"] = rng.randint(2, top)
    if kind in ("generate", "shells"):
        case["ncorr"] = rng.randint(0, 4)
    return case


# ---------------------------------------------------------------------------
# inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _ell(lmax):
    return torch.arange(lmax + 1, dtype=torch.float64, device="cuda")


def _hp_lm(lmax):
    """(l, m) of every coefficient in healpy order."""
    m = torch.repeat_interleave(torch.arange(lmax + 1, device="cuda"),
                                torch.arange(lmax + 1, 0, -1, device="cuda"))
    first = m * (2 * lmax + 1 - m) // 2
    return torch.arange(m.numel(), device="cuda") - first, m


def _alm(lmax, g):
    """Gaussian coefficients of a red spectrum (the workloads' synthetic family)."""
    l, m = _hp_lm(lmax)
    x = l.double()
    c = torch.sqrt(1e-4 * (x + 1.0) ** -1.2 * torch.exp(-((x / 1500.0) ** 2)) / 2)
    z = torch.randn((2, l.numel()), generator=g, dtype=torch.float64, device="cuda") * c
    re = torch.where(m == 0, z[0] * math.sqrt(2.0), z[0])
    im = torch.where(m == 0, torch.zeros_like(z[1]), z[1])
    return torch.complex(re, im)


def _contrast(shape, g, dtype):
    """A density-like map: lognormal pixels on a slow gradient, above -1."""
    x = torch.randn(shape, generator=g, dtype=torch.float32, device="cuda")
    ramp = torch.linspace(-0.3, 0.3, shape[-1], device="cuda")
    return torch.expm1(0.5 * x + ramp - 0.125).to(dtype)


def _gls(case, seed):
    n = case["shells"]
    scale = 1.0 + 0.3 * np.random.default_rng(seed).random()
    return shell_spectra(n, case["lmax"], rho=RHO[case["ncorr"]],
                         amp=lambda i: scale * (1.0 + 3.0 * i / max(n - 1, 1)))


def _target_cl(case, seed):
    r = np.random.default_rng(seed)
    ell = np.arange(case["lmax"] + 1, dtype=np.float64)
    amp, tilt = r.uniform(0.5, 4.0), r.uniform(-1.5, -1.0)
    return amp * 1e-4 * (ell + 1.0) ** tilt * np.exp(-((ell / 1500.0) ** 2))


class _Cosmology:
    """Distances of an Einstein-de Sitter universe in units of the Hubble
    distance: what the multi-plane recursion asks of a cosmology."""

    Omega_m0 = 1.0
    hubble_distance = 1.0

    def H_over_H0(self, z):
        return (1.0 + np.asarray(z)) ** 1.5

    def transverse_comoving_distance(self, z1, z2=None):
        def d(z):
            return 2.0 * (1.0 - 1.0 / np.sqrt(1.0 + np.asarray(z, dtype=np.float64)))
        return d(z1) if z2 is None else d(z2) - d(z1)


def prepare(case, seed):
    kind, s = case["kind"], dict(case)
    g = _gen(seed)
    if kind == "solve":
        s["cl"] = _target_cl(case, seed)
        s["field"] = glass_amd.grf.Lognormal(1.0)
        return s
    nside = case["nside"]
    npix = 12 * nside * nside
    if kind == "planes":
        dtype = torch.float32 if case["bits"] == 32 else torch.float64
        s["deltas"] = [_contrast((npix,), g, dtype) for _ in range(case["shells"])]
        s["cosmo"] = _Cosmology()
        return s
    lmax = case["lmax"]
    # the tables that a program keeps for a geometry are made by its first calls
    zero = torch.zeros((lmax + 1) * (lmax + 2) // 2, dtype=torch.complex128, device="cuda")
    if kind in ("alm2map", "map2alm", "generate"):
        healpix.alm2map(zero, nside, lmax=lmax)
    if kind == "alm2map":
        s["alm"] = _alm(lmax, g)
    elif kind == "map2alm":
        s["map"] = _contrast((npix,), g, torch.float64)
    elif kind == "spin":
        healpix.alm2map_spin([zero, zero], nside, case["spin"], lmax)
        s["alms"] = [_alm(lmax, g), 0.1 * _alm(lmax, g)]
    elif kind == "convergence":
        healpix.alm2map_spin([zero, zero], nside, 1, lmax)
        healpix.alm2map_spin([zero, zero], nside, 2, lmax)
        healpix.pixel_weights(nside)
        healpix.pixwin(nside, lmax=lmax, pol=True)
        s["kappa"] = 0.02 * _contrast((npix,), g, torch.float64)
    elif kind == "generate":
        s["gls"] = [torch.as_tensor(c) for c in _gls(case, seed)]
        s["fields"] = [glass_amd.grf.Lognormal(1.0)] * case["shells"]
        s["rng"] = glass_amd.DeviceRNG(seed)
    elif kind == "shells":
        s["engine"] = LognormalShells(_gls(case, seed), nside, ncorr=case["ncorr"], shift=1.0,
                                      seed=seed, lmax=lmax)
    elif kind == "shear":
        s["kappa"] = 0.02 * _contrast((case["shells"], npix), g, torch.float32)
        s["engine"] = ShearShells(nside, lmax, case["shells"])
    return s


# ---------------------------------------------------------------------------
# one pass


def run(s):
    kind = s["kind"]
    if kind == "alm2map":
        return healpix.alm2map(s["alm"], s["nside"], lmax=s["lmax"])
    if kind == "map2alm":
        return healpix.map2alm(s["map"], lmax=s["lmax"], iter=s["iter"])
    if kind == "spin":
        return healpix.alm2map_spin(s["alms"], s["nside"], s["spin"], s["lmax"])
    if kind == "convergence":
        return glass_amd.from_convergence(s["kappa"], s["lmax"], deflection=True, shear=True)
    if kind == "generate":
        return list(glass_amd.generate(s["fields"], s["gls"], s["nside"], ncorr=s["ncorr"],
                                       rng=s["rng"]))
    if kind == "shells":
        return s["engine"].run()
    if kind == "shear":
        return s["engine"].run(s["kappa"])
    if kind == "planes":
        planes = glass_amd.MultiPlaneConvergence(s["cosmo"])
        for i, delta in enumerate(s["deltas"]):
            planes.add_plane(delta, 0.1 * (i + 1), 0.1)
        return planes.kappa
    gl, cl, info = glass_amd.grf.solve(s["cl"], s["field"], s["field"], pad=2 * len(s["cl"]))
    return {"gl": gl, "cl": cl, "info": info}


def work(case):
    """Inputs read once and outputs written once; four operations per
    coefficient and ring pair for the sum over l, and the ring transforms."""
    kind = case["kind"]
    if kind == "solve":
        n = case["lmax"] + 1
        # the first guess, then at least one evaluation, on 3 n nodes
        return {"bytes": 8.0 * (n + n + 3 * n), "flops": 4.0 * n * n + 2 * 4.0 * 9 * n * n}
    npix = 12 * case["nside"] ** 2
    if kind == "planes":
        # the last density plane lies behind its own source plane and adds nothing yet
        n = case["bits"] / 8 * npix
        return {"bytes": n * case["shells"], "flops": 2.0 * npix * case["shells"]}
    lmax, S = case["lmax"], case.get("shells", 1)
    na = (lmax + 1) * (lmax + 2) // 2
    one = 4.0 * na * 2 * case["nside"] + 2.5 * npix * math.log2(4 * case["nside"])
    if kind == "alm2map":
        return {"bytes": 16.0 * na + 8.0 * npix, "flops": one}
    if kind == "map2alm":
        return {"bytes": 16.0 * na + 8.0 * npix, "flops": (2 * case["iter"] + 1) * one}
    if kind == "spin":
        return {"bytes": 32.0 * na + 16.0 * npix, "flops": 4 * one}
    if kind == "convergence":
        return {"bytes": 8.0 * npix + 32.0 * npix, "flops": 7 * one + 2 * 2 * one}
    if kind == "generate":
        return {"bytes": 8.0 * S * npix, "flops": S * one}
    if kind == "shells":
        return {"bytes": 4.0 * S * npix, "flops": S * one}
    return {"bytes": 12.0 * S * npix, "flops": S * (7 * one + 2 * one)}


# ---------------------------------------------------------------------------
# the same in 64 bits


def exact(case, seed):
    kind = case["kind"]
    if kind == "generate":
        return None  # float64 maps, but of normals that the device draws in 32 bits
    if kind == "planes":
        return _exact_planes(case, seed)
    if kind == "solve":
        return _exact_solve(_target_cl(case, seed))
    nside, lmax, S = case["nside"], case["lmax"], case.get("shells", 1)
    passes = {"alm2map": 1, "spin": 2, "shells": 1, "map2alm": 2 * case.get("iter", 0) + 1,
              "convergence": 22, "shear": 24}[kind]
    # about 20 seconds: launches of the recurrences, and the rings' transforms
    if passes * (8e-5 * lmax * (lmax // 256 + 1) + 6e-8 * S * 12 * nside * nside) > 16:
        return None
    npix = 12 * nside * nside
    g = _gen(seed)
    sky = _Sky(nside, lmax)
    if kind == "alm2map":
        return sky.synth(_alm(lmax, g)[None])[0]
    if kind == "map2alm":
        f = _contrast((1, npix), g, torch.float64)
        return sky.analysis(f, torch.full((npix,), 4 * math.pi / npix, dtype=torch.float64,
                                          device="cuda"), case["iter"])[0]
    if kind == "spin":
        e, b = _alm(lmax, g), 0.1 * _alm(lmax, g)
        q, u = sky.synth_spin(e[None], b[None], case["spin"])
        return [q[0], u[0]]
    if kind == "shells":
        return _exact_shells(sky, case, seed)
    l = sky.l.double()
    if kind == "shear":
        kappa = 0.02 * _contrast((S, npix), g, torch.float32)
        alm = sky.analysis(kappa.double(), sky.weights(), 3)
        f = -torch.sqrt((l + 2) * (l + 1) * l * (l - 1).clamp(min=0)) / (l * (l + 1)).clamp(min=1)
        q, u = sky.synth_spin(alm * f, None, 2)
        return torch.stack([q, u], dim=1)
    kappa = 0.02 * _contrast((npix,), g, torch.float64)
    alm = sky.analysis(kappa[None], sky.weights(), 3)
    f = torch.where(l > 0, -2.0 / (l * (l + 1)).clamp(min=1), torch.zeros_like(l))
    q, u = sky.synth_spin(alm * f * torch.sqrt(l * (l + 1)), None, 1)
    return torch.complex(q[0], u[0]), None  # the shear depends on the pixel window


class _Sky:
    """Spherical-harmonic sums on the HEALPix rings of one (nside, lmax) in
    64 bits: alm [S, nalm] in healpy order, maps [S, npix]."""

    def __init__(self, nside, lmax):
        self.nside, self.lmax = nside, lmax
        i = np.arange(1, 4 * nside, dtype=np.int64)
        south = 4 * nside - i
        cap = np.minimum(np.minimum(i, south), nside)
        belt = (i >= nside) & (i <= 3 * nside)
        t = cap.astype(np.float64) ** 2 / (3.0 * nside * nside)
        z = np.where(belt, 2.0 * (2 * nside - i) / (3.0 * nside), np.where(i < nside, 1 - t, t - 1))
        sth = np.where(belt, np.sqrt((1 - z) * (1 + z)), np.sqrt(t * (2 - t)))
        self.n = torch.as_tensor(4 * cap).cuda()
        self.shift = torch.as_tensor(np.where(belt, 1 - ((i + nside) & 1), 1)).cuda()
        self.start = torch.cumsum(self.n, 0) - self.n
        self.x, self.sth = torch.as_tensor(z).cuda(), torch.as_tensor(sth).cuda()
        self.R, self.npix = 4 * nside - 1, 12 * nside * nside
        ch = np.sqrt(0.5 * (1 + z))  # cos and sin of theta / 2, the small one from sin theta
        sh = np.where(z > 0.5, sth / (2 * ch), np.sqrt(0.5 * (1 - z)))
        ch = np.where(z < -0.5, sth / (2 * sh), ch)
        self.log_ch = np.log2(ch.astype(np.longdouble))
        self.log_sh = np.log2(sh.astype(np.longdouble))
        k = np.arange(1, 2 * lmax + 8, dtype=np.longdouble)
        self.log_fact = np.concatenate([[np.longdouble(0)], np.cumsum(np.log2(k))])
        self.l, self.m = _hp_lm(lmax)
        M = max(32, min(256, int(2.4e10 / (8 * (lmax + 1) * self.R))))
        self.seeds = {}
        self.blocks = [(m0, min(m0 + M, lmax + 1)) for m0 in range(0, lmax + 1, M)]

    def _seed(self, m0, m1, s):
        """The functions at l0 = max(m, |s|), as p 2^(600 k), and l0."""
        mi = np.arange(m0, m1)
        a = abs(s)
        l0 = np.maximum(mi, a)
        norm = 0.5 * (np.log2((2 * l0 + 1) / np.longdouble(4 * np.pi)) + self.log_fact[2 * l0]
                      - self.log_fact[mi + a] - self.log_fact[np.abs(mi - a)])
        ps, pc = (mi + a, np.abs(mi - a)) if s >= 0 else (np.abs(mi - a), mi + a)
        e = norm[:, None] + ps[:, None] * self.log_sh + pc[:, None] * self.log_ch
        k = np.minimum(0, np.ceil(e / 600)).astype(np.int32)
        p = np.exp2(e - 600 * k).astype(np.float64)
        p *= np.where((mi >= a) | (s >= 0), (-1.0) ** mi, (-1.0) ** a)[:, None]
        return [torch.as_tensor(v).cuda() for v in (p, k, l0[:, None])]

    def wigner(self, m0, m1, s):
        """[m1 - m0, R, lmax + 1 - m0]: normalised spin-s functions of every
        ring for m0 <= m < m1 and l = m0 .. lmax, from the three-term recurrence
        in l with the scale kept apart (values below 2^-300 count as zero)."""
        a = abs(s)
        if (m0, s) not in self.seeds:
            self.seeds[m0, s] = self._seed(m0, m1, s)
        seed, k, first = self.seeds[m0, s]
        m = torch.arange(m0, m1, device="cuda", dtype=torch.float64)[:, None]
        out = torch.zeros((self.lmax + 1 - m0, m1 - m0, self.R), dtype=torch.float64,
                          device="cuda")
        p0 = torch.zeros_like(seed)
        p1 = torch.zeros_like(seed)
        for l in range(m0, self.lmax + 1):
            L = l - 1.0
            if l > 0:
                den = torch.sqrt(((l * l - m * m) * (l * l - a * a)).clamp(min=1e-30))
                A = math.sqrt((2 * L + 3) * (2 * L + 1)) * l / den
                B = m * s / max(L * l, 1.0)
                C = (math.sqrt(2 * L + 3) * l
                     * torch.sqrt(((L * L - m * m) * (L * L - a * a)).clamp(min=0))
                     / (max(L, 1.0) * math.sqrt(max(2 * L - 1, 1.0)) * den))
                p0, p1 = p1, A * (self.x + B) * p1 - C * p0
            if l <= max(m1 - 1, a):
                p1 = torch.where(first == l, seed, torch.where(first > l, 0.0, p1))
                p0 = torch.where(first >= l, 0.0, p0)
            big = (k < 0) & (p1.abs() > 2.0**300)
            p0, p1 = torch.where(big, p0 * 2.0**-600, p0), torch.where(big, p1 * 2.0**-600, p1)
            k = k + big.int()
            out[l - m0] = torch.where(k == 0, p1, 0.0)
        return out.permute(1, 2, 0).contiguous()

    def _coefficients(self, alm, m0, m1):
        """[m1 - m0, lmax + 1 - m0, 2 S] real columns (re, im) of alm, zero for l < m."""
        S, lmax = alm.shape[0], self.lmax
        c = torch.zeros((m1 - m0, lmax + 1 - m0, S), dtype=torch.complex128, device="cuda")
        for m in range(m0, m1):
            i = m * (2 * lmax + 1 - m) // 2
            c[m - m0, m - m0:] = alm[:, i + m: i + lmax + 1].T
        if m0 == 0:
            c[0] = torch.complex(c[0].real, torch.zeros_like(c[0].real))
        return torch.view_as_real(c).reshape(m1 - m0, lmax + 1 - m0, 2 * S)

    def _to_rings(self, alm, s):
        """F[m, ring, S] = sum_l lambda^s_lm(ring) a_lm."""
        S = alm.shape[0]
        F = torch.empty((self.lmax + 1, self.R, S), dtype=torch.complex128, device="cuda")
        for m0, m1 in self.blocks:
            f = torch.bmm(self.wigner(m0, m1, s), self._coefficients(alm, m0, m1))
            F[m0:m1] = torch.view_as_complex(f.reshape(m1 - m0, self.R, S, 2))
        return F

    def _chirp(self, sign, rings, rows, cols):
        """Y[ring, j] = sum_m X[ring, m] e^(sign 2 pi i m j / n), m < rows,
        j < cols, as a function of X [rings, S, rows] (Bluestein)."""
        L = 1 << (rows + cols - 2).bit_length()
        n = self.n[rings][:, None]

        def w(k):  # e^(i pi k^2 / n)
            q = (k * k) % (2 * n)
            return torch.polar(torch.ones((), dtype=torch.float64, device="cuda"),
                               sign * math.pi * q.double() / n.double())

        def go(X):
            m = torch.arange(rows, device="cuda")[None]
            j = torch.arange(cols, device="cuda")[None]
            h = torch.zeros((len(rings), L), dtype=torch.complex128, device="cuda")
            h[:, :cols] = w(j).conj()
            if rows > 1:
                h[:, L - rows + 1:] = w(torch.arange(rows - 1, 0, -1, device="cuda")[None]).conj()
            y = torch.fft.fft(X * w(m)[:, None], n=L, dim=-1)
            y = torch.fft.ifft(y * torch.fft.fft(h)[:, None], dim=-1)[..., :cols]
            return y * w(j)[:, None]
        return go

    def _ring_chunks(self, S):
        by_len = {}
        for i, n in enumerate(self.n.tolist()):
            by_len.setdefault(1 << (self.lmax + n - 1).bit_length(), []).append(i)
        for L, idx in by_len.items():
            step = max(1, int(4e9 / (16 * L * S)))
            for i in range(0, len(idx), step):
                yield torch.as_tensor(idx[i:i + step], device="cuda")

    def _phase(self, rings):
        """e^(i m phi0) [rings, lmax + 1], phi0 = pi / n or 0."""
        m = torch.arange(self.lmax + 1, device="cuda")[None]
        n = self.n[rings][:, None]
        q = (m * self.shift[rings][:, None]) % (2 * n)
        return torch.polar(torch.ones((), dtype=torch.float64, device="cuda"),
                           math.pi * q.double() / n.double())

    def _to_pixels(self, F):
        S = F.shape[-1]
        out = torch.empty((S, self.npix), dtype=torch.float64, device="cuda")
        two = torch.full((self.lmax + 1,), 2.0, dtype=torch.float64, device="cuda")
        two[0] = 1.0
        for rings in self._ring_chunks(S):
            X = F[:, rings].permute(1, 2, 0) * (self._phase(rings) * two)[:, None]
            X[..., 0] = X[..., 0].real.to(torch.complex128)
            cols = int(self.n[rings].max())
            y = self._chirp(1, rings, self.lmax + 1, cols)(X).real
            ok, at = self._pixels(rings, cols)
            out[:, at] = y.permute(1, 0, 2)[:, ok]
        return out

    def _pixels(self, rings, cols):
        j = torch.arange(cols, device="cuda")[None]
        ok = j < self.n[rings][:, None]
        return ok, (self.start[rings][:, None] + j)[ok]

    def synth(self, alm):
        return self._to_pixels(self._to_rings(alm, 0))

    def synth_spin(self, E, B, s):
        lp = self._to_rings(E if B is None else torch.cat([E, B]), s)
        lm = self._to_rings(E if B is None else torch.cat([E, B]), -s)
        sg, S = (-1.0) ** s, E.shape[0]
        fp, fm = -0.5 * (lp + sg * lm), -0.5 * (lp - sg * lm)
        q, u = fp[..., :S], -1j * fm[..., :S]
        if B is not None:
            q, u = q + 1j * fm[..., S:], u + fp[..., S:]
        return self._to_pixels(q), self._to_pixels(u)

    def adjoint(self, f):
        """sum_p f_p Y*_lm(p) of maps [S, npix]."""
        S = f.shape[0]
        G = torch.empty((self.lmax + 1, self.R, S), dtype=torch.complex128, device="cuda")
        for rings in self._ring_chunks(S):
            cols = int(self.n[rings].max())
            ok, at = self._pixels(rings, cols)
            X = torch.zeros((S, len(rings), cols), dtype=torch.float64, device="cuda")
            X[:, ok] = f[:, at]
            y = self._chirp(-1, rings, cols, self.lmax + 1)(X.permute(1, 0, 2))
            G[:, rings] = (y * self._phase(rings).conj()[:, None]).permute(2, 0, 1)
        out = torch.empty((S, self.l.numel()), dtype=torch.complex128, device="cuda")
        for m0, m1 in self.blocks:
            lam = self.wigner(m0, m1, 0).transpose(1, 2).contiguous()
            g = torch.view_as_real(G[m0:m1]).reshape(m1 - m0, self.R, 2 * S)
            a = torch.view_as_complex(torch.bmm(lam, g).reshape(m1 - m0, -1, S, 2))
            for m in range(m0, m1):
                i = m * (2 * self.lmax + 1 - m) // 2
                out[:, i + m: i + self.lmax + 1] = a[m - m0, m - m0:].T
        return torch.where(self.m == 0, out.real.to(torch.complex128), out)

    def analysis(self, f, w, niter):
        alm = self.adjoint(f * w)
        for _ in range(niter):
            alm = alm + self.adjoint((f - self.synth(alm)) * w)
        return alm

    def weights(self):
        """The smallest correction of the uniform pixel weights with
        sum_p w_p Y*_lm(p) = sqrt(4 pi) delta_l0 for l <= 2 nside."""
        sky = self if self.lmax == 2 * self.nside else _Sky(self.nside, 2 * self.nside)
        two = torch.where(sky.m == 0, 1.0, 2.0).double()

        def dot(a, b):
            return float((two * (a.conj() * b).real).sum())

        w0 = torch.full((1, sky.npix), 4 * math.pi / sky.npix, dtype=torch.float64, device="cuda")
        r = -sky.adjoint(w0)[0]
        r[0] += math.sqrt(4 * math.pi)
        lam, p, rr = torch.zeros_like(r), r.clone(), dot(r, r)
        stop = 1e-26 * rr
        for _ in range(30):
            q = sky.adjoint(sky.synth(p[None]))[0]
            a = rr / dot(p, q)
            lam, r = lam + a * p, r - a * q
            new = dot(r, r)
            if new <= stop:
                break
            p, rr = r + (new / rr) * p, new
        return (w0 + sky.synth(lam[None]))[0]


def _philox(g, u, seed):
    """Philox4x32-10 words of counter (g, u) under the key seed."""
    mask = 0xFFFFFFFF
    c = [g & mask, g >> 32, torch.full_like(g, u & mask), torch.full_like(g, u >> 32)]
    k0, k1 = seed & mask, seed >> 32
    for _ in range(10):
        hi, lo = [], []
        for mul, v in ((0xD2511F53, c[0]), (0xCD9E8D57, c[2])):
            low, high = mul * (v & 0xFFFF), mul * (v >> 16)
            t = (low >> 16) + high
            hi.append(t >> 16)
            lo.append(((t & 0xFFFF) << 16) | (low & 0xFFFF))
        c = [hi[1] ^ c[1] ^ k0, lo[1], hi[0] ^ c[3] ^ k1, lo[0]]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    return c


def _exact_shells(sky, case, seed):
    """The lognormal shells from the generator's words: Box-Muller, the
    conditional weights of each mode from its covariance matrix, synthesis."""
    S, k, nl = case["shells"], case["ncorr"], case["lmax"] + 1
    gls = _gls(case, seed)
    g = sky.l * (sky.l + 1) // 2 + sky.m

    def pair(t):
        w = _philox(g, t >> 1, seed)
        w0, w1 = (w[2], w[3]) if t & 1 else (w[0], w[1])
        u1 = ((w0.float() + 0.5) * 2.0**-32).double()
        u2 = (w1 >> 8).double() * 2.0**-24
        return torch.polar(torch.sqrt(-2.0 * torch.log(u1)), 2 * math.pi * u2)

    def cl(i, j):
        c = np.zeros(nl)
        h = gls[i * (i + 1) // 2 + i - j]
        c[: len(h)] = h
        return torch.as_tensor(c).cuda() / 2

    alm = torch.empty((S, sky.l.numel()), dtype=torch.complex128, device="cuda")
    # state per mode: M with M C M^T = 1 for the last k fields (zero rows before the first)
    M = torch.zeros((nl, k, k), dtype=torch.float64, device="cuda")
    a = torch.zeros((nl, k), dtype=torch.float64, device="cuda")
    sd = torch.ones(nl, dtype=torch.float64, device="cuda")
    z = []
    for t in range(S):
        if t > 0 and k:
            div = torch.where(sd > 0, sd, 1.0)
            row = torch.cat([-(a[:, None] @ M)[:, 0], (sd > 0).double()[:, None]], 1) / div[:, None]
            M = torch.cat([torch.cat([M, M.new_zeros((nl, k, 1))], 2), row[:, None]], 1)[:, 1:, 1:]
        past = [cl(t, t - d) if t - d >= 0 else torch.zeros_like(sd) for d in range(k, 0, -1)]
        a = (M @ torch.stack(past, 1)[:, :, None])[..., 0] if k else a
        sd = torch.sqrt((cl(t, t) - (a * a).sum(1)).clamp(min=0))
        z = (z + [pair(t)])[-(k + 1):]
        w = torch.cat([a, sd[:, None]], 1)[:, k + 1 - len(z):]
        x = sum(w[sky.l, j] * zj for j, zj in enumerate(z))
        alm[t] = torch.where(sky.m == 0, (x.real + x.imag).to(torch.complex128), x)
    l = np.arange(nl)
    var = [float(np.sum((2 * l + 1) * gls[i * (i + 1) // 2]) / (4 * np.pi)) for i in range(S)]
    x = sky.synth(alm)
    return torch.expm1(x - torch.as_tensor(var).cuda()[:, None] / 2)


def _exact_planes(case, seed):
    g = _gen(seed)
    dtype = torch.float32 if case["bits"] == 32 else torch.float64
    npix, n, c = 12 * case["nside"] ** 2, case["shells"], _Cosmology()
    deltas = [_contrast((npix,), g, dtype) for _ in range(n)]
    z = np.concatenate([[0.0], 0.1 * (np.arange(n) + 1)])
    kappa = torch.zeros(npix, dtype=torch.float64, device="cuda")
    for i in range(n - 1):  # the Born sum: each plane's weight at the last source
        f = (1.5 * c.Omega_m0 * (1 + z[i + 1]) / c.H_over_H0(z[i + 1]) * 0.1
             * c.transverse_comoving_distance(z[i + 1])
             * c.transverse_comoving_distance(z[i + 1], z[n])
             / c.transverse_comoving_distance(z[n]))
        kappa += float(f) * deltas[i].double()
    return kappa


def _legendre_pair(n):
    """C_l <-> C(theta) on n Gauss-Legendre nodes as matrix products."""
    i = torch.arange(1, n + 1, dtype=torch.float64, device="cuda")
    x = -torch.cos(math.pi * (i - 0.25) / (n + 0.5))

    def value(x):
        p0, p1 = torch.ones_like(x), x.clone()
        for k in range(2, n + 1):
            p0, p1 = p1, ((2 * k - 1) * x * p1 - (k - 1) * p0) / k
        d = n * (x * p1 - p0) / (x * x - 1)
        return p1, d
    for _ in range(3):
        p, d = value(x)
        x = x - p / d
    w = 2 / ((1 - x * x) * value(x)[1] ** 2)
    P = torch.empty((n, n), dtype=torch.float64, device="cuda")
    P[0] = 1.0
    P[1:2] = x
    for k in range(2, n):
        P[k] = ((2 * k - 1) * x * P[k - 1] - (k - 1) * P[k - 2]) / k
    c = (2 * _ell(n - 1) + 1) / (4 * math.pi)
    return (lambda cl: (c * cl) @ P), (lambda xi: 2 * math.pi * (P @ (w * xi)))


def _exact_solve(cl):
    """The solver's iteration for a lognormal field of unit scale (no monopole)."""
    n = len(cl)
    cl = torch.as_tensor(cl).cuda()
    to_xi, to_cl = _legendre_pair(n)
    gl = to_cl(torch.log1p(to_xi(cl)))
    to_xi, to_cl = _legendre_pair(3 * n)

    def pad(v):
        return torch.nn.functional.pad(v, (0, 2 * n))

    def relerr(d, v):
        return float(torch.where(d != 0, d / v, torch.zeros_like(d)).abs().max())

    gt = to_xi(pad(gl))
    rl = to_cl(torch.expm1(gt))
    fl = rl[:n] - cl
    err, info = relerr(fl, cl), 0
    for _ in range(20):
        info |= err <= 1e-5
        if info:
            break
        xl = -to_cl(to_xi(pad(fl)) / torch.exp(gt))[:n]
        while True:
            new = gl + xl
            gt_ = to_xi(pad(new))
            rl_ = to_cl(torch.expm1(gt_))
            fl_ = rl_[:n] - cl
            err_ = relerr(fl_, cl)
            if err_ <= err:
                break
            xl = xl / 2
        info |= 2 * (relerr(xl, gl) <= 1e-5)
        gl, gt, rl, fl, err = new, gt_, rl_, fl_, err_
    return {"gl": gl, "cl": rl, "info": int(info)}
