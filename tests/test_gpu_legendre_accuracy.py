"""Rounding errors of the FP64 Legendre stages: those of the recurrence
lambda_l = a (x lambda_{l-1} - b lambda_{l-2}) with one fused multiply-add, coefficients a
and b rounded once and seeds by repeated squaring, restated here in double
precision.  Both against values in
extended precision (the 64-bit mantissa of numpy's long double) at the same cos(theta),
on a sample of rings from the pole to the equator, each ring counting by its
number of pixels, as in the RMS over a map.

A tenth is allowed for the sampling and for the other roundings (the sums and the
ring transforms, a few 1e-16).  In the same restatement the normalised form with
coefficients from double products has 1.2 to 1.6 times this error."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from glass_amd import healpix as hp  # noqa: E402

X = np.longdouble
PI = 4 * np.arctan(X(1))


def rings(nside):
    """(first pixel, pixels, cos, sin, phi0 in units of pi / pixels) of the north
    rings, the equator last"""
    r = np.arange(1, 2 * nside + 1)
    t = (r * r) / (3.0 * (nside * nside))
    z = np.where(r < nside, 1 - t, (2 * nside - r) * 2.0 / (3.0 * nside))
    s = np.where(r < nside, np.sqrt(t * (2 - t)), np.sqrt((1 - z) * (1 + z)))
    n = np.minimum(4 * r, 4 * nside)
    start = np.where(r < nside, 2 * r * (r - 1), 2 * nside * (nside - 1) + (r - nside) * 4 * nside)
    shift = np.where(r < nside, 1, 1 - ((r + nside) & 1))
    return start, n, z, s, shift


def fma(a, b, c):
    return (a.astype(X) * b + c).astype(np.float64)


def sin_power(s, m):
    """sin^m in double precision by repeated squaring, as mantissa and exponent"""
    b, eb = np.frexp(s)
    r, er = np.ones_like(s), np.zeros(len(s), int)
    while m:
        if m & 1:
            r, t = np.frexp(r * b)
            er += eb + t
        m >>= 1
        if m:
            b, t = np.frexp(b * b)
            eb = 2 * eb + t
    return r, er


def rows(lmax, z, s, dtype):
    """lambda_lm at the rings for l = 0, 1, ...: arrays [m <= l, ring]; the double
    recurrence starts from sin^m by repeated squaring"""
    m = np.arange(lmax + 1)
    k = np.arange(1, lmax + 1, dtype=X)
    prod = np.concatenate([[X(1)], np.cumprod((2 * k - 1) / (2 * k))])
    cm = ((-1.0) ** m * np.sqrt((2 * m.astype(X) + 1) / (4 * PI) * prod)).astype(np.float64)
    if dtype is X:
        seed = cm[:, None] * s.astype(X) ** m[:, None]
    else:
        pw = [sin_power(s, int(i)) for i in m]
        seed = np.array([np.ldexp(c * r, e) for c, (r, e) in zip(cm, pw)])
    x = z.astype(dtype)[None, :]
    p0, p1 = np.zeros((2, lmax + 1, len(z)), dtype)
    for l in range(lmax + 1):
        if l:
            t, mm = dtype(l), m[:l].astype(dtype)
            a = np.sqrt((4 * t * t - 1) / (t * t - mm * mm))[:, None]
            b = np.sqrt(((t - 1) ** 2 - mm * mm) / (4 * (t - 1) ** 2 - 1))[:, None] if l > 1 else x * 0
            if dtype is X:
                y = a * (x * p1[:l] - b * p0[:l])
            else:
                y = a * fma(x, p1[:l], -(b * p0[:l]))
            p0[:l] = p1[:l]
            p1[:l] = y
        p1[l] = seed[l]
        yield l, p1[: l + 1]


def sample(nside, rng):
    """up to 48 rings from the pole to the equator, and 16 pixels (with repeats) on
    each and on its mirror"""
    start, n, z, s, shift = rings(nside)
    sel = np.unique(np.linspace(0, 2 * nside - 2, 48).astype(int))
    start, n, z, s, shift = (v[sel] for v in (start, n, z, s, shift))
    j = rng.integers(0, n[:, None], (len(sel), 16))
    south = 12 * nside * nside - start - n
    return n, z, s, shift, j, start[:, None] + j, south[:, None] + j


def phases(lmax, n, shift, j):
    """cos and sin of m phi: [m, ring, pixel]"""
    q = (np.arange(lmax + 1)[:, None, None] * (2 * j + shift[:, None])) % (2 * n[:, None])
    a = PI * q.astype(X) / n[:, None]
    return np.cos(a), np.sin(a)


def rms(a, weight=1.0):
    return float(np.sqrt(np.mean(weight * np.abs(a) ** 2)))


CASES = [(16, 300), (64, 700), (200, 600), (512, 1030)]  # the last with two ring pairs a lane


def synthesis(nside, lmax, lam=rows):
    """(alm, pixels, their weights, exact map there, map from the double recurrence)"""
    rng = np.random.default_rng(nside + lmax)
    n, z, s, shift, j, pn, ps = sample(nside, rng)
    c, sn = phases(lmax, n, shift, j)
    # real alm, healpy order (the imaginary parts go through the same sums)
    cols = [rng.standard_normal(l + 1) for l in range(lmax + 1)]
    alm = np.zeros((lmax + 1) * (lmax + 2) // 2, np.complex128)
    m = np.arange(lmax + 1)
    for l, v in enumerate(cols):
        alm[m[: l + 1] * (2 * lmax + 1 - m[: l + 1]) // 2 + l] = v
    maps = []
    for dtype in (X, np.float64):
        F = np.zeros((2, lmax + 1, len(n)), dtype)  # by the parity of l - m
        for l, v in lam(lmax, z, s, dtype):
            par = (l - np.arange(l + 1)) & 1
            for p in (0, 1):
                F[p, : l + 1][par == p] += v[par == p] * cols[l][par == p, None]
        e, o = F.astype(X)
        e[1:] *= 2
        o[1:] *= 2
        maps.append(np.stack([((e + o)[:, :, None] * c).sum(0), ((e - o)[:, :, None] * c).sum(0)]))
    return alm, np.stack([pn, ps]), n[None, :, None], maps[0], maps[1]


def analysis(nside, lmax, lam=rows):
    """(map, exact alm, alm from the double recurrence)"""
    rng = np.random.default_rng(nside + 7 * lmax)
    n, z, s, shift, j, pn, ps = sample(nside, rng)
    c, sn = phases(lmax, n, shift, j)
    f = np.zeros(12 * nside * nside)
    vals = rng.standard_normal((2,) + j.shape) * np.sqrt(n)[:, None]
    keep = np.ones(j.shape, bool)  # one value per pixel
    for r in range(len(n)):
        keep[r] = False
        keep[r, np.unique(j[r], return_index=True)[1]] = True
    vals *= keep
    for p, v in zip((pn, ps), vals):
        f[p[keep]] = v[keep]
    w = 4 * PI / (12 * nside * nside)
    north, south = (w * ((v * c).sum(-1) - 1j * (v * sn).sum(-1)) for v in vals.astype(X))
    q = (north + south, north - south)
    alms = []
    m = np.arange(lmax + 1)
    for dtype in (X, np.float64):
        alm = np.zeros((lmax + 1) * (lmax + 2) // 2, np.clongdouble)
        for l, v in lam(lmax, z, s, dtype):
            par = (l - np.arange(l + 1)) & 1
            t = np.where(par[:, None], q[1][: l + 1], q[0][: l + 1])
            alm[m[: l + 1] * (2 * lmax + 1 - m[: l + 1]) // 2 + l] = (v.astype(X) * t).sum(-1)
        alms.append(alm)
    return f, alms[0], alms[1]


@pytest.mark.parametrize("nside,lmax", CASES)
def test_synthesis_error(nside, lmax):
    alm, pix, wt, exact, plain = synthesis(nside, lmax)
    got = hp.alm2map(torch.as_tensor(alm).cuda(), nside, lmax=lmax, pol=False).cpu().numpy()[pix]
    err, ref = (rms(v - exact, wt) / rms(exact, wt) for v in (got, plain))
    print(f"synthesis nside={nside} lmax={lmax}: {err:.2e}, recurrence in (a, b) {ref:.2e}")
    assert err <= 1.1 * ref


@pytest.mark.parametrize("nside,lmax", CASES)
def test_analysis_error(nside, lmax):
    f, exact, plain = analysis(nside, lmax)
    got = hp.map2alm(torch.as_tensor(f).cuda(), lmax=lmax, iter=0, pol=False).cpu().numpy()
    err, ref = (rms(v - exact) / rms(exact) for v in (got, plain))
    print(f"analysis nside={nside} lmax={lmax}: {err:.2e}, recurrence in (a, b) {ref:.2e}")
    assert err <= 1.1 * ref
