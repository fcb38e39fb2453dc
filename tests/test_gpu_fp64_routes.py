"""Routes of the FP64 transforms that sizes alone do not reach: memory that the
normalised synthesis may not use as its scratch, and the longest rings.

Tolerance: as for the stages, 64 (lmax + 1) 2^-52 of the RMS."""

import numpy as np
import pytest
import torch
from test_gpu_legendre_accuracy import PI, X, phases, rings, rows

from oracle import oracle as O

pytestmark = pytest.mark.gpu

from glass_amd import _lib  # noqa: E402
from glass_amd import healpix as hp  # noqa: E402


def bound(lmax):
    return 64 * (lmax + 1) * 2.0**-52


def alm2map(plan, alm, out):
    ws = _lib.workspace(plan.workspace_bytes(1, 8))
    _lib.call("ga_alm2map_f64", plan.h, _lib.ptr(alm), _lib.ptr(out), _lib.ptr(ws), ws.numel(),
              _lib.stream_ptr())


def random_alm(lmax, rng):
    n = (lmax + 1) * (lmax + 2) // 2
    alm = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    alm[: lmax + 1] = alm[: lmax + 1].real
    return alm


def test_alm_larger_than_the_map():
    """Enough waves for the normalised form (4096 values of m, four waves each), but
    16.8 million doubles of alm against a map of 196608: nothing is written
    around the map."""
    nside, lmax, room = 128, 4095, 1 << 16
    npix = 12 * nside * nside
    alm = random_alm(lmax, np.random.default_rng(1))
    buf = torch.full((npix + 2 * room,), 7.0, dtype=torch.float64, device="cuda")
    out = buf[room:room + npix]
    alm2map(_lib.get_plan(nside, lmax), torch.as_tensor(alm).cuda(), out)
    assert (buf[:room] == 7.0).all() and (buf[room + npix:] == 7.0).all()
    ref = O.alm2map_rings(alm, nside, 3, 37, nthreads=8)
    sel = ref != 0
    got = out.cpu().numpy()[sel]
    assert np.max(np.abs(got - ref[sel])) / np.sqrt(np.mean(ref[sel] ** 2)) < bound(lmax)


@pytest.mark.parametrize("where", ["inside", "over the end", "over the start", "apart"])
def test_alm_and_map_in_one_buffer(where):
    """The alm may lie in the memory of the map: they are read before it is
    written, and the map is no scratch then."""
    nside, lmax = 512, 1030
    npix, nalm = 12 * nside * nside, (lmax + 1) * (lmax + 2) // 2
    first = 2 * nalm + 64  # of the map
    start = {"inside": first + 1000, "over the end": first + npix - nalm,
             "over the start": first - nalm, "apart": 0}[where]
    alm = torch.as_tensor(random_alm(lmax, np.random.default_rng(2))).cuda()
    plan = _lib.get_plan(nside, lmax)
    ref = torch.empty(npix, dtype=torch.float64, device="cuda")
    alm2map(plan, alm, ref)
    buf = torch.zeros(first + npix + 2 * nalm, dtype=torch.float64, device="cuda")
    buf[start:start + 2 * nalm] = torch.view_as_real(alm).reshape(-1)
    alm2map(plan, buf[start:], buf[first:first + npix])
    got = buf[first:first + npix]
    if where == "apart":
        assert torch.equal(got, ref)
    else:
        assert float((got - ref).abs().max() / ref.square().mean().sqrt()) < bound(lmax)


def some_rings(nside, rng):
    """rings at the borders of the kernels' lengths, with 16 pixels of each and of
    its mirror"""
    start, n, z, s, shift = rings(nside)
    want = [0, 1, 2, 63, 1023, 1024, 2046, 2047, 2048, 2049, nside - 2, nside - 1, nside, 2 * nside - 2]
    sel = np.unique([r for r in want if r < 2 * nside - 1])
    start, n, z, s, shift = (v[sel] for v in (start, n, z, s, shift))
    j = np.array([rng.permutation(min(int(k), 4096))[:16] if k >= 16 else np.resize(np.arange(k), 16)
                  for k in n])
    j[n >= 32, 1] = n[n >= 32] - 1  # the last pixel
    south = 12 * nside * nside - start - n
    return n, z, s, shift, j, start[:, None] + j, south[:, None] + j


@pytest.mark.parametrize("nside", [2048, 2100, 4096])
def test_synthesis_of_the_longest_rings(nside):
    """Power-of-two rings up to r = 4096 (nside 4096) and Bluestein rings of transform
    length 8192 (2048 < r < 4096)."""
    lmax = 12
    rng = np.random.default_rng(nside)
    n, z, s, shift, j, pn, ps = some_rings(nside, rng)
    c, sn = phases(lmax, n, shift, j)
    alm = random_alm(lmax, rng)
    m = np.arange(lmax + 1)
    F = np.zeros((2, lmax + 1, len(n)), np.clongdouble)
    for l, v in rows(lmax, z, s, X):
        a = alm[m[: l + 1] * (2 * lmax + 1 - m[: l + 1]) // 2 + l]
        for p in (0, 1):
            on = (l - m[: l + 1]) % 2 == p
            F[p, : l + 1][on] += v[on] * a[on, None]
    F[:, 1:] *= 2
    north, south = F[0] + F[1], F[0] - F[1]
    ref = np.stack([(f.real[:, :, None] * c - f.imag[:, :, None] * sn).sum(0) for f in (north, south)])
    out = hp.alm2map(torch.as_tensor(alm).cuda(), nside, lmax=lmax, pol=False)
    got = out[torch.as_tensor(np.stack([pn, ps])).cuda()].cpu().numpy()
    assert np.max(np.abs(got - ref)) / np.sqrt(float(np.mean(ref**2))) < bound(lmax)


@pytest.mark.parametrize("nside", [2048, 2100, 2482])
def test_analysis_of_the_longest_rings(nside):
    lmax = 12
    rng = np.random.default_rng(nside)
    n, z, s, shift, j, pn, ps = some_rings(nside, rng)
    c, sn = phases(lmax, n, shift, j)
    first = np.array([[v not in row[:i] for i, v in enumerate(row)] for row in j.tolist()])
    vals = rng.standard_normal((2,) + j.shape) * first
    f = torch.zeros(12 * nside * nside, dtype=torch.float64, device="cuda")
    for p, v in zip((pn, ps), vals):
        f[torch.as_tensor(p[first]).cuda()] = torch.as_tensor(v[first]).cuda()
    w = 4 * PI / (12 * nside * nside)
    north, south = (w * ((v * c).sum(-1) - 1j * (v * sn).sum(-1)) for v in vals.astype(X))
    m = np.arange(lmax + 1)
    ref = np.zeros((lmax + 1) * (lmax + 2) // 2, np.clongdouble)
    for l, v in rows(lmax, z, s, X):
        sign = np.where((l - m[: l + 1]) % 2, -1, 1)[:, None]
        ref[m[: l + 1] * (2 * lmax + 1 - m[: l + 1]) // 2 + l] = (
            v * (north[: l + 1] + sign * south[: l + 1])).sum(-1)
    got = hp.map2alm(f, lmax=lmax, iter=0, pol=False).cpu().numpy()
    err = np.max(np.abs(got - ref)) / float(np.sqrt(np.mean(np.abs(ref) ** 2)))
    assert err < bound(lmax)


def test_analysis_above_its_limit_is_refused():
    f = torch.zeros(12 * 2483 * 2483, dtype=torch.float64, device="cuda")
    with pytest.raises(NotImplementedError):
        hp.map2alm(f, lmax=4, iter=0, pol=False)
