"""The FP64 Legendre stages where their loops change shape: band limits around
a whole number of chunks of rows, ring-pair counts around whole waves, fewer
rows than the spin, and m so large that the polar rings' values start
thousands of binary orders below one.

Tolerance: one FP64 recurrence step perturbs a value by a few ulp, and the
perturbations of lmax steps add, so max |error| / RMS of the oracle's result
stays below 64 (lmax + 1) 2^-52.
"""

import ctypes

import numpy as np
import pytest
import torch
from scipy.special import eval_legendre

from oracle import oracle as O

pytestmark = pytest.mark.gpu

from glass_amd import _lib  # noqa: E402
from glass_amd import healpix as hp  # noqa: E402


def rand_alm(lmax, rng):
    n = O.nalm(lmax)
    return rng.standard_normal(n) + 1j * rng.standard_normal(n)


def bound(lmax):
    return 64 * (lmax + 1) * 2.0**-52


@pytest.mark.parametrize("spin", [1, 2])
@pytest.mark.parametrize("nside,lmax", [(1, 1), (1, 2), (3, 6), (5, 7), (16, 8), (31, 15), (33, 17),
                                        (96, 64), (130, 41), (40, 600)])
def test_spin_synthesis_edges(spin, nside, lmax):
    print(f"spin={spin} nside={nside} lmax={lmax}", flush=True)
    rng = np.random.default_rng(1000 * nside + 10 * lmax + spin)
    E, B = rand_alm(lmax, rng), rand_alm(lmax, rng)
    rq, ru = O.alm2map_spin([E, B], nside, spin, lmax, nthreads=4)
    q, u = hp.alm2map_spin([E, B], nside, spin, lmax)
    scale = np.sqrt(np.mean(rq**2 + ru**2))
    if scale == 0:  # lmax < spin: nothing to synthesise
        assert not q.any() and not u.any()
        return
    assert np.max(np.abs(q - rq)) / scale < bound(lmax)
    assert np.max(np.abs(u - ru)) / scale < bound(lmax)


# npairs = 2 nside: one wave (<= 64 pairs), two to four waves, two / four / eight
# pairs per lane (from 257, 513, 1025 pairs), two workgroups for each m (2060)
@pytest.mark.parametrize("nside,lmax,niter", [(1, 0, 0), (1, 4, 1), (32, 14, 0), (33, 15, 1),
                                              (100, 16, 0), (128, 31, 0), (129, 33, 1),
                                              (257, 47, 0), (513, 40, 0), (1030, 20, 1),
                                              (40, 600, 0)])
def test_analysis_edges(nside, lmax, niter):
    print(f"analysis nside={nside} lmax={lmax} niter={niter}", flush=True)
    rng = np.random.default_rng(nside + 7 * lmax)
    f = rng.standard_normal(12 * nside * nside)
    ref = O.map2alm(f, lmax, niter=niter, nthreads=8)
    got = hp.map2alm(f, lmax=lmax, iter=niter)
    assert np.max(np.abs(got - ref)) / np.sqrt(np.mean(np.abs(ref) ** 2)) < bound(lmax)


# the plain form (few waves), the normalised one with two ring pairs per lane
# (at least 16384 waves: nside 512, lmax 1030 and nside 520, lmax 1023 with a
# part-filled last wave), and no room in the map for the scaled alm (lmax 600
# at nside 40)
@pytest.mark.parametrize("nside,lmax", [(1, 0), (1, 6), (2, 7), (33, 8), (64, 15), (65, 16),
                                        (40, 600), (512, 1030), (520, 1023)])
def test_synthesis_edges(nside, lmax):
    print(f"synthesis nside={nside} lmax={lmax}", flush=True)
    rng = np.random.default_rng(3 * nside + lmax)
    alm = rand_alm(lmax, rng)
    ref = O.alm2map(alm, nside, nthreads=8)
    got = hp.alm2map(alm, nside)
    assert np.max(np.abs(got - ref)) / np.sqrt(np.mean(ref**2)) < bound(lmax)


def test_synthesis_longest_rings():
    """Rings of more than 4 * 2048 pixels (eight values of a thread), both for
    a power of two and for Bluestein lengths above 4096."""
    nside, lmax = 2100, 12
    rng = np.random.default_rng(5)
    alm = rand_alm(lmax, rng)
    got = hp.alm2map(alm, nside)
    first, step = 1, 419  # a sample of rings through the oracle
    ref = O.alm2map_rings(alm, nside, first, step, nthreads=8)
    sel = ref != 0
    assert sel.sum() > nside
    err = np.max(np.abs(got[sel] - ref[sel])) / np.sqrt(np.mean(ref[sel] ** 2))
    assert err < bound(lmax)


@pytest.mark.parametrize("nl,n", [(1, 64), (2, 3), (16, 65), (33, 63), (64, 64), (65, 130), (97, 40),
                                  (200, 129)])
def test_transforms_of_unequal_lengths(nl, n):
    """nl coefficients on n nodes around whole batches of rows (16, 32, 64) and
    whole waves of nodes, against direct sums over scipy's Legendre
    polynomials; tolerance: nl steps of a few ulp, 16 nl 2^-52 of the sum of
    absolute terms."""
    rng = np.random.default_rng(nl * 1000 + n)
    x = np.sort(rng.uniform(-1, 1, n))
    w, cl, corr = rng.uniform(0, 1, n), rng.standard_normal(nl), rng.standard_normal(n)
    P = np.array([eval_legendre(l, x) for l in range(nl)])
    dev = [torch.as_tensor(v).cuda() for v in (x, w, cl, corr)]
    out_c = torch.empty(n, dtype=torch.float64, device="cuda")
    out_l = torch.empty(nl, dtype=torch.float64, device="cuda")
    _lib.call("ga_cl2corr", nl, _lib.ptr(dev[2]), n, _lib.ptr(dev[0]), _lib.ptr(out_c),
              _lib.stream_ptr())
    nb = ctypes.c_size_t()
    _lib.call("ga_corr2cl_workspace_size", n, nl, ctypes.byref(nb))
    ws = _lib.workspace(nb.value)
    _lib.call("ga_corr2cl", n, _lib.ptr(dev[0]), _lib.ptr(dev[1]), _lib.ptr(dev[3]), nl,
              _lib.ptr(out_l), _lib.ptr(ws), ws.numel(), _lib.stream_ptr())
    f = (2 * np.arange(nl) + 1) / (4 * np.pi) * cl
    assert np.all(np.abs(out_c.cpu().numpy() - f @ P) <= 16 * nl * 2.0**-52 * np.sum(np.abs(f)))
    g = 2 * np.pi * w * corr
    assert np.all(np.abs(out_l.cpu().numpy() - P @ g) <= 16 * nl * 2.0**-52 * np.sum(np.abs(g)))


@pytest.mark.parametrize("k", range(9))
def test_iternorm_row_lengths(k):
    """Every row length of the register form (k <= 7) and the first of the
    general one, in two calls that hand the state over, for 1 and 70 modes."""
    rng = np.random.default_rng(k)
    n = 2 * k + 5
    for nl in (1, 70):
        a = rng.standard_normal((nl, n, n + 3))
        full = a @ a.transpose(0, 2, 1) / (n + 3) + np.eye(n)
        rows = np.zeros((n, nl, k + 1))
        for t in range(n):
            for d in range(min(k, t) + 1):
                rows[t, :, d] = full[:, t, t - d] * (1.0 if d == 0 else 0.5**d)
        ref = list(O.iternorm(list(rows)))
        m = ctypes.c_int32()
        _lib.call("ga_iternorm_state_doubles", k, ctypes.byref(m))
        state = torch.empty(nl * m.value, dtype=torch.float64, device="cuda")
        flag = torch.zeros(1, dtype=torch.int32, device="cuda")
        cov = torch.as_tensor(rows).cuda()
        w = torch.empty_like(cov)
        for lo, hi in ((0, k + 2), (k + 2, n)):
            _lib.call("ga_iternorm_batch", nl, k, k, k, hi - lo, int(lo == 0), _lib.ptr(cov[lo]),
                      _lib.ptr(state), _lib.ptr(w[lo]), _lib.ptr(flag), _lib.stream_ptr())
        assert not int(flag.item())
        np.testing.assert_allclose(w.cpu().numpy(), np.array(ref), rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("nl", [1, 2, 3, 64, 257, 1500])
def test_alm_order(nl):
    """(l, m) of every healpy index: the reordered index itself comes back."""
    g = np.arange(nl * (nl + 1) // 2)
    a = torch.as_tensor(g.astype(np.complex128)).cuda()
    out = torch.empty_like(a)
    _lib.call("ga_glass_to_healpix_alm_f64", nl, _lib.ptr(a), _lib.ptr(out), _lib.stream_ptr())
    ref = np.concatenate([np.arange(m, nl) * (np.arange(m, nl) + 1) // 2 + m for m in range(nl)])
    np.testing.assert_array_equal(out.cpu().numpy().real, ref)


@pytest.mark.parametrize("S,offset,path", [(1, 0, 0), (3, 0, 0), (4, 1, 0), (5, 2, 0), (3, 0, 1)])
def test_weighted_batch_analysis_routes(S, offset, path):
    """Weights in the ring stage's load (16-byte aligned maps, register form) and
    in a pass of their own (maps off by one or two floats; the first ring form)
    against the FP64 analysis of the same maps."""
    nside, lmax, niter = 24, 48, 1
    npix = 12 * nside * nside
    rng = np.random.default_rng(S + offset)
    maps = rng.standard_normal((S, npix)).astype(np.float32)
    buf = torch.empty(S * npix + 4, dtype=torch.float32, device="cuda")
    d = buf[offset:offset + S * npix]
    d.copy_(torch.as_tensor(maps.reshape(-1)))
    w = hp.pixel_weights(nside)
    plan = _lib.get_plan(nside, lmax)
    plan.set_tuning(_lib.TUNE_RING_PATH, path)
    try:
        ws = _lib.workspace(plan.workspace_bytes(S, 4, analysis=True))
        tmp = torch.empty(S * npix, dtype=torch.float32, device="cuda")
        alm = torch.empty((O.nalm(lmax), S), dtype=torch.complex64, device="cuda")
        _lib.call("ga_map2alm_weighted_batch_f32", plan.h, S, _lib.ptr(d), _lib.ptr(w),
                  _lib.ptr(alm), niter, _lib.ptr(tmp), _lib.ptr(ws), ws.numel(),
                  _lib.stream_ptr())
    finally:
        plan.set_tuning(_lib.TUNE_RING_PATH, 0)
    got = alm.cpu().numpy()
    for s in range(S):
        ref = O.map2alm_weighted(maps[s].astype(np.float64), w.cpu().numpy(), lmax, niter)
        err = np.max(np.abs(got[:, s] - ref)) / np.sqrt(np.mean(np.abs(ref) ** 2))
        assert err < 1e-5  # the FP32 path's target, as in the other tests
