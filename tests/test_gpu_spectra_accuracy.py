"""Rounding errors of the Legendre sums: no larger than those of the textbook
recurrence l P_l = (2l - 1) x P_{l-1} - (l - 1) P_{l-2} in double precision, whose
coefficients are exact and which divides in every step.  Both against sums in
extended precision on the same nodes, coefficients of equal variance.  (The
difference form of the kernels is ten times below and more; rows with rounded
coefficients (2l - 1) / l and (l - 1) / l are above at these sizes.)"""

import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from glass_amd import _lib  # noqa: E402


def sums(nl, x, f, g, dtype):
    """sum_l f_l P_l(x_k) and sum_k g_k P_l(x_k)"""
    x = x.astype(dtype)
    p0, p1 = np.ones_like(x), x.copy()
    corr, cl = f[0] * p0 + f[1] * p1, [(g * p0).sum(), (g * p1).sum()]
    for l in range(2, nl):
        t = dtype(l)
        p0, p1 = p1, ((2 * t - 1) * x * p1 - (t - 1) * p0) / t
        corr += f[l] * p1
        cl.append((g * p1).sum())
    return corr, np.array(cl)


def rms(a):
    return float(np.sqrt(np.mean(np.asarray(a, dtype=np.longdouble) ** 2)))


@pytest.mark.parametrize("n", [200, 500, 1000, 3000])
def test_errors_of_the_legendre_sums(n):
    rng = np.random.default_rng(n)
    x = np.cos(np.pi * (np.arange(n) + 0.75) / (n + 0.5))
    cl, corr, w = rng.standard_normal(n), rng.standard_normal(n), rng.uniform(0, 1, n)
    f = (2 * np.arange(n) + 1) / (4 * np.longdouble(np.pi)) * cl
    g = 2 * np.longdouble(np.pi) * w * corr
    exact = sums(n, x, f, g, np.longdouble)
    plain = sums(n, x, f.astype(np.float64), g.astype(np.float64), np.float64)
    dev = [torch.as_tensor(v).cuda() for v in (x, w, cl, corr)]
    out_c, out_l = (torch.empty(n, dtype=torch.float64, device="cuda") for _ in range(2))
    _lib.call("ga_cl2corr", n, _lib.ptr(dev[2]), n, _lib.ptr(dev[0]), _lib.ptr(out_c),
              _lib.stream_ptr())
    nb = ctypes.c_size_t()
    _lib.call("ga_corr2cl_workspace_size", n, n, ctypes.byref(nb))
    ws = _lib.workspace(nb.value)
    _lib.call("ga_corr2cl", n, _lib.ptr(dev[0]), _lib.ptr(dev[1]), _lib.ptr(dev[3]), n,
              _lib.ptr(out_l), _lib.ptr(ws), ws.numel(), _lib.stream_ptr())
    for got, p, e in zip((out_c, out_l), plain, exact):
        err, ref = rms(got.cpu().numpy() - e), rms(p - e)
        print(f"n={n}: {err / rms(e):.2e}, textbook form {ref / rms(e):.2e}")
        assert err <= ref
