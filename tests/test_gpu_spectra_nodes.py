"""The Legendre sums on nodes of one's own, also outside [-1, 1], where P_l grows
without bound: rows past the last coefficient must not enter, however large
they would be.

Tolerance: nl steps of a few ulp each, 16 nl 2^-52 of the sum of absolute terms."""

import numpy as np
import pytest
import torch
from scipy.special import eval_legendre

pytestmark = pytest.mark.gpu

from glass_amd import _lib  # noqa: E402


# P_l(3/2) overflows at l = 738, inside the last batch of 64 rows of 720
@pytest.mark.parametrize("nl", [1, 2, 63, 65, 500, 720])
def test_nodes_outside_the_interval(nl):
    x = np.array([-1.5, -1.0, -0.3, 0.0, 0.7, 1.0, 1.001, 1.5])
    cl = np.random.default_rng(nl).standard_normal(nl)
    dc, dx = (torch.as_tensor(v).cuda() for v in (cl, x))
    out = torch.empty(len(x), dtype=torch.float64, device="cuda")
    _lib.call("ga_cl2corr", nl, _lib.ptr(dc), len(x), _lib.ptr(dx), _lib.ptr(out),
              _lib.stream_ptr())
    f = (2 * np.arange(nl) + 1) / (4 * np.pi) * cl
    terms = f[:, None] * np.array([eval_legendre(l, x) for l in range(nl)])
    err = np.abs(out.cpu().numpy() - terms.sum(axis=0))
    assert np.all(err <= 16 * nl * 2.0**-52 * np.abs(terms).sum(axis=0))
