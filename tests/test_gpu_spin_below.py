"""A spin-s field has no coefficients with l < s: whatever E and B hold there
(factors such as 1 / sqrt((l - 1)(l + 2)) leave NaN and infinities) the maps
are, byte for byte, those of zeros in their place."""

import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

from glass_amd import healpix as hp  # noqa: E402


# band limits below the spin, shorter than the kernel's chunk of 8 rows (m = 0
# and 1), one row around it, and several chunks
@pytest.mark.parametrize("lmax", [0, 1, 2, 3, 7, 8, 9, 10, 40])
@pytest.mark.parametrize("spin", [1, 2])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_entries_below_the_spin_are_not_read(spin, lmax, bad):
    nside = 12
    rng = np.random.default_rng(100 * lmax + spin)
    n = O.nalm(lmax)
    clean = rng.standard_normal((2, n)) + 1j * rng.standard_normal((2, n))
    ell = np.concatenate([np.arange(m, lmax + 1) for m in range(lmax + 1)])
    clean[:, ell < spin] = 0.0
    dirty = clean.copy()
    dirty[:, ell < spin] = complex(bad, bad)
    ref, got = (hp.alm2map_spin([torch.as_tensor(a).cuda() for a in pair], nside, spin, lmax)
                for pair in (clean, dirty))
    for r, g in zip(ref, got):
        assert torch.isfinite(r).all()
        assert torch.equal(r, g)
