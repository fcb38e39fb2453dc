"""An odd number of 32-column tiles in the split-FP16 synthesis: the last
column group of the two-tile form runs the one-tile body.  Every accumulator
takes the same products in the same order as in the one-tile form, so the maps
are the same bytes, in each accumulation form."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from glass_amd import _lib  # noqa: E402
from glass_amd import healpix as hp  # noqa: E402


@pytest.mark.parametrize("form", [-1, -2, -3])
@pytest.mark.parametrize("nside,lmax,S", [(16, 32, 5), (33, 70, 33), (64, 190, 47), (40, 127, 65)])
def test_odd_tile_counts(nside, lmax, S, form):
    print(f"nside={nside} lmax={lmax} S={S} form={form}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(100 * nside + S)
    alm = torch.randn(((lmax + 1) * (lmax + 2) // 2, S), dtype=torch.complex64, device="cuda",
                      generator=g)
    plan = _lib.get_plan(nside, lmax)
    knobs = (_lib.TUNE_F16_FLUSH, _lib.TUNE_CHUNK_MIN, _lib.TUNE_MFMA_TILES)
    old = [plan.get_tuning(k) for k in knobs]
    maps = {}
    try:
        plan.set_tuning(_lib.TUNE_F16_FLUSH, form)
        plan.set_tuning(_lib.TUNE_CHUNK_MIN, 2)  # short ranges are cut in two as well
        for tiles in (1, 2):
            plan.set_tuning(_lib.TUNE_MFMA_TILES, tiles)
            maps[tiles] = hp.synth_batch_f32(alm, nside, lmax)
    finally:
        for k, v in zip(knobs, old):
            plan.set_tuning(k, v)
    assert torch.equal(maps[1], maps[2])
