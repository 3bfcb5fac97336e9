"""The final stage of 32 x 32 tiles with one, two or four waves a tile (FSH_FINAL_SPLIT) at the edges of its chunks of eight
samples and groups of eight subapertures, with tiles that do not fill a workgroup and cropped ones, against the form of
images with few tiles (FSH_FINAL_SPLIT 8) on the same inputs.

Both take the same table entries and add a pixel's 2 Pf Qf fused multiply-adds in other orders: a rounding of at most
2^-24 a term, random, sqrt(2 Pf Qf) 2^-24 of the sum for either form, sqrt(4 Pf Qf) 2^-24 between them."""
import numpy as np
import pytest

from fastsar_amd import _hip, plan as pl
from oracle import plain_db as db

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('split', [1, 2, 4])
@pytest.mark.parametrize('Pf,Qf,weights', [(1, 1, False), (9, 8, True), (8, 9, False), (17, 64, True), (40, 7, False), (3, 33, True)])
def test_final_tiles_order_edges(Pf, Qf, weights, split, monkeypatch):
    rng = np.random.default_rng(100 * Pf + Qf)
    T, B, spx, spy, crop = 32, 5, 0.5, 0.45, 5
    f0, df = 9.45e9, 3e6
    a0, a1, fc2 = 2 * f0 / pl.C, 2 * df / pl.C, 2 * (f0 + (Qf - 1) / 2 * df) / pl.C
    d = (rng.standard_normal((B, Pf, Qf)) + 1j * rng.standard_normal((B, Pf, Qf))).astype(np.complex64)
    ux, uy = rng.uniform(-0.05, 0.15, (B, Pf)), rng.uniform(0.8, 0.9, (B, Pf))
    geo = np.stack([rng.uniform(0, .1, B), rng.uniform(.8, .9, B), rng.uniform(9e3, 1.1e4, B)], 1)
    nx, ny = B * T - 2 * crop, T - 2 * crop
    txy = np.stack([np.arange(B) * T, np.zeros(B)], 1).astype(np.int32)
    dd, dux, duy, dgeo, dtxy = (_hip.DeviceArray.from_host(a) for a in (d, ux, uy, geo, txy))
    dw = [None] * 3
    if weights:
        dw = [_hip.DeviceArray.from_host(w.astype(np.float32)) for w in
              (rng.uniform(0.5, 1.5, (B, Pf)), rng.uniform(-0.01, 0.01, (B, Pf)), rng.uniform(-0.01, 0.01, (B, Pf)))]
    out = _hip.DeviceArray((nx, ny), np.complex64)

    def form(lanes):
        monkeypatch.setenv('FSH_FINAL_SPLIT', str(lanes))
        _hip.check(_hip.lib().fsh_final_tiles(_hip.ptr(dd), B, Pf, Qf, T, _hip.ptr(dux), _hip.ptr(duy), _hip.ptr(dgeo), spx,
                                              spy, a0, a1, fc2, *[_hip.ptr(w) for w in dw], _hip.ptr(dtxy), crop, crop, nx,
                                              ny, _hip.ptr(out), None))
        return out.to_host()

    e = db(form(split), form(8))
    print(f'Pf={Pf} Qf={Qf} split {split}: {e:.1f} dB apart')
    assert e < 20 * np.log10(np.sqrt(4 * Pf * Qf) * 2.0**-24), e
