"""The final stage of 16 x 16 and 32 x 32 tiles on the matrix instructions at the edges of its split: subapertures below,
at and past a wave's share (16, or 8 in 32 x 32 blocks) and its contraction steps of four, single samples, cropped
tiles, both block sizes (FSH_FINAL_SPLIT 16 and 8), against the register form (FSH_FINAL_SPLIT 1) on the same inputs and
both against float64.

The two forms share their table entries bit for bit and differ in the order of a pixel's 2 Pf Qf fused multiply-adds:
rounding 2^-24 a term, random, so sqrt(2 Pf Qf) 2^-24 of the sum for either, 2.8e-6 (-111 dB) at 17 x 64. Against float64
the matrix form may not be worse than the register form by more than that rounding: 1 dB."""
import numpy as np
import pytest

import oracle
from fastsar_amd import _hip, plan as pl
from oracle import plain_db as db

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('split', [16, 8])
@pytest.mark.parametrize('T,Pf,Qf,weights', [(16, 1, 1, False), (16, 17, 64, True), (16, 67, 9, False), (32, 3, 2, False),
                                             (32, 8, 33, True), (32, 41, 7, False), (32, 130, 5, True)])
def test_final_tiles_matrix_edges(T, Pf, Qf, weights, split, monkeypatch):
    rng = np.random.default_rng(1000 * T + Pf)
    B, spx, spy, crop = 3, 0.5, 0.45, 5
    f0, df = 9.45e9, 3e6
    a0, a1, fc2 = 2 * f0 / pl.C, 2 * df / pl.C, 2 * (f0 + (Qf - 1) / 2 * df) / pl.C
    d = (rng.standard_normal((B, Pf, Qf)) + 1j * rng.standard_normal((B, Pf, Qf))).astype(np.complex64)
    ux, uy = rng.uniform(-0.05, 0.15, (B, Pf)), rng.uniform(0.8, 0.9, (B, Pf))
    geo = np.stack([rng.uniform(0, .1, B), rng.uniform(.8, .9, B), rng.uniform(9e3, 1.1e4, B)], 1)
    dlx, dly = (np.arange(T) - (T - 1) / 2.0) * spx, (np.arange(T) - (T - 1) / 2.0) * spy
    wts = None
    if weights:
        wts = tuple(w.astype(np.float32) for w in (rng.uniform(0.5, 1.5, (B, Pf)), rng.uniform(-0.01, 0.01, (B, Pf)),
                                                   rng.uniform(-0.01, 0.01, (B, Pf))))
    ore, oim = oracle.final_tiles(d.real, d.imag, ux, uy, dlx, dly, a0, a1, geo[:, 0], geo[:, 1], geo[:, 2], fc2, T, wts)
    want = (ore + 1j * oim).reshape(B * T, T)[crop:B * T - crop, crop:T - crop]
    nx, ny = want.shape
    txy = np.stack([np.arange(B) * T, np.zeros(B)], 1).astype(np.int32)
    dd, dux, duy, dgeo, dtxy = (_hip.DeviceArray.from_host(a) for a in (d, ux, uy, geo, txy))
    dw = [None] * 3 if wts is None else [_hip.DeviceArray.from_host(w) for w in wts]
    out = _hip.DeviceArray((nx, ny), np.complex64)

    def form(lanes):
        monkeypatch.setenv('FSH_FINAL_SPLIT', str(lanes))
        _hip.check(_hip.lib().fsh_final_tiles(_hip.ptr(dd), B, Pf, Qf, T, _hip.ptr(dux), _hip.ptr(duy), _hip.ptr(dgeo), spx,
                                              spy, a0, a1, fc2, *[_hip.ptr(w) for w in dw], _hip.ptr(dtxy), crop, crop, nx,
                                              ny, _hip.ptr(out), None))
        return out.to_host()

    reg, mat = form(1), form(split)
    e, er, d = db(mat, want), db(reg, want), db(mat, reg)
    print(f'T={T} Pf={Pf} Qf={Qf} split {split}: {e:.1f} dB, register form {er:.1f} dB, apart {d:.1f} dB')
    assert d < -111 and e < er + 1.0, (d, e, er)
