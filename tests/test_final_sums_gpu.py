"""The final stage on the matrix instructions in 16 x 16 blocks may be no further from float64 than the register form with 16
lanes a pixel block, which it replaced: both take the same tables, so only the sums' float32 rounding differs.

0.05 dB is allowed: the tables' error, common to both, is at least three times the sums' (measured: a sum four times as long
adds 0.1 dB), so over n pixels the mean squares of the two forms differ by 2 x 1/3 x sqrt(2 / n) of the tables' by chance,
0.02 dB at 25,600 pixels; 0.05 is two and a half times that."""
import numpy as np
import pytest

import oracle
from fastsar_amd import _hip, plan as pl
from oracle import plain_db as db

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('T,B,Pf,Qf,weights', [(16, 100, 24, 30, False), (16, 100, 24, 30, True), (32, 25, 24, 30, False),
                                               (16, 100, 17, 64, True), (32, 25, 44, 40, True)])
def test_no_further_from_float64_than_the_register_form(T, B, Pf, Qf, weights, monkeypatch):
    rng = np.random.default_rng(T + 10 * Pf + Qf)
    spx = spy = 0.5
    f0, df = 9.45e9, 3e6 * 64 / Qf
    a0, a1, fc2 = 2 * f0 / pl.C, 2 * df / pl.C, 2 * (f0 + (Qf - 1) / 2 * df) / pl.C
    d = (rng.standard_normal((B, Pf, Qf)) + 1j * rng.standard_normal((B, Pf, Qf))).astype(np.complex64)
    ux, uy = rng.uniform(-0.05, 0.05, (B, Pf)), rng.uniform(0.8, 0.9, (B, Pf))
    geo = np.stack([rng.uniform(0, .1, B), rng.uniform(.8, .9, B), rng.uniform(9e3, 1.1e4, B)], 1)
    dl = (np.arange(T) - (T - 1) / 2.0) * spx
    w = None
    if weights:
        w = tuple(v.astype(np.float32) for v in (rng.uniform(0.5, 1.5, (B, Pf)), rng.uniform(-0.01, 0.01, (B, Pf)),
                                                 rng.uniform(-0.01, 0.01, (B, Pf))))
    re, im = oracle.final_tiles(d.real, d.imag, ux, uy, dl, dl, a0, a1, geo[:, 0], geo[:, 1], geo[:, 2], fc2, T, w)
    want = (re + 1j * im).reshape(B * T, T)
    txy = np.stack([np.arange(B) * T, np.zeros(B)], 1).astype(np.int32)
    dd, dux, duy, dgeo, dtxy = (_hip.DeviceArray.from_host(a) for a in (d, ux, uy, geo, txy))
    dw = [None] * 3 if w is None else [_hip.DeviceArray.from_host(v) for v in w]
    out = _hip.DeviceArray((B * T, T), np.complex64)

    def form():
        _hip.check(_hip.lib().fsh_final_tiles(_hip.ptr(dd), B, Pf, Qf, T, _hip.ptr(dux), _hip.ptr(duy), _hip.ptr(dgeo), spx,
                                              spy, a0, a1, fc2, *[_hip.ptr(v) for v in dw], _hip.ptr(dtxy), 0, 0, B * T, T,
                                              _hip.ptr(out), None))
        return db(out.to_host(), want)

    monkeypatch.setenv('FSH_FINAL_SPLIT', '16')
    e = form()
    monkeypatch.setenv('FSH_FINAL_KERNEL', 'reg')
    er = form()
    print(f'T={T} Pf={Pf} Qf={Qf}: {e:.3f} dB, register form {er:.3f} dB')
    assert e < er + 0.05, (e, er)
