"""The final stage's forms against each other and float64. k_final_tiles_order (32 x 32 tiles on the matrix instructions)
gives k_final_tiles_reg's images bit for bit (FSH_FINAL_KERNEL=reg), with one, two and four waves a tile. k_final_tiles_reg
gives the same bits with one thread a pixel block and with two, which it takes up to 65,536 lanes a launch, so that an image
does not depend on how its tiles are grouped into launches.

Against float64: a table's run of eight entries starts from a first entry and a ratio that are advanced over the samples by
their own float32 ratios, seeded with an error of 2^-25. After q of Qf samples that is q 2^-25 in either, and e times the
ratio's in entry e: rms over e = 0 .. 7 and q, 4.2 x 0.58 Qf 2^-25 = 7.3e-8 Qf, for both tables sqrt(2) of it. Twice that
and the sums' 2^-24 sqrt(2 Pf Qf) are allowed."""
import numpy as np
import pytest

import oracle
from fastsar_amd import _hip, plan as pl
from oracle import plain_db as db

pytestmark = pytest.mark.gpu


def _stage(T, B, Pf, Qf, weights, spx=0.5, spy=0.45):
    rng = np.random.default_rng(T * 1000 + Pf + Qf)
    f0, df = 9.45e9, 3e6
    a0, a1, fc2 = 2 * f0 / pl.C, 2 * df / pl.C, 2 * (f0 + (Qf - 1) / 2 * df) / pl.C
    d = (rng.standard_normal((B, Pf, Qf)) + 1j * rng.standard_normal((B, Pf, Qf))).astype(np.complex64)
    ux, uy = rng.uniform(-0.05, 0.15, (B, Pf)), rng.uniform(0.8, 0.9, (B, Pf))
    geo = np.stack([rng.uniform(0, .1, B), rng.uniform(.8, .9, B), rng.uniform(9e3, 1.1e4, B)], 1)
    w = None
    if weights:
        w = tuple(v.astype(np.float32) for v in (rng.uniform(0.5, 1.5, (B, Pf)), rng.uniform(-0.01, 0.01, (B, Pf)),
                                                 rng.uniform(-0.01, 0.01, (B, Pf))))

    def form(first, count):
        sl = slice(first, first + count)
        txy = np.stack([np.arange(count) * T, np.zeros(count)], 1).astype(np.int32)
        dd, dux, duy, dgeo, dtxy = (_hip.DeviceArray.from_host(np.ascontiguousarray(a)) for a in
                                    (d[sl], ux[sl], uy[sl], geo[sl], txy))
        dw = [None] * 3 if w is None else [_hip.DeviceArray.from_host(np.ascontiguousarray(v[sl])) for v in w]
        out = _hip.DeviceArray((count * T, T), np.complex64)
        _hip.check(_hip.lib().fsh_final_tiles(_hip.ptr(dd), count, Pf, Qf, T, _hip.ptr(dux), _hip.ptr(duy), _hip.ptr(dgeo),
                                              spx, spy, a0, a1, fc2, *[_hip.ptr(v) for v in dw], _hip.ptr(dtxy), 0, 0,
                                              count * T, T, _hip.ptr(out), None))
        return out.to_host()

    def want(sl):
        ww = None if w is None else tuple(v[sl] for v in w)
        dlx, dly = (np.arange(T) - (T - 1) / 2.0) * spx, (np.arange(T) - (T - 1) / 2.0) * spy
        re, im = oracle.final_tiles(d[sl].real, d[sl].imag, ux[sl], uy[sl], dlx, dly, a0, a1, geo[sl, 0], geo[sl, 1], geo[sl, 2],
                                    fc2, T, ww)
        return (re + 1j * im).reshape(-1, T)
    return form, want


def _bound(Pf, Qf):
    return 20 * np.log10(2 * np.sqrt(2) * 7.3e-8 * Qf + 2.0**-24 * np.sqrt(2 * Pf * Qf))


@pytest.mark.parametrize('split', [1, 2, 4])
@pytest.mark.parametrize('Pf,Qf,weights', [(1, 1, False), (9, 8, True), (8, 9, False), (17, 64, True), (40, 7, False),
                                           (3, 33, True), (66, 30, False)])
def test_order_form_is_the_register_form(Pf, Qf, weights, split, monkeypatch):
    form, want = _stage(32, 5, Pf, Qf, weights)
    monkeypatch.setenv('FSH_FINAL_SPLIT', str(split))
    order = form(0, 5)
    monkeypatch.setenv('FSH_FINAL_KERNEL', 'reg')
    assert np.array_equal(order, form(0, 5))
    e = db(order, want(slice(0, 5)))
    print(f'Pf={Pf} Qf={Qf} split {split}: {e:.1f} dB, bound {_bound(Pf, Qf):.1f}')
    assert e < _bound(Pf, Qf)


@pytest.mark.parametrize('weights', [False, True])
@pytest.mark.parametrize('T,B,Pf,Qf', [(8, 65600, 3, 5), (16, 16400, 2, 7)])
def test_one_thread_a_block_and_two(T, B, Pf, Qf, weights, monkeypatch):
    monkeypatch.setenv('FSH_FINAL_SPLIT', '1')
    form, want = _stage(T, B, Pf, Qf, weights)
    whole = form(0, B)                                       # 65,600 lanes: one thread a block
    parts = [(0, 700), (700, 1), (B - 3000, 3000)]           # fewer: two
    for first, count in parts:
        assert np.array_equal(whole[first * T:(first + count) * T], form(first, count))
    for sl in (slice(0, 3), slice(B // 2, B // 2 + 3), slice(B - 3, B)):
        e = db(whole[sl.start * T:sl.stop * T], want(sl))
        assert e < _bound(Pf, Qf), (e, _bound(Pf, Qf))
