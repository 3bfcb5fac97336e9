"""The float32 matrix range filter's complex taps and sums: its error against float64 may not pass that of the VALU form
(FSH_ROT_KERNEL=valu) on the same inputs, which seeds runs of four to eight taps in float64 and, where a row's window leaves
a block few outputs, deals an output's taps to several threads. The phase slopes reach 0.8 cycles a sample; the filters
have 134 to 434 taps, 7 to 16 a phase, 16 being the most the form takes.

0.1 dB is allowed for the two orders of the sums: the mean square of the error over n outputs scatters by sqrt(2 / n),
0.04 dB at 20,000 outputs, so 0.06 dB for the ratio of two."""
import numpy as np
import pytest

import oracle
from fastsar_amd import _hip, plan as pl
from oracle import plain_db as db

pytestmark = pytest.mark.gpu

CASES = [(16, 0.47, 25, 1100), (12, 0.66, 32, 900), (9, 0.72, 25, 1300), (25, 0.58, 16, 2400),
         (25, 0.36, 17, 2400), (30, 0.7, 16, 2700), (40, 0.6, 19, 3200)]


@pytest.mark.parametrize('D,pf,Cn,K', CASES)
def test_taps_as_accurate_as_the_valu_form(D, pf, Cn, K, monkeypatch):
    rng = np.random.default_rng(7 * D + Cn)
    P = 12
    fr, _ = pl.decimator_fir(K, D, pf)
    L, Ko, kc = fr['L'], fr['n_out'], (K - 1) / 2.0
    assert L > 128 and -(-L // D) <= 16 and Cn * P * Ko >= 20000
    x = (rng.standard_normal((1, P, K)) + 1j * rng.standard_normal((1, P, K))).astype(np.complex64)
    c0 = rng.uniform(-0.5, 0.5, (1, Cn, P)).astype(np.float32)
    sl = rng.uniform(-0.8, 0.8, (1, Cn, P)).astype(np.float32)
    taps = fr['kern'].astype(np.float32)
    yre, yim = oracle.rot_fir_k(x.real, x.imag, c0, sl, dict(fr, kern=taps.astype(np.float64)), D, Ko, kc)
    dx, dc, ds, dt = (_hip.DeviceArray.from_host(a) for a in (x, c0, sl, taps))
    dy = _hip.DeviceArray((Cn, P, Ko), np.complex64)

    def run():
        _hip.check(_hip.lib().fsh_rot_fir_k(_hip.ptr(dx), 1, P, K, _hip.ptr(dc), _hip.ptr(ds), Cn, _hip.ptr(dt), L, fr['pl'],
                                            D, Ko, kc, _hip.ptr(dy), None))
        return dy.to_host()

    mat = run()
    monkeypatch.setenv('FSH_ROT_KERNEL', 'valu')
    valu = run()
    assert not np.array_equal(mat, valu)
    e, ev = db(mat, yre + 1j * yim), db(valu, yre + 1j * yim)
    print(f'D={D} L={L} U={-(-L // D)} C={Cn} -> {Ko}: {e:.2f} dB, VALU form {ev:.2f} dB')
    assert e < ev + 0.1, (e, ev)
