"""The float32 matrix range filter (filters of more than 128 taps) at the edges of its tiles: outputs below, at and past a
16-wide tile and a four-tile run, children below and past an N-tile of 8 and a block of 32, odd decimations (a padding
plane), runs of 16 taps a phase, a window cut into chunks, the widest decimation of the stage's tests. Against the
float64 oracle at the VALU form's bound (-120 dB: float32 taps within 16 steps of a float64 seed, float32 sums)."""
import numpy as np
import pytest

import oracle
from fastsar_amd import _hip, plan as pl
from oracle import plain_db as db

pytestmark = pytest.mark.gpu

CASES = [(16, 0.5, 25, 1, 4088), (17, 0.6, 1, 2, 401), (31, 0.7, 9, 1, 1501), (9, 0.72, 33, 1, 300), (64, 0.5, 8, 1, 9001),
         (40, 0.3, 3, 2, 700), (23, 0.5, 17, 1, 1111), (120, 0.5, 2, 1, 12000)]


@pytest.mark.parametrize('D,pf,Cn,Np,K', CASES)
def test_long_range_filter(D, pf, Cn, Np, K):
    rng = np.random.default_rng(D + Cn)
    P = 7
    fr, _ = pl.decimator_fir(K, D, pf)
    assert fr['L'] > 128
    x = (rng.standard_normal((Np, P, K)) + 1j * rng.standard_normal((Np, P, K))).astype(np.complex64)
    c0 = rng.uniform(-0.5, 0.5, (Np, Cn, P)).astype(np.float32)
    sl = rng.uniform(-0.8, 0.8, (Np, Cn, P)).astype(np.float32)
    kc, Ko = (K - 1) / 2.0, fr['n_out']
    yre, yim = oracle.rot_fir_k(x.real, x.imag, c0, sl, fr, D, Ko, kc)
    dx, dc, ds, dt = (_hip.DeviceArray.from_host(a) for a in (x, c0, sl, fr['kern'].astype(np.float32)))
    dy = _hip.DeviceArray((Np * Cn, P, Ko), np.complex64)
    print(f'D={D} L={fr["L"]} C={Cn} K={K} -> {Ko}', flush=True)
    _hip.check(_hip.lib().fsh_rot_fir_k(_hip.ptr(dx), Np, P, K, _hip.ptr(dc), _hip.ptr(ds), Cn, _hip.ptr(dt), fr['L'], fr['pl'],
                                        D, Ko, kc, _hip.ptr(dy), None))
    e = db(dy.to_host(), yre + 1j * yim)
    print(f'  {e:.1f} dB')
    assert e < -120, e
