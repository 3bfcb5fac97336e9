"""Where the float32 matrix range filter is taken for filters of more than 128 taps: not for few children at a large
decimation, where it is the slower form, and never in place of the direct form that a window longer than LDS takes, whose
sums are more accurate. The forms differ in the order of their sums, so equal bits show which one ran. FSH_ROT_KERNEL=f32
takes the matrix form wherever it fits: its tile edges against the float64 oracle at the VALU form's bound (-120 dB)."""
import numpy as np
import pytest

import oracle
from fastsar_amd import _hip, plan as pl
from oracle import plain_db as db

pytestmark = pytest.mark.gpu


def _stage(D, pf, Cn, Np, K, P=7):
    rng = np.random.default_rng(3 * D + Cn)
    fr, _ = pl.decimator_fir(K, D, pf)
    x = (rng.standard_normal((Np, P, K)) + 1j * rng.standard_normal((Np, P, K))).astype(np.complex64)
    c0 = rng.uniform(-0.5, 0.5, (Np, Cn, P)).astype(np.float32)
    sl = rng.uniform(-0.8, 0.8, (Np, Cn, P)).astype(np.float32)
    dev = [_hip.DeviceArray.from_host(a) for a in (x, c0, sl, fr['kern'].astype(np.float32))]
    dy = _hip.DeviceArray((Np * Cn, P, fr['n_out']), np.complex64)

    def run(monkeypatch, kernel=None):
        monkeypatch.delenv('FSH_ROT_KERNEL', raising=False)
        if kernel:
            monkeypatch.setenv('FSH_ROT_KERNEL', kernel)
        dx, dc, ds, dt = (_hip.ptr(d) for d in dev)
        _hip.check(_hip.lib().fsh_rot_fir_k(dx, Np, P, K, dc, ds, Cn, dt, fr['L'], fr['pl'], D, fr['n_out'], (K - 1) / 2.0,
                                            _hip.ptr(dy), None))
        return dy.to_host()
    return fr, x, c0, sl, run


# below the line, on it and past it; the last three rows' windows are longer than LDS
@pytest.mark.parametrize('D,pf,Cn,K,matrix', [(40, 0.6, 4, 1500, True), (41, 0.6, 4, 1500, False), (16, 0.5, 3, 900, True),
                                              (25, 0.5, 3, 900, False), (20, 0.5, 2, 900, False), (30, 0.6, 1, 900, False),
                                              (50, 0.7, 25, 2500, False), (64, 0.5, 25, 2000, False),
                                              (120, 0.5, 9, 4000, False)])
def test_where_the_matrix_form_is_taken(D, pf, Cn, K, matrix, monkeypatch):
    fr, _, _, _, run = _stage(D, pf, Cn, 1, K)
    assert fr['L'] > 128
    got, valu, f32 = run(monkeypatch), run(monkeypatch, 'valu'), run(monkeypatch, 'f32')
    assert not np.array_equal(valu, f32)
    assert np.array_equal(got, f32 if matrix else valu)


@pytest.mark.parametrize('D,pf,Cn,Np,K', [(17, 0.6, 1, 2, 401), (40, 0.3, 3, 2, 700), (64, 0.5, 8, 1, 9001),
                                          (120, 0.5, 2, 1, 12000), (31, 0.7, 9, 1, 1501), (9, 0.72, 33, 1, 300)])
def test_matrix_form_edges(D, pf, Cn, Np, K, monkeypatch):
    fr, x, c0, sl, run = _stage(D, pf, Cn, Np, K)
    yre, yim = oracle.rot_fir_k(x.real, x.imag, c0, sl, fr, D, fr['n_out'], (K - 1) / 2.0)
    e = db(run(monkeypatch, 'f32'), yre + 1j * yim)
    print(f'D={D} L={fr["L"]} C={Cn} K={K} -> {fr["n_out"]}: {e:.1f} dB')
    assert e < -120, e
