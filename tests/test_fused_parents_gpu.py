"""The one-pass VALU level at many parents of few columns (blocks of two waves, a wave's rows a chunk) against the same
parents a few hundred at a time (blocks of four waves, larger chunks): every output sums the same terms in the same order
whatever the chunk, so the results are the same bits. Rows below, at and past a chunk and a pulse period, the smallest
parent count that takes it and one that the 8 XCDs do not divide."""
import numpy as np
import pytest

from fastsar_amd import _hip, plan as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('Dk,Dp,Cn,Np,P,K', [(2, 2, 4, 4096, 67, 37), (2, 3, 4, 4099, 33, 30), (3, 2, 4, 4097, 21, 60),
                                             (1, 2, 4, 4098, 24, 32), (4, 3, 2, 4096, 50, 120), (2, 2, 4, 4096, 22, 40)])
def test_many_parents(Dk, Dp, Cn, Np, P, K):
    rng = np.random.default_rng(Dk * 100 + Dp * 10 + Cn + P)
    x = (rng.standard_normal((Np, P, K)) + 1j * rng.standard_normal((Np, P, K))).astype(np.complex64)
    c0 = rng.uniform(-0.5, 0.5, (Np, Cn, P)).astype(np.float32)
    sl = rng.uniform(-0.8, 0.8, (Np, Cn, P)).astype(np.float32)
    frk = pl.decimator_fir(K, Dk, 0.5)[0] if Dk > 1 else dict(n_out=K, pl=0, kern=np.ones(1))
    frp = pl.decimator_fir(P, Dp, 0.5)[0]
    Ko, Po = frk['n_out'], frp['n_out']
    dtk, dtp = (_hip.DeviceArray.from_host(f['kern'].astype(np.float32)) for f in (frk, frp))

    def run(a, b):
        dx, dc, ds = (_hip.DeviceArray.from_host(np.ascontiguousarray(v[a:b])) for v in (x, c0, sl))
        dz = _hip.DeviceArray(((b - a) * Cn, Po, Ko), np.complex64)
        _hip.check(_hip.lib().fsh_level_fused(_hip.ptr(dx), b - a, P, K, _hip.ptr(dc), _hip.ptr(ds), Cn, _hip.ptr(dtk),
                                              len(frk['kern']), frk['pl'], Dk, Ko, _hip.ptr(dtp), len(frp['kern']), frp['pl'],
                                              Dp, Po, (K - 1) / 2.0, _hip.ptr(dz), None), 'level_fused')
        return dz.to_host()

    print(f'Dk={Dk} Dp={Dp} C={Cn} Np={Np} P={P} K={K} -> [{Po} x {Ko}]', flush=True)
    whole = run(0, Np)
    parts = np.concatenate([run(a, min(a + 700, Np)) for a in range(0, Np, 700)])
    assert np.isfinite(whole.view(np.float32)).all() and np.array_equal(whole, parts)
