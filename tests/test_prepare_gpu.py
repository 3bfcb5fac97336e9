"""The history's first pass at the edges of its runs of 1,024 samples: a non-finite sample is found, and the largest
component (the scale of float16 intermediates) is not missed, in a run's first, last and only sample.

One sample is 10^4 times the rest: a scale that missed it would overflow float16's range of 65,504. With it, each of the
three levels' stored values keep 11 bits, a relative error of at most 2^-11 a component and level: 3 x 2^-11 of the image."""
import numpy as np
import pytest

from fastsar_amd import sim
from fastsar_amd.api import ImageFormer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('P,K', [(130, 500), (130, 1024), (131, 1025), (70, 2050)])
def test_runs_of_the_first_pass(P, K):
    rng = np.random.default_rng(P + K)
    col = sim.spotlight(P, K, 1.0)
    args = (col.ant, col.fmin, col.df, K, 96, 80, 0.5, 0.5, (0.0, 1.0, 0.0), (1.0, 0.0, 0.0))
    full = ImageFormer(*args, window=False)
    half = ImageFormer(*args, window=False, precision='float16')
    S = (rng.standard_normal((P, K)) + 1j * rng.standard_normal((P, K))).astype(np.complex64)
    for p, k in {(0, 0), (P - 1, K - 1), (P // 2, min(1023, K - 1)), (1, K // 1024 * 1024 % K)}:
        print(f'{P} x {K}: sample {p}, {k}', flush=True)
        T = S.copy()
        T[p, k] = 1e4j
        a, b = full(T), half(T)
        assert np.linalg.norm(a - b) <= 3 * 2.0**-11 * np.linalg.norm(a)
        T[p, k] = np.inf
        with pytest.raises(ValueError, match=f'pulse {p}$'):
            full(T)
