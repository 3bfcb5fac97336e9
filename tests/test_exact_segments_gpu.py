"""Exact backprojection of grids of few regions, whose chunks' pulses are dealt to several images added at the end, against
the same former with chunks too short to be dealt (fewer than 128 pulses): the smallest count that is dealt, a last share
that is partial or empty, grids smaller than and just past a region, both reads. The bound is that of images of different
chunks (float32 sums in another order)."""
import numpy as np
import pytest

import oracle
from fastsar_amd import ExactFormer, sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('interp', ['cubic', 'linear'])
@pytest.mark.parametrize('nx,ny,P', [(33, 31, 128), (7, 90, 129), (64, 65, 1024), (40, 100, 1100), (500, 200, 300)])
def test_pulses_dealt_to_images(nx, ny, P, interp):
    rng = np.random.default_rng(P + nx)
    col = sim.spotlight(P, 256, 2.0)
    S = (rng.standard_normal((P, 256)) + 1j * rng.standard_normal((P, 256))).astype(np.complex64)
    args = (col.ant, col.fmin, col.df, 256, nx, ny, 0.5, 0.5, (0.0, 1.0, 0.0), (1.0, 0.0, 0.0))
    a = ExactFormer(*args, interp=interp)(S)
    b = ExactFormer(*args, interp=interp, chunk=127)(S)
    e = oracle.plain_db(a, b)
    print(f'{nx} x {ny} from {P} {interp}: {e:.1f} dB')
    assert e < -120, e


def test_one_image_where_several_do_not_fit(monkeypatch):
    rng = np.random.default_rng(3)
    col = sim.spotlight(1024, 256, 2.0)
    S = (rng.standard_normal((1024, 256)) + 1j * rng.standard_normal((1024, 256))).astype(np.complex64)
    args = (col.ant, col.fmin, col.df, 256, 64, 65, 0.5, 0.5, (0.0, 1.0, 0.0), (1.0, 0.0, 0.0))
    a = ExactFormer(*args)(S)
    monkeypatch.setenv('FSH_FAIL_ALLOC_SIZE', str(16 * 64 * 65 * 8))
    b = ExactFormer(*args)(S)
    monkeypatch.delenv('FSH_FAIL_ALLOC_SIZE')
    assert oracle.plain_db(a, b) < -120 and not np.array_equal(a, b)
