"""Exact backprojection of a grid of few regions whose chunk's pulses do not divide among the images planned: a share is a
whole number of window batches, so that fewer images take them all, and no more are allocated. A chunk of 1,000 pulses is
planned for 15 images and 840 for 13; where an allocation of that many fails, nothing changes, and where one of the
images there are fails, one image takes their place (the sums then in another order)."""
import numpy as np
import pytest

import oracle
from fastsar_amd import ExactFormer, sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('P,planned', [(1000, 15), (840, 13)])
def test_no_more_images_than_shares(P, planned, monkeypatch):
    rng = np.random.default_rng(P)
    nx, ny = 64, 65
    col = sim.spotlight(P, 256, 2.0)
    S = (rng.standard_normal((P, 256)) + 1j * rng.standard_normal((P, 256))).astype(np.complex64)

    def form(images=0):
        monkeypatch.setenv('FSH_FAIL_ALLOC_SIZE', str(images * nx * ny * 8))
        return ExactFormer(col.ant, col.fmin, col.df, 256, nx, ny, 0.5, 0.5, (0.0, 1.0, 0.0), (1.0, 0.0, 0.0))(S)

    a = form()
    taken = [n for n in range(2, 17) if not np.array_equal(a, form(n))]
    print(f'{P} pulses: {taken} images')
    assert len(taken) == 1 and taken[0] < planned
    assert oracle.plain_db(a, form(taken[0])) < -120
