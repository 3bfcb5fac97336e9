"""Which form a level of 64 to 127 columns a parent takes. With both axes decimated the one-pass VALU form; with an axis
left alone the two-pass form, unless the level has 1,024 children or more (where the one-pass form is the faster) or a
pulse filter of 80 rows or fewer. Each image against the float64 oracle's of the same plan, whatever the form."""
import numpy as np
import pytest

import oracle
from fastsar_amd import plan as pl, sim
from fastsar_amd.ffbp_hip import make_ffbp_hip

pytestmark = pytest.mark.gpu

E1, E2 = (0.0, 1.0, 0.0), (1.0, 0.0, 0.0)
# nx, ny, P, K, T, levels, aperture, level, (Dk, Dp), form (0 two passes, 1 one pass on VALU)
CASES = [(64, 64, 96, 512, 4, 2, 1.0, 1, (2, 1), 0), (320, 64, 96, 96, 4, 3, 1.0, 2, (2, 1), 1),
         (64, 64, 96, 24, 8, 3, 3.0, 2, (1, 3), 0), (96, 64, 96, 20, 8, 4, 2.0, 3, (1, 2), 1),
         (64, 64, 96, 20, 16, 3, 3.0, 1, (1, 1), 0), (512, 128, 400, 20, 8, 3, 2.0, 2, (1, 1), 1),
         (64, 64, 96, 96, 4, 2, 4.0, 1, (2, 2), 1)]


@pytest.mark.parametrize('nx,ny,P,K,T,nlev,aperture,level,D,form', CASES)
def test_form_of_a_level_of_few_columns(nx, ny, P, K, T, nlev, aperture, level, D, form):
    rng = np.random.default_rng(nx + P)
    col = sim.spotlight(P, K, aperture)
    p = pl.make_plan(col, nx, ny, 0.5, 0.5, T=T, nlev=nlev, e1=E1, e2=E2)
    lv = p['levels'][level]
    assert 64 <= lv['C'] * lv['Ko'] < 128 and (lv['Dk'], lv['Dp']) == D
    coll = pl.collection_arrays(p, col.ant)
    S = (rng.standard_normal((P, K)) + 1j * rng.standard_normal((P, K))).astype(np.complex64)
    f = make_ffbp_hip(p, coll)
    e = oracle.plain_db(f(S), oracle.ffbp_image(p, coll, S, 'oracle'))
    print(f'{nx} x {ny} level {level}: {lv["ref"].shape[0]} parents of {lv["C"]} x {lv["Ko"]}, forms {f.level_forms()}: {e:.1f} dB')
    assert f.level_forms()[level] == form
    assert e < -90, e
