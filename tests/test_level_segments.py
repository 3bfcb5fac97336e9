"""The cut of a one-pass matrix-core level's walk along the pulses (host code, no GPU). A segment re-reads the filter's rows,
as far as they lie on the axis, so a cut that leaves some segment all of them costs blocks and saves nothing; and blocks
that do not fit on a CU beside each other take turns."""
import ctypes
import os

import pytest

from fastsar_amd import _hip, plan as pl


def _segments(Np, P, C, fk, Dk, fp, Dp):
    if not os.path.exists(_hip.LIBPATH):
        from fastsar_amd import build
        build.build()
    n = ctypes.c_int()
    _hip.check(_hip.lib().fsh_level_mfma_segments(Np, P, C, fk['L'], Dk, fk['n_out'], fp['L'], Dp, fp['pl'], fp['n_out'],
                                                  ctypes.byref(n)))
    return n.value


def _longest_walk(P, fp, Dp, segments):
    size = -(-fp['n_out'] // segments)
    starts = range(0, fp['n_out'], size)
    assert len(starts) == segments
    return max(min(P, Dp * (min(i + size, fp['n_out']) - 1) - fp['pl'] + fp['L']) - max(0, Dp * i - fp['pl']) for i in starts)


@pytest.mark.parametrize('D', [2, 3])
@pytest.mark.parametrize('pass_frac', [0.4, 0.6, 0.7])
@pytest.mark.parametrize('K', [100, 160, 300])
def test_cuts_shorten_the_walk(K, pass_frac, D, monkeypatch):
    monkeypatch.delenv('FSH_LMFMA_BLOCKS', raising=False)
    fk = pl.decimator_fir(K, D, pass_frac)[0]
    for P in (70, 100, 150, 400, 1000):
        fp = pl.decimator_fir(P, D, pass_frac)[0]
        for C in (4, 9, 16):
            for Np in (1, 4, 25, 64, 144, 225, 400, 1024):
                n = _segments(Np, P, C, fk, D, fp, D)
                assert n == 1 or _longest_walk(P, fp, D, n) < P, (P, C, Np, n)
                if Np * -(-C // 8) <= 16 and P >= 400:          # few blocks, many rows: cut
                    assert n > 4, (P, C, Np, n)


# rows of 66 and 116 outputs, blocks of five and eight waves; 12 accumulators a filter take 145 registers a thread, so
# that a SIMD holds three waves and a CU one such block: 256 blocks fill the device
@pytest.mark.parametrize('K,Np,C', [(108, 256, 4), (208, 256, 8), (108, 128, 9)])
def test_blocks_that_take_turns(K, Np, C, monkeypatch):
    monkeypatch.delenv('FSH_LMFMA_BLOCKS', raising=False)
    fk, fp = pl.decimator_fir(K, 2, 0.6)[0], pl.decimator_fir(100, 2, 0.6)[0]
    assert -(-fp['L'] // 2) == 12 and fk['n_out'] in (66, 116)
    assert _segments(Np, 100, C, fk, 2, fp, 2) == 1


def test_forced_block_count(monkeypatch):
    fk, fp = pl.decimator_fir(108, 2, 0.6)[0], pl.decimator_fir(400, 2, 0.6)[0]
    for blocks, want in (('1', 1), ('64', 1), ('256', 4), ('1000', 16)):
        monkeypatch.setenv('FSH_LMFMA_BLOCKS', blocks)
        assert _segments(64, 400, 4, fk, 2, fp, 2) == want
