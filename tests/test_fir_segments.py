"""The segments of the streaming pulse filter (host code, no GPU). With two columns a thread (from 2^17 columns) the device
holds 1,024 blocks at once: segments that do not fit beside each other take turns, so that as many are cut as do, or none
below the longest segment of 128 outputs. With one column a thread, segments until there are 1,280 blocks."""
import ctypes
import os

import pytest

from fastsar_amd import _hip


def _segments(B, Ko, Po):
    if not os.path.exists(_hip.LIBPATH):
        from fastsar_amd import build
        build.build()
    n = ctypes.c_int()
    _hip.check(_hip.lib().fsh_fir_p_segments(B, Ko, Po, ctypes.byref(n)))
    return n.value


@pytest.mark.parametrize('B,Ko', [(400, 352), (850, 157), (1100, 157), (1681, 157), (800, 330), (1100, 330), (3000, 131)])
@pytest.mark.parametrize('Po', [9, 40, 79, 110, 150, 410, 1510])
def test_two_columns_a_thread(B, Ko, Po, monkeypatch):
    for v in ('FSH_FIRP_IC', 'FSH_FIRP_COLS'):
        monkeypatch.delenv(v, raising=False)
    blocks = -(-B * -(-Ko // 2) // 256)
    n, fewest = _segments(B, Ko, Po), -(-Po // 128)
    assert n == fewest or blocks * n <= 1024, (blocks, n)


@pytest.mark.parametrize('B,Ko,Po', [(64, 157, 260), (1, 300, 60), (64, 352, 2000), (56, 523, 3000)])
def test_one_column_a_thread(B, Ko, Po, monkeypatch):
    for v in ('FSH_FIRP_IC', 'FSH_FIRP_COLS'):
        monkeypatch.delenv(v, raising=False)
    blocks, n = -(-B * Ko // 256), _segments(B, Ko, Po)
    size = -(-Po // n)
    assert size <= 128 and (blocks * n >= 1280 or size <= 8 or blocks * -(-Po // (size - 1)) >= 1280)
