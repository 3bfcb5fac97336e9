"""The one-pass VALU level's registers. A block of four waves gets a quarter of a CU's LDS, so that four blocks share the CU;
that takes four waves a SIMD, 128 registers a thread or fewer, in the form with its decimation factors read at run time
as in those with them fixed."""
import ctypes
import subprocess

import pytest

from fastsar_amd import _hip

pytestmark = pytest.mark.gpu


def test_four_blocks_a_cu():
    lib = _hip.lib()
    names = [l.split()[-1] for l in subprocess.run(['nm', '-D', '--defined-only', _hip.LIBPATH], capture_output=True, text=True,
                                                   check=True).stdout.splitlines()]
    kernels = [n for n in names if n.startswith('_ZN3fsh13k_level_fusedILi')]
    assert len(kernels) >= 100
    hip = ctypes.CDLL('libamdhip64.so')
    worst = {}
    for n in kernels:
        # hipFuncAttributes: int x 2, size_t x 2, int maxDynamicSharedSizeBytes, maxThreadsPerBlock, numRegs, ...
        attr = (ctypes.c_char * 128)()
        fn = ctypes.addressof(ctypes.c_char.in_dll(lib, n))
        assert hip.hipFuncGetAttributes(attr, ctypes.c_void_p(fn)) == 0, n
        block, regs = (ctypes.c_int.from_buffer(attr, off).value for off in (28, 32))
        assert block >= 256 and 0 < regs <= 512, (n, block, regs)
        form = 'run-time' if 'ELi0ELi0E' in n else 'fixed'
        worst[form] = max(worst.get(form, (0, '')), (regs, n))
    print(worst)
    assert worst['run-time'][0] <= 128, worst
