"""ntk_gemm_short_takes answers for the launch: what ntk_gemm_short refuses by its size is not taken, so that the engine looks for another form ahead of the pass (host code only)."""
import ctypes as C

import pytest

from ntransformer_amd import _lib

RAW = {2: 34 / 32, 3: 18 / 32, 4: 144 / 256, 6: 176 / 256, 5: 210 / 256}     # bytes a weight: Q8_0, Q4_0, Q4_K, Q5_K, Q6_K


@pytest.mark.parametrize("dt", sorted(RAW))
def test_matrices_beyond_32_bit_offsets_are_not_taken(dt):
    L = _lib.lib()
    takes = L.ntk_gemm_short_takes
    takes.argtypes = [C.POINTER(C.c_int)] + [C.c_int] * 4
    inf = 8192
    most = int(0xFFFFFF00 / (RAW[dt] * inf)) // 16 * 16
    for T in (2, 16):
        assert takes((C.c_int * 1)(1024), 1, T, inf, dt)
        assert takes((C.c_int * 1)(most * 9 // 10 // 16 * 16), 1, T, inf, dt)
        assert not takes((C.c_int * 1)(most + 16), 1, T, inf, dt)
        assert not takes((C.c_int * 2)(1024, most + 16), 2, T, inf, dt)
