"""What a pass takes from the host as arguments of a launch (ntk_store_words) and leaves in pinned memory by a launch's own stores (ntk_copy_out): counts at the ends of their ranges, sizes
that are no multiple of a wide store, addresses that allow none."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import _lib
from ntransformer_amd.ops import DeviceBuffer as DB

pytestmark = pytest.mark.gpu
VP = C.c_void_p


@pytest.mark.parametrize("na,nb", [(1, 0), (0, 1), (1, 1), (16, 16), (31, 1), (32, 0)])
def test_words(na, nb):
    L = _lib.lib()
    L.ntk_store_words.argtypes = [VP, C.c_int, VP, C.c_int, C.POINTER(C.c_int), VP]
    a, b = DB.from_numpy(np.full(na + 1, -7, np.int32)), DB.from_numpy(np.full(nb + 1, -7, np.int32))
    vals = (C.c_int * (na + nb))(*range(100, 100 + na + nb))
    _lib.check(L.ntk_store_words(a.ptr, na, b.ptr if nb else None, nb, vals, None), "store_words")
    assert a.numpy(np.int32).tolist()[:na + 1] == list(range(100, 100 + na)) + [-7]
    assert b.numpy(np.int32).tolist()[:nb + 1] == list(range(100 + na, 100 + na + nb)) + [-7]
    assert L.ntk_store_words(a.ptr, 32, b.ptr, 1, vals, None) != 0 and L.ntk_store_words(None, 1, b.ptr, 0, vals, None) != 0


@pytest.mark.parametrize("n,off", [(1, 0), (3, 0), (4, 0), (1023, 0), (1024, 0), (1025, 0), (32000, 0), (128256, 0), (1025, 1), (7, 3)])
def test_copy_out(n, off):
    L = _lib.lib()
    L.nt_hip_malloc_host.restype = VP
    L.nt_hip_malloc_host.argtypes = [C.c_size_t]
    L.nt_hip_free_host.argtypes = [VP]
    L.ntk_copy_out.argtypes = [VP, VP, C.c_size_t, VP]
    x = np.random.default_rng(n).standard_normal(n + off).astype(np.float32)
    src = DB.from_numpy(x)
    h = L.nt_hip_malloc_host(4 * (n + off + 1))
    view = np.ctypeslib.as_array(C.cast(h, C.POINTER(C.c_float)), (n + off + 1,))
    view[:] = 3.0
    _lib.check(L.ntk_copy_out(h + 4 * off, src.ptr + 4 * off, 4 * n, None), "copy_out")
    _lib.check(L.ntk_stream_synchronize(None), "synchronize")
    assert np.array_equal(view[off:off + n], x[off:]) and (view[:off] == 3.0).all() and view[n + off] == 3.0
    assert L.ntk_copy_out(h, src.ptr, 6, None) != 0
    L.nt_hip_free_host(h)
