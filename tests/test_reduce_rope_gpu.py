"""ntk_reduce_rope_kv_store (rotation and cache rows from the partial sums of the projections) against the sums in the same order followed by ntk_rope_kv_store: the same bits of q and of
both caches, with one split and several, a matrix whose sums are there already, both pairings, and positions past the cache's end left out."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import _lib
from ntransformer_amd.ops import DeviceBuffer as DB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,G,hd,splits", [(1, 1, 1, 2, (2, 1, 1)), (4, 8, 2, 128, (3, 3, 3)), (16, 32, 8, 128, (4, 4, 1)), (64, 6, 3, 64, (1, 9, 9)), (65, 5, 5, 256, (2, 2, 2)), (200, 32, 8, 96, (5, 5, 5))])
@pytest.mark.parametrize("interleaved", [0, 1])
def test_rotation_from_partial_sums(T, H, G, hd, splits, interleaved):
    g = np.random.default_rng(T + H)
    rows = (H * hd, G * hd, G * hd)
    parts = [g.standard_normal((n, T, r)).astype(np.float32) for n, r in zip(splits, rows)]
    sums = []
    for p in parts:
        s = p[0].copy()
        for i in range(1, len(p)):
            s = s + p[i]
        sums.append(s)
    start, cap = 7, 7 + T - (2 if T > 4 else 0)
    pos = DB.from_numpy(np.arange(start, start + T, dtype=np.int32))
    L = _lib.lib()
    L.ntk_rope_kv_store.argtypes = [C.c_void_p] * 4 + [C.c_int] * 4 + [C.c_float, C.c_float, C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p]
    L.ntk_reduce_rope_kv_store.argtypes = [C.c_void_p, C.POINTER(C.c_void_p), C.POINTER(C.c_int), C.c_void_p] + [C.c_int] * 4 + [C.c_float, C.c_float, C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int,
                                                                                                                                C.c_void_p]
    out = []
    for fused in (0, 1):
        kc, vc = (DB.from_numpy(np.full((cap, rows[1]), 3.0, np.float16)) for _ in range(2))
        if fused:
            bufs = [DB.from_numpy(p) for p in parts]
            q = bufs[0] if splits[0] == 1 else DB.from_numpy(np.zeros((T, rows[0]), np.float32))
            _lib.check(L.ntk_reduce_rope_kv_store(q.ptr, (C.c_void_p * 3)(*[b.ptr for b in bufs]), (C.c_int * 3)(*splits), pos.ptr, T, H, G, hd, 500000.0, 1.0, interleaved, kc.ptr, vc.ptr,
                                                  start, cap, None), "reduce_rope_kv_store")
        else:
            q, k, v = (DB.from_numpy(s) for s in sums)
            _lib.check(L.ntk_rope_kv_store(q.ptr, k.ptr, v.ptr, pos.ptr, T, H, G, hd, 500000.0, 1.0, interleaved, kc.ptr, vc.ptr, start, cap, None), "rope_kv_store")
        out.append((q.numpy(np.float32)[:T * rows[0]], kc.numpy(np.uint16)[:cap * rows[1]], vc.numpy(np.uint16)[:cap * rows[1]]))
    for a, b in zip(*out):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
