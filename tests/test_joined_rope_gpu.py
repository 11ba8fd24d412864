"""ntk_reduce_rope_kv_store_joined: pieces of query, key and value side by side give the bits of the same pieces apart."""
import ctypes as C

import numpy as np
import pytest

from ntransformer_amd import _lib
from ntransformer_amd.ops import DeviceBuffer as DB

pytestmark = pytest.mark.gpu
VP, I, F = C.c_void_p, C.c_int, C.c_float


@pytest.mark.parametrize("T", [1, 64, 65, 256, 257])      # (up to 64 tokens a workgroup per 256 pairs, beyond four a token)
@pytest.mark.parametrize("H,G,hd,splits,interleaved", [(4, 2, 64, 2, 0), (8, 2, 128, 3, 1), (3, 3, 34, 1, 0)])
def test_pieces_side_by_side(T, H, G, hd, splits, interleaved):
    L, g = _lib.lib(), np.random.default_rng(T + H)
    tail = [VP] + [I] * 4 + [F, F, I, VP, VP, I, I, VP]
    L.ntk_reduce_rope_kv_store.argtypes = [VP, C.POINTER(VP), C.POINTER(I)] + tail
    L.ntk_reduce_rope_kv_store_joined.argtypes = [VP, VP, I] + tail
    rows = (H * hd, G * hd, G * hd)
    all_ = g.standard_normal((splits, T, sum(rows))).astype(np.float32)
    at = np.cumsum((0,) + rows)
    pos, out = DB.from_numpy(np.arange(5, 5 + T, dtype=np.int32)), []
    for joined in (0, 1):
        q, kc, vc = DB.zeros(T * rows[0] * 4), DB.zeros((T + 5) * rows[1] * 2), DB.zeros((T + 5) * rows[1] * 2)
        args = (pos.ptr, T, H, G, hd, 500000.0, 1.0, interleaved, kc.ptr, vc.ptr, 5, T + 4, None)
        if joined:
            b = DB.from_numpy(all_)
            _lib.check(L.ntk_reduce_rope_kv_store_joined(q.ptr, b.ptr, splits, *args), "joined")
        else:
            b = [DB.from_numpy(np.ascontiguousarray(all_[:, :, at[i]:at[i + 1]])) for i in range(3)]
            _lib.check(L.ntk_reduce_rope_kv_store(q.ptr, (VP * 3)(*[x.ptr for x in b]), (I * 3)(*[splits] * 3), *args), "apart")
        out.append([x.numpy(np.uint8) for x in (q, kc, vc)])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert L.ntk_reduce_rope_kv_store_joined(q.ptr, pos.ptr, 0, *args) != 0
