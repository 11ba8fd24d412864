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


@pytest.mark.parametrize("n,off", [(1, 0), (4095, 0), (4096, 0), (4097, 0), (32000, 0), (128256, 0), (8193, 1), (5, 3)])
def test_copy_out_in_pieces(n, off):
    """every piece is whole once its word holds the launch's turn: read as the words come, without a wait for the stream, several turns one after the other"""
    L = _lib.lib()
    L.nt_hip_malloc_host.restype = VP
    L.nt_hip_malloc_host.argtypes = [C.c_size_t]
    L.nt_hip_free_host.argtypes = [VP]
    L.ntk_copy_out_words.restype = C.c_size_t
    L.ntk_copy_out_words.argtypes = [C.c_size_t]
    L.ntk_copy_out_pieces.argtypes = [VP, VP, C.c_size_t, VP, C.c_uint, VP, VP]
    pieces = L.ntk_copy_out_words(n)
    assert pieces == (n + 4095) // 4096
    h, w = L.nt_hip_malloc_host(4 * (n + off + 1)), L.nt_hip_malloc_host(4 * (pieces + 1))
    view = np.ctypeslib.as_array(C.cast(h, C.POINTER(C.c_float)), (n + off + 1,))
    words = np.ctypeslib.as_array(C.cast(w, C.POINTER(C.c_uint)), (pieces + 1,))
    view[:], words[:] = 3.0, 0
    bump = DB.from_numpy(np.array([41, -1], np.int32))
    for turn in range(1, 30):
        x = np.random.default_rng(n + turn).standard_normal(n + off).astype(np.float32)
        src = DB.from_numpy(x)
        _lib.check(L.ntk_copy_out_pieces(h + 4 * off, src.ptr + 4 * off, n, w, turn, bump.ptr, None), "copy_out_pieces")
        for i in range(pieces):
            for _ in range(1000000):
                if words[i] == turn:
                    break
            assert words[i] == turn
            at, end = off + 4096 * i, min(off + 4096 * (i + 1), off + n)
            assert np.array_equal(view[at:end], x[at:end])
        assert (view[:off] == 3.0).all() and view[n + off] == 3.0 and words[pieces] == 0
    assert bump.numpy(np.int32).tolist() == [41 + 29, -1]
    assert L.ntk_copy_out_pieces(h, src.ptr, 0, w, 1, None, None) != 0 and L.ntk_copy_out_pieces(h, src.ptr, n, None, 1, None, None) != 0
    L.nt_hip_free_host(h)
    L.nt_hip_free_host(w)


@pytest.mark.parametrize("graph", [False, True])
def test_given_tokens_beside_generated_ones(graph):
    """decode_fused (its words with the embedding's launch, the position advanced by the launch that takes the logits out) between generated tokens, whose launches do both themselves"""
    from ntransformer_amd import engine as E
    eng = E.Engine()
    eng.load_synthetic(E.synth_spec("small", "Q4_K_M", seed=5, layers=2), 128)
    prompt = [int(t) for t in np.random.default_rng(7).integers(0, E.PRESETS["small"]["vocab"], 9)]
    def given():
        eng.forward(prompt, 0)
        rows, tok = [], 5
        for k in range(6):
            rows.append(eng.decode_fused(tok, len(prompt) + k, graph=graph))
            tok = int(np.argmax(rows[-1]))
        return np.stack(rows)
    one, text = given(), eng.generate_tokens(prompt, 8, temperature=0.0, stop_at_eos=False)
    two = given()
    assert np.array_equal(one, two) and eng.generate_tokens(prompt, 8, temperature=0.0, stop_at_eos=False) == text
    eng.forward(prompt, 0)
    tok = 5
    for k in range(6):                              # the launches of a prompt's token, position by position
        row = eng.forward([tok], len(prompt) + k)
        assert np.abs(row - one[k]).max() <= 1e-3
        tok = int(np.argmax(one[k]))
    eng.close()
