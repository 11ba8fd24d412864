"""Prompts longer than one internal pass of the model folders (4096 tokens), whole and in portions that end elsewhere, against each family's oracle: what a pass leaves for the next -- cache rows,
states, carried convolution inputs, blended values, the pair in front of a pass's first token."""
import ctypes as C
import functools
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import fabolorn_oracle  # noqa: E402
import fifotar_oracle  # noqa: E402
import gibevik_oracle  # noqa: E402
import nizorax_oracle  # noqa: E402
import tubazen_oracle  # noqa: E402
import zalazen_oracle  # noqa: E402

pytestmark = pytest.mark.gpu
N, PASS = 4250, 4096
TOL = 2e-4          # (the families' own)

CASES = {
    "fifotar": (fifotar_oracle, lambda O: O.config([O.attention_layer(size=88), O.delta_layer(), O.attention_layer(size=200), O.latent_layer(ff=0)])),
    "zalazen": (zalazen_oracle, lambda O: O.config([O.layer(size=88, kept=4), O.layer(size=200, kept=1), O.layer(size=30, kept=7, kv_from=0)])),
    "gibevik": (gibevik_oracle, lambda O: O.config([O.layer_attention(every=100, mlp=O.dense()), O.layer_latent(heads=2)])),
    "tubazen": (tubazen_oracle, lambda O: O.small_config(positions=4400, bias_max=500, buckets=24, temp=(0.5, 128), layers=("parallel", "gla"), mlps=(True, True))),
    "nizorax": (nizorax_oracle, lambda O: O.small_config(layers=("attention", "lightning"), mlps=("dense", None), window=200, width=32, ff=40, vocab=40)),
    "fabolorn": (fabolorn_oracle, lambda O: O.small_config(window=70, layers=("latent_attention", "latent_attention"))),
}


@pytest.mark.parametrize("family", list(CASES))
def test_a_prompt_beyond_one_internal_pass(tmp_path, monkeypatch, family):
    from ntransformer_amd.engine import Engine
    monkeypatch.setattr(tubazen_oracle, "distance_bucket", functools.lru_cache(None)(tubazen_oracle.distance_bucket))     # (nine million questions about 4250 distances)
    O, config = CASES[family]
    cfg = config(O)
    w = O.random_weights(cfg, 9)
    O.save_model(str(tmp_path / "m"), cfg, w)
    toks = [int(t) for t in np.random.default_rng(10).integers(0, cfg["vocab"], N)]
    ref = O.forward(cfg, w, toks)
    ref = np.asarray(ref[0] if isinstance(ref, tuple) else ref, np.float64)
    want = [0, 1023, 1024, PASS - 1, PASS, N - 1]
    rel = lambda got, at: float(np.sqrt(np.mean((got - ref[at]) ** 2)) / np.sqrt(np.mean(ref[at] ** 2)))
    e = Engine()
    e.load_folder(str(tmp_path / "m"), max_context=4400, dtype="float32")
    s = e.seq_acquire()
    assert rel(e.seq_forward(s, toks, want=want), want) < TOL
    e.seq_release(s)
    s = e.seq_acquire()
    e.seq_forward(s, toks[:130], want=[])
    assert rel(e.seq_forward(s, toks[130:], want=[PASS - 1, PASS, N - 131]), [PASS + 129, PASS + 130, N - 1]) < TOL
    e.close()


# What the first ones leave out: a mixture and a layer over another's latents, a layer without cache rows of its own at the end, a window on latents, a token's choices that halve the pass (9 of 12 experts: 2048
# tokens).  bfloat16: sizes of whole chunks, so that norms and gates leave rounded rows and products read them (ntk_dense_direct_ahead), over a whole pass and across its edge.
MORE = {
    "gibevik": ("float32", gibevik_oracle, lambda O: O.config([O.layer_attention(every=100, mlp=O.dense()), O.layer_latent(mlp=O.moe(4, 2, 12, identity=1, shared=12)), O.layer_latent(kv_from=1, heads=2)])),
    "zalazen": ("float32", zalazen_oracle, lambda O: O.config([O.layer(size=88, kept=4), O.layer(size=200, kept=1), O.layer(size=30, kept=7, kv_from=0), O.layer(size=0, kv_from=1, ff=0)])),
    "fabolorn": ("float32", fabolorn_oracle, lambda O: O.small_config(window=70, layers=("latent_attention", "latent_attention_2"))),
    "fabolorn, nine choices": ("float32", fabolorn_oracle, lambda O: O.small_config(window=70, experts=12, top=9)),
    "fifotar, bfloat16": ("bfloat16", fifotar_oracle, lambda O: O.config([O.attention_layer(size=88, dim=16, vdim=16, ff=64), O.delta_layer(dim=16, vdim=16, ff=64),
                                                                         O.latent_layer(heads=4, dim=16, vdim=16, rot_dim=8, kv_rank=64, q_rank=64, ff=64)], width=64)),
    "fabolorn, bfloat16": ("bfloat16", fabolorn_oracle, lambda O: O.small_config(window=70, heads=4, dim=16, vdim=16, kv_rank=64, q_rank=64, mlp_on=(False, False))),
}


@pytest.mark.parametrize("case", list(MORE))
def test_a_prompt_beyond_one_internal_pass_and_tokens_behind_it(tmp_path, case):
    from ntransformer_amd import _lib
    from ntransformer_amd.engine import Engine
    dtype, O, config = MORE[case]
    cfg = config(O)
    w = O.random_weights(cfg, 9)
    O.save_model(str(tmp_path / "m"), cfg, w)
    toks = [int(t) for t in np.random.default_rng(11).integers(0, cfg["vocab"], N + 4)]
    ref = O.forward(cfg, w, toks)
    ref = np.asarray(ref[0] if isinstance(ref, tuple) else ref, np.float64)
    tol = TOL if dtype == "float32" else 4e-2          # (the families' own)
    if dtype == "bfloat16":
        f = _lib.lib().ntk_dense_direct_ahead
        f.argtypes, f.restype = [C.c_int] * 4 + [C.c_size_t], C.c_int
        assert f(PASS, 64, 64, 0, 1 << 24) == f(PASS, 64, 64, 1, 1 << 24) == 1
    rel = lambda got, at: float(np.sqrt(np.mean((got - ref[at]) ** 2)) / np.sqrt(np.mean(ref[at] ** 2)))
    want = [0, 1023, 1024, 2047, 2048, PASS - 1, PASS, N - 1]
    e = Engine()
    e.load_folder(str(tmp_path / "m"), max_context=4400, dtype=dtype)
    s = e.seq_acquire()
    got = e.seq_forward(s, toks[:N], want=want)
    assert max(rel(got[k:k + 1], at) for k, at in enumerate(want)) < 3 * tol and rel(got, want) < tol
    for k in range(N, N + 4):
        assert rel(e.seq_forward(s, [toks[k]]), [k]) < 3 * tol
    e.close()


def _left_of(L, most):
    """what is left of the malloc budget, to the byte"""
    left, held = 0, []
    for bit in range(most.bit_length(), -1, -1):
        p = L.nt_hip_malloc(1 << bit)
        if p:
            left += 1 << bit
            held.append(p)
    for p in held:
        L.nt_hip_free(p)
    return left


def test_a_pass_yields_to_memory(tmp_path):
    """a long pass is a matter of speed: with a budget that its buffers do not fit the folder loads with passes half as long, down to 1024 tokens, and computes the same; below those it is refused"""
    from ntransformer_amd import _lib
    from ntransformer_amd.engine import Engine
    L, O = _lib.lib(), fabolorn_oracle
    L.ntk_debug_malloc_budget.argtypes, L.ntk_debug_malloc_budget.restype = [C.c_longlong], None
    L.nt_hip_malloc.argtypes, L.nt_hip_malloc.restype, L.nt_hip_free.argtypes = [C.c_size_t], C.c_void_p, [C.c_void_p]
    cfg = O.small_config(layers=("latent_attention", "latent_attention_2"), dim=72, ff=256, shared_ff=192)
    w = O.random_weights(cfg, 3)
    O.save_model(str(tmp_path / "m"), cfg, w)
    toks = [int(t) for t in np.random.default_rng(4).integers(0, cfg["vocab"], 2500)]
    want = [0, 1023, 1024, 2047, 2048, 2499]
    ref = np.asarray(O.forward(cfg, w, toks), np.float64)[want]
    whole, used = 1 << 30, []

    def load(budget):
        L.ntk_debug_malloc_budget(budget)
        try:
            e = Engine()
            e.load_folder(str(tmp_path / "m"), max_context=4400, dtype="float32")
            used.append(budget - _left_of(L, budget))
        finally:
            L.ntk_debug_malloc_budget(-1)
        got = e.seq_forward(e.seq_acquire(), toks, want=want)
        e.close()
        assert np.sqrt(np.mean((got - ref) ** 2)) < TOL * np.sqrt(np.mean(ref ** 2))
    image = L.ntk_prompt_attention_image_bytes
    image.argtypes, image.restype = [C.c_int] * 4, C.c_size_t
    room = image(4400, cfg["layers"][0]["mixer"]["heads"], 72 + 8, 24)
    load(whole)
    load(used[0] - 1)                                  # (the image alone does not fit: the pass yields before it does)
    load(used[0] - room - 1)
    load(used[1] - 1)
    assert used[1] == used[2] < used[0] - room and used[3] < used[1] and used[1] - used[3] < used[0] - used[1]
    load(used[3] - 1)                                  # passes of 1024, no image
    with pytest.raises(Exception):
        load(used[4] - 1)
