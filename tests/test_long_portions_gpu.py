"""Prompts longer than one internal pass of the model folders (4096 tokens), whole and in portions that end elsewhere, against each family's oracle: what a pass leaves for the next -- cache rows,
states, carried convolution inputs, blended values, the pair in front of a pass's first token."""
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
