"""Tokens and wanted places of a folder's prompt on their way to the device: more words than a launch's arguments hold go through pinned memory, in two halves in turn."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import fabolorn_oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


def engine(tmp_path, ctx, **kw):
    from ntransformer_amd.engine import Engine
    cfg = O.small_config(layers=("latent_attention", "latent_attention"), **kw)
    w = O.random_weights(cfg, 4)
    O.save_model(str(tmp_path / "m"), cfg, w)
    e = Engine()
    e.load_folder(str(tmp_path / "m"), max_context=ctx, dtype="float32")
    return e, cfg, w


def waits():
    from ntransformer_amd import _lib
    f = _lib.lib().ntk_debug_stream_waits
    f.argtypes, f.restype = [], C.c_longlong
    return f()


def test_prompts_one_after_the_other(tmp_path):
    """around the 32 words of a launch's arguments, each prompt's last row fetched: no wait for the stream beside the fetch; and each prompt's rows are its own, whatever half brought its words"""
    e, cfg, w = engine(tmp_path, 256)
    rng = np.random.default_rng(6)
    prompts = [[int(t) for t in rng.integers(0, cfg["vocab"], n)] for n in (40, 31, 32, 90, 33, 64, 30, 200)]
    ref = [np.asarray(O.forward(cfg, w, p), np.float64) for p in prompts]
    off = lambda got, want: float(np.sqrt(np.mean((got - want) ** 2)) / np.sqrt(np.mean(want ** 2)))

    def one(p, want):
        s = e.seq_acquire()
        got = e.seq_forward(s, p, want=want)
        e.seq_release(s)
        return got
    one(prompts[0], [39])                                  # (the logits' buffer)
    before = waits()
    for p, r in zip(prompts, ref):
        assert off(one(p, [len(p) - 1]), r[-1:]) < 2e-4
    assert waits() == before
    for p, r in zip(prompts, ref):                         # several rows or none: those calls wait themselves
        at = [0, len(p) // 2, len(p) // 2, len(p) - 1]
        assert off(one(p, at), r[at]) < 2e-4
        assert one(p, []).shape[0] == 0
    e.close()


def test_limits(tmp_path):
    """a captured portion beyond 1024 tokens, and more (repeated) wanted places than a pass has room for, are refused; what is at the bound runs"""
    e, cfg, w = engine(tmp_path, 1100)
    toks = [int(t) for t in np.random.default_rng(8).integers(0, cfg["vocab"], 1100)]
    s = e.seq_acquire()
    e.seq_capture(True)
    with pytest.raises(Exception):
        e.seq_forward(s, toks, want=[0])
    e.seq_forward(s, toks[:1024], want=[0])
    assert np.isfinite(e.seq_captured(1024)).all()
    e.seq_capture(False)
    e.seq_truncate(s, 0)
    with pytest.raises(Exception):
        e.seq_forward(s, toks[:40], want=[39] * 1101)
    got = e.seq_forward(s, toks[:40], want=[39] * 1100)
    assert (got == got[0]).all()
    e.close()
