"""Prompt passes of GGUF models whose tensors have different formats inside a layer: what a launch leaves for the next one (token maxima, split activations) has to belong to
the activations that the next one reads, whichever formats the layer's other matrices have."""
import numpy as np
import pytest

from ntransformer_amd import engine as E
from ntransformer_amd import gguf as G

pytestmark = pytest.mark.gpu

WIDE = G.LlamaShape("wide", 4096, 4096, 2, 32, 8, 512, ctx=256, bos=256, eos=257)     # (half-precision matrices go out as tiles from 3072 inputs on)
NAMES = ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down")


def make(path, shape, formats, monkeypatch, boost=False):
    """formats: one name per matrix of NAMES.  Tokens 128 .. 255 have one entry that towers over the others; boost: gate and up answer to that entry"""
    types = {"token_embd.weight": G.GGML_F16, "output.weight": G.GGML_Q8_0}
    for i in range(shape.layers):
        types.update({"blk.%d.%s.weight" % (i, n): G.NAME_TO_GGML[f] for n, f in zip(NAMES, formats)})
    monkeypatch.setattr(G, "tensor_types", lambda *_: types)
    G.make_synthetic_llama(path, shape, "mixed")
    f = G.read_gguf(path)

    def rows(name):
        t = f.tensors[name]
        return np.memmap(path, "<f2", "r+", f.data_offset + t.offset, shape=(t.dims[1], t.dims[0]))

    e = rows("token_embd.weight")
    e[:, 7] = 0.0
    e[128:256, 7] = 1000.0
    if boost:
        for i in range(shape.layers):
            rows("blk.%d.ffn_gate.weight" % i)[:, 7] *= 3000.0
            rows("blk.%d.ffn_up.weight" % i)[:, 7] *= 3000.0


def loaded(path, **options):
    eng = E.Engine()
    eng.load(path, 256)
    for k, v in options.items():
        eng.set_option(k, v)
    return eng


def near(a, b, rel=1e-3):       # (a cache of halves: a value at a rounding boundary falls to the other side)
    a, b = a.astype(np.float64), b.astype(np.float64)
    return np.linalg.norm(a - b) <= rel * np.linalg.norm(b)


PLAIN, TOWERING = list(range(1, 101)), list(range(128, 228))


@pytest.mark.parametrize("formats,boost", [
    (("Q8_0", "Q8_0", "F16", "Q8_0", "Q8_0", "Q8_0", "Q8_0"), False),        # half-precision values beside quantised queries and keys
    (("Q4_K", "F16", "Q6_K", "Q4_K", "Q4_K", "Q4_K", "Q4_K"), False),        # a quantised matrix behind a half-precision one
    (("Q8_0", "Q8_0", "Q8_0", "Q8_0", "Q8_0", "F16", "F16"), False),         # half-precision up beside a quantised gate
    (("Q8_0", "Q8_0", "Q8_0", "Q8_0", "F16", "F16", "F16"), True),           # half-precision feed-forward behind quantised attention
])
def test_a_prompt_does_not_depend_on_the_prompts_before_it(formats, boost, tmp_path, monkeypatch):
    """a short prompt behind a longer one of other magnitudes: the same bits as on a fresh engine, and the per-token path's logits"""
    path = str(tmp_path / "m.gguf")
    make(path, WIDE, formats, monkeypatch, boost)
    before, short = (TOWERING, PLAIN[:40]) if boost else (PLAIN, TOWERING[:40])
    eng = loaded(path)
    eng.forward(before, 0)
    behind = eng.forward(short, 0)
    eng.close()
    eng = loaded(path)
    fresh = eng.forward(short, 0)
    eng.close()
    assert np.isfinite(behind).all() and np.array_equal(behind, fresh)
    eng = loaded(path, batched_prefill=0)
    assert near(fresh, eng.forward(short, 0))
    eng.close()


@pytest.mark.parametrize("width,inter", [(4096, 4096), (3072, 4096), (2048, 3072)])       # (the last: one-token products everywhere but in ffn_down)
@pytest.mark.parametrize("T", [2, 3, 9, 70])
def test_half_precision_prompts(T, width, inter, tmp_path, monkeypatch):
    """every matrix in F16: the tiles with the maxima that norms and activations leave, on their own and summed onto the stream, against the one-token products; a short pass
    behind a longer one"""
    path = str(tmp_path / "m.gguf")
    make(path, G.LlamaShape("wide", width, inter, 2, width // 128, 8, 512, ctx=256, bos=256, eos=257), ("F16",) * 7, monkeypatch)
    got = []
    for batched in (1, 0):
        eng = loaded(path, batched_prefill=batched)
        eng.forward(PLAIN, 0)
        got.append(eng.forward(TOWERING[:T], 0))
        eng.close()
    assert near(*got)


@pytest.mark.parametrize("gate,up", [("Q8_0", "Q4_0"), ("Q4_K", "Q6_K"), ("F16", "F16"), ("F32", "Q8_0")])
@pytest.mark.parametrize("T", [2, 40, 64, 65])
def test_gate_and_up_of_two_formats_in_front_of_a_quantised_down(gate, up, T, tmp_path, monkeypatch):
    """the gated activation is formed once, whichever launch forms it"""
    path = str(tmp_path / "m.gguf")
    make(path, G.SMALL, ("Q8_0", "Q8_0", "Q8_0", "Q8_0", gate, up, "Q8_0"), monkeypatch)
    prompt = list(range(1, T + 1))
    got = []
    for batched in (1, 0):
        eng = loaded(path, batched_prefill=batched)
        got.append(eng.forward(prompt, 0))
        eng.close()
    assert near(*got)
