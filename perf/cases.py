"""The work that users of this framework have it do, as cases that can be timed and compared: prompts and decoded tokens of GGUF models through
nt_engine_forward / nt_engine_decode_fused, and of model folders through nt_engine_seq_*.  Weights, tokens and folders are made from a seed.

A case is a dict of plain values.  GGUF cases: `shape` (a preset of ntransformer_amd.engine), `mix` (the tensor format), `layers`, and for op "prompt" the
number of `tokens` of one prompt pass, for op "decode" the `steps` single tokens decoded behind a context of `tokens`.  Folder cases: `family`, `size` (a preset of
ntransformer_amd.synth_folder), `layers`, `dtype`, the mixture's `experts` and `top` (0: the family has none), and for op "prompt" a prompt of `tokens`, for "decode" `steps`
tokens behind a context of `tokens` that is there already, for "turn" a fresh sequence: prompt and `steps` tokens.  Every op returns logits."""
from __future__ import annotations

import json
import math
import os
import shutil
import struct
import tempfile

import numpy as np
import torch

from ntransformer_amd import engine as E
from ntransformer_amd import synth_folder as S

F64 = torch.float64


# ------------------------------------------------------------------------------------------------------------------------------------ the cases
def _gguf(name, op, shape, layers, mix, tokens, steps=0):
    return {"name": name, "kind": "gguf", "op": op, "shape": shape, "layers": layers, "mix": mix, "tokens": tokens, "steps": steps}


def _folder(name, op, family, size, layers, dtype, tokens, steps=0, experts=0, top=0):
    return {"name": name, "kind": "folder", "op": op, "family": family, "size": size, "layers": layers, "dtype": dtype, "experts": experts, "top": top,
            "tokens": tokens, "steps": steps}


def listed():
    return [
        # a small model on a short context: every launch is latency
        _gguf("decode_small_q6_k", "decode", "small", 4, "Q6_K", 100, 4),
        # a chat reply behind a short prompt: the benchmark's model and format
        _gguf("decode_8b_q8_0", "decode", "8b", 32, "Q8_0", 16, 4),
        # a reply behind a long document, four-bit weights
        _gguf("decode_8b_q4_k_m_ctx3900", "decode", "8b", 32, "Q4_K_M", 3900, 4),
        # the wide model's layers (eight of them), six-bit weights, a context of a few hundred
        _gguf("decode_70b_q6_k", "decode", "70b", 8, "Q6_K", 600, 3),
        # a one-line question: the smallest prompt pass
        _gguf("prompt_8b_q4_k_m_16", "prompt", "8b", 32, "Q4_K_M", 16),
        # a page of text, a length that is a multiple of nothing
        _gguf("prompt_8b_q8_0_1003", "prompt", "8b", 32, "Q8_0", 1003),
        # unquantised half-precision weights, a paragraph
        _gguf("prompt_8b_f16_200", "prompt", "8b", 8, "F16", 200),
        # a mixture of experts with latent attention: a page of text
        _folder("prompt_fabolorn_1024", "prompt", "fabolorn", "lite", 2, "bfloat16", 1024, 0, 32, 6),
        # ... and a reply behind it
        _folder("decode_fabolorn_ctx1100", "decode", "fabolorn", "lite", 2, "bfloat16", 1100, 4, 32, 6),
        # attention, recurrence and latent attention one after the other: a document longer than one internal pass
        _folder("prompt_fifotar_1999", "prompt", "fifotar", "lite", 4, "bfloat16", 1999),
        # a short chat turn: a question of forty tokens and the first tokens of the answer
        _folder("turn_fifotar_40", "turn", "fifotar", "lite", 4, "bfloat16", 40, 6),
        # 32-bit weights, as they are used to check other implementations against
        _folder("turn_fifotar_float32_150", "turn", "fifotar", "lite", 3, "float32", 150, 2),
    ]


def _spread(rng, lo, hi):
    """a whole number between lo and hi, spread over its logarithm"""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    if rng.random() < 0.55:
        shape, most = rng.choice([("small", 4), ("8b", 16), ("8b", 16), ("70b", 4)])
        mix = rng.choice(["Q8_0", "Q8_0", "Q4_K_M", "Q4_K_M", "Q4_0", "Q5_K", "Q6_K", "F16"])
        if mix == "F16":
            most = min(most, 4)
        layers = rng.randint(max(1, most // 4), most)
        if rng.random() < 0.5:
            c = _gguf("", "prompt", shape, layers, mix, _spread(rng, 2, 200 if mix == "F16" else 1000))
        else:
            c = _gguf("", "decode", shape, layers, mix, _spread(rng, 1, 200 if mix == "F16" else 1900 if shape == "small" else 3900), rng.randint(1, 4))
    else:
        family = rng.choice(["fabolorn", "fifotar"])
        dtype = rng.choice(["bfloat16", "bfloat16", "bfloat16", "float32"])
        op = rng.choice(["prompt", "turn", "decode"] if family == "fabolorn" else ["prompt", "turn"])
        most = 200 if dtype == "float32" else 1999
        size = rng.choice(["tiny", "lite", "lite"])
        if family == "fabolorn":
            experts = rng.choice([8, 16, 24, 32])
            layers, top = rng.randint(1, 2), rng.choice([2, 4, 6])
        else:
            layers, experts, top = rng.randint(1, 4), 0, 0
        tokens = _spread(rng, 2, most if op != "turn" else 200)
        c = _folder("", op, family, size, layers, dtype, tokens, 0 if op == "prompt" else rng.randint(1, 6), experts, top)
    del c["name"]
    return c


# ------------------------------------------------------------------------------------------------------------------------------------ inputs
def _spec(case, seed):
    return E.synth_spec(case["shape"], case["mix"], seed=1 + seed, layers=case["layers"])


def _tokens(case, seed):
    """prompt or context, then the tokens that the decoding steps are given (a given text: what comes next does not depend on near-ties)"""
    vocab = E.PRESETS[case["shape"]]["vocab"] if case["kind"] == "gguf" else S.PRESETS[case["size"]]["vocab"]
    g = np.random.Generator(np.random.Philox(key=[seed, 4711]))
    t = [int(x) for x in g.integers(0, vocab, case["tokens"] + case["steps"])]
    return t[:case["tokens"]], t[case["tokens"]:]


def _config(case):
    if case["family"] == "fifotar":
        return S.fifotar_config(case["size"], case["layers"])
    cfg = S.fabolorn_config(case["size"], case["layers"])
    for L in cfg["layers"]:
        L["mlp"]["router"] = {"experts": case["experts"], "top": case["top"]}
    return cfg


def _weights(cfg, seed):
    """(name, bfloat16 tensor on the GPU) one after the other: matrices keep a row's size, norm weights lie around one (the parallel family stores most of
    them around zero), rates and biases are small"""
    shapes = S.fabolorn_shapes(cfg) if cfg["architecture"] == "Fabolorn" else S.fifotar_shapes(cfg)
    g = torch.Generator(device="cuda").manual_seed(1000003 * seed + 17)
    for name, shp in shapes.items():
        t = torch.randn(shp, generator=g, device="cuda", dtype=torch.float32)
        last = name.rsplit(".", 1)[-1]
        if name.endswith("vmix"):
            t = torch.sigmoid(t)
        elif len(shp) == 1:
            plain = cfg["architecture"] != "Fabolorn" or (last == "norm" and name != "final.norm")
            t = 0.1 * t + (1.0 if plain and "norm" in last else 0.0)
        elif name != "embed":
            t = t / math.sqrt(shp[-1])
        yield name, t.to(torch.bfloat16)


def _write_folder(folder, cfg, seed):
    shapes = S.fabolorn_shapes(cfg) if cfg["architecture"] == "Fabolorn" else S.fifotar_shapes(cfg)
    header, at = {}, 0
    for name, shp in shapes.items():
        n = 2 * math.prod(shp)
        header[name] = {"dtype": "BF16", "shape": list(shp), "data_offsets": [at, at + n]}
        at += n
    text = json.dumps(header).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(folder, "config.json"), "w") as f:
        json.dump(cfg, f)
    with open(os.path.join(folder, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)))
        f.write(text)
        for _, t in _weights(cfg, seed):
            f.write(t.reshape(-1).view(torch.int16).cpu().numpy().data)


def _place_for(nbytes):
    for d in ("/dev/shm", None):
        if d is None or (os.path.isdir(d) and os.access(d, os.W_OK) and shutil.disk_usage(d).free > 2 * nbytes):
            return d


def prepare(case, seed):
    """a loaded model; for decoding also the context in its cache"""
    eng = E.Engine()
    first, then = _tokens(case, seed)
    state = {"engine": eng, "case": case, "first": first, "then": then}
    room = case["tokens"] + case["steps"]
    if case["kind"] == "gguf":
        eng.load_synthetic(_spec(case, seed), max(room, 64))
        if case["op"] == "decode":
            eng.forward(first, 0)
        return state
    cfg = _config(case)
    folder = tempfile.mkdtemp(prefix="cases_", dir=_place_for(_weight_elements(case) * 2))
    try:
        _write_folder(folder, cfg, seed)
        eng.load_folder(folder, max_context=max(room, 64), dtype=case["dtype"])
    finally:
        shutil.rmtree(folder, ignore_errors=True)
    if case["op"] == "decode":
        state["slot"] = eng.seq_acquire()
        eng.seq_forward(state["slot"], first, want=[])
    return state


def run(state):
    eng, case, first, then = state["engine"], state["case"], state["first"], state["then"]
    if case["kind"] == "gguf":
        if case["op"] == "prompt":
            return [eng.forward(first, 0)]
        return [eng.decode_fused(t, len(first) + i, graph=True) for i, t in enumerate(then)]
    if case["op"] == "decode":
        slot = state["slot"]
        out = [eng.seq_forward(slot, [t], want=[0])[0] for t in then]
        eng.seq_truncate(slot, len(first))
        return out
    slot = eng.seq_acquire()
    out = [eng.seq_forward(slot, first, want=[len(first) - 1])[0]]
    out += [eng.seq_forward(slot, [t], want=[0])[0] for t in then]
    eng.seq_release(slot)
    return out


# ------------------------------------------------------------------------------------------------------------------------------------ bytes and operations
_BLOCK = {"F16": (1, 2), "Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210)}


def _more_bits(i, n):
    return i < n // 8 or i >= 7 * n // 8 or (i - n // 8) % 3 == 2


def _formats(case, i):
    """the formats of layer i's matrices, and of the head (i = None)"""
    mix = case["mix"]
    if mix != "Q4_K_M":
        return mix if i is None else {k: mix for k in ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down")}
    if i is None:
        return "Q6_K"
    more, p = _more_bits(i, case["layers"]), E.PRESETS[case["shape"]]
    v = "Q6_K" if more else "Q5_K" if p["heads"] // p["kv_heads"] >= 4 and p["hidden"] >= 8192 else "Q4_K"
    return {"attn_q": "Q4_K", "attn_k": "Q4_K", "attn_v": v, "attn_output": "Q4_K", "ffn_gate": "Q4_K", "ffn_up": "Q4_K", "ffn_down": "Q6_K" if more else "Q4_K"}


def _sizes(shape):
    p = E.PRESETS[shape]
    W, hd = p["hidden"], p["hidden"] // p["heads"]
    q, kv = p["heads"] * hd, p["kv_heads"] * hd
    return {"attn_q": (q, W), "attn_k": (kv, W), "attn_v": (kv, W), "attn_output": (W, q), "ffn_gate": (p["inter"], W), "ffn_up": (p["inter"], W),
            "ffn_down": (W, p["inter"])}


def _weight_elements(case):
    cfg = _config(case)
    shapes = S.fabolorn_shapes(cfg) if case["family"] == "fabolorn" else S.fifotar_shapes(cfg)
    return sum(math.prod(s) for s in shapes.values())


def _pairs(T, start, window=0, chunks=False):
    """(query, visible key) pairs of T tokens behind `start`"""
    n = 0
    for i in range(start, start + T):
        n += i % window + 1 if window and chunks else min(i + 1, window) if window else i + 1
    return n


def _gguf_work(case):
    p, sizes = E.PRESETS[case["shape"]], _sizes(case["shape"])
    hd = p["hidden"] // p["heads"]
    weights, ops = 0, 0
    for i in range(case["layers"]):
        for k, f in _formats(case, i).items():
            bw, bb = _BLOCK[f]
            weights += sizes[k][0] * sizes[k][1] // bw * bb
            ops += 2 * sizes[k][0] * sizes[k][1]
    bw, bb = _BLOCK[_formats(case, None)]
    head, head_ops = p["vocab"] * p["hidden"] // bw * bb, 2 * p["vocab"] * p["hidden"]
    row = 2 * p["kv_heads"] * hd * 2 * case["layers"]                       # cache bytes of one position
    T, n = case["tokens"], case["steps"]
    att = 4 * p["heads"] * hd * case["layers"]
    if case["op"] == "prompt":
        return {"bytes": weights + head + T * row + 4 * p["vocab"], "flops": ops * T + head_ops + att * _pairs(T, 0)}
    return {"bytes": n * (weights + head + 4 * p["vocab"]) + row * (_pairs(n, T) + n), "flops": n * (ops + head_ops) + att * _pairs(n, T)}


def _folder_pass(case, cfg, T, start):
    """bytes and operations of T tokens behind `start` that end in one row of logits: a matrix counts once however many rows use it, of the experts those that T
    tokens reach at most"""
    W, V, es = cfg["width"], cfg["vocab"], 2 if case["dtype"] == "bfloat16" else 4
    by, fl = V * W * es + T * W * es + 4 * V, 2 * V * W
    for L in cfg["layers"]:
        mx, ml = L["mixer"], L["mlp"]
        H, dn, dv = mx["heads"], mx["dim"], mx["vdim"]
        win = (mx.get("mask") or {}).get("size", 0)
        if L["type"] == "attention":
            G = mx["kv_heads"]
            el = W * (H * dn + G * dn + G * dv + 2 * H * dv)
            fl += 2 * _pairs(T, start, win, True) * H * (dn + dv)
            by += 4 * (start % win + 2 * T) * G * (dn + dv)
        elif L["type"] == "delta":
            G = mx["kv_heads"]
            el = W * (2 * G * dn + 3 * H * dv + 2 * H)
            fl += 7 * T * H * dn * dv
            by += 8 * H * dn * dv
        else:
            dr, R, Q = mx["rot_dim"], mx["kv_rank"], mx.get("q_rank", 0)
            gate = H if cfg["architecture"] == "Fifotar" else H * dv
            el = W * (R + dr + gate + H * dv) + (Q * (W + H * (dn + dr)) if Q else W * H * (dn + dr)) + H * (dn + dv) * R
            fl += 2 * _pairs(T, start, win) * H * (dn + dr + dv)
            by += 4 * (min(start, win) if win else start) * (R + dr) + 8 * T * (R + dr)
        fl += 2 * T * el
        by += es * el
        if ml["kind"] == "dense":
            by, fl = by + es * 3 * W * ml["ff"], fl + 6 * T * W * ml["ff"]
        else:
            e, top, sf = ml["router"]["experts"], ml["router"]["top"], ml["shared"]["ff"]
            by += es * 3 * W * (min(e, T * top) * ml["expert"]["ff"] + sf) + es * (e + 1) * W
            fl += 6 * T * W * (top * ml["expert"]["ff"] + sf) + 2 * T * (e + 1) * W
    return by, fl


def work(case):
    if case["kind"] == "gguf":
        return _gguf_work(case)
    cfg = _config(case)
    passes = [(1, case["tokens"] + i) for i in range(case["steps"])]
    if case["op"] != "decode":
        passes.insert(0, (case["tokens"], 0))
    both = [_folder_pass(case, cfg, T, s) for T, s in passes]
    return {"bytes": sum(b for b, _ in both), "flops": sum(f for _, f in both)}


def tolerance(case):
    """about four times the largest distance from the 64-bit results (`exact`) over the listed and some drawn cases"""
    if case["kind"] == "folder" and case["dtype"] == "bfloat16":
        return {"rel": 1e-2, "max": 5e-2}      # every product's input rounded to eight bits: 2.7e-3 / 9.2e-3 seen
    if case["kind"] == "folder":
        return {"rel": 2e-6, "max": 1e-5}      # 32-bit sums: 2.0e-7 / 1.5e-6 seen on 150 tokens
    return {"rel": 1e-3, "max": 5e-3}          # 32-bit sums, but a cache of halves (a value at a rounding boundary falls to the other side): 2.4e-4 / 1.1e-3 seen


# ------------------------------------------------------------------------------------------------------------------------------------ 64-bit results
def _dequantise(raw, fmt, rows, cols):
    """raw GGUF blocks (uint8 on the GPU) -> [rows, cols] float64"""
    if fmt in ("F16", "F32"):
        return raw.view(torch.float16 if fmt == "F16" else torch.float32).to(F64).view(rows, cols)
    bw, bb = _BLOCK[fmt]
    b = raw.view(-1, bb)

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).to(F64)
    if fmt == "Q8_0":
        out = half(0) * b[:, 2:].contiguous().view(torch.int8).to(F64)
    elif fmt == "Q4_0":
        q = b[:, 2:]
        out = half(0) * (torch.cat([q & 15, q >> 4], 1).to(F64) - 8.0)
    elif fmt in ("Q4_K", "Q5_K"):
        s = b[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).to(F64)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(F64)
        q = b[:, bb - 128:].view(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).view(-1, 8, 32)                  # sub-block 2j: low nibbles, 2j + 1: high ones
        if fmt == "Q5_K":
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
            q = q | (((b[:, 16:48].view(-1, 1, 32) >> bit) & 1) << 4)
        out = (half(0) * sc).view(-1, 8, 1) * q.to(F64) - (half(2) * mn).view(-1, 8, 1)
    else:                                                                  # Q6_K
        ql, qh = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)                              # [blocks, half, quarter, 32]
        sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8).view(1, 1, 4, 1)
        q = (lo | (((qh >> sh) & 3) << 4)).to(F64) - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).to(F64).view(-1, 16, 1)
        out = half(208).view(-1, 1, 1) * sc * q.reshape(-1, 16, 16)
    return out.reshape(rows, cols)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _exact_gguf(case, seed):
    spec, p, sizes = _spec(case, seed), E.PRESETS[case["shape"]], _sizes(case["shape"])
    first, then = _tokens(case, seed)
    toks = torch.tensor(first + then, device="cuda")
    T, H, G, hd = len(first) + len(then), p["heads"], p["kv_heads"], p["hidden"] // p["heads"]

    def tensor(name, fmt, rows, cols):
        raw = torch.from_numpy(E.synth_tensor(spec, name)).cuda()
        if rows is None:                                                   # the embedding: only the rows of the tokens
            return _dequantise(raw.view(p["vocab"], -1)[toks].contiguous().view(-1), fmt, T, cols)
        return _dequantise(raw, fmt, rows, cols)

    def norm(x, name):
        return _rms(x, tensor(name, "F32", 1, p["hidden"])[0], float(np.float32(1e-5)))
    embd = "Q4_K" if case["mix"] in ("Q4_K_M", "Q5_K") else case["mix"]
    x = tensor("token_embd.weight", embd, None, p["hidden"])
    # angles as the format's users form them: frequency and angle in 32 bits, sine and cosine of that
    f = (1.0 / (np.float32(500000.0) ** (2.0 * torch.arange(hd // 2, dtype=torch.float32) / hd))).to(torch.float32).cuda()
    a = (torch.arange(T, device="cuda", dtype=torch.float32)[:, None] * f).to(F64)
    cos, sin = torch.cos(a)[:, None], torch.sin(a)[:, None]

    def turn(z):
        u, v = z[..., :hd // 2], z[..., hd // 2:]
        return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)
    hide = torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1)
    for i in range(case["layers"]):
        fm, at = _formats(case, i), "blk.%d." % i
        h = norm(x, at + "attn_norm.weight")
        q, k, v = (h @ tensor(at + n + ".weight", fm[n], *sizes[n]).T for n in ("attn_q", "attn_k", "attn_v"))
        q, k = turn(q.view(T, H, hd)), turn(k.view(T, G, hd))
        k, v = k.to(torch.float16).to(F64), v.view(T, G, hd).to(torch.float16).to(F64)      # the cache holds halves
        o = torch.empty(T, H, hd, device="cuda", dtype=F64)
        for g in range(G):
            for hh in range(g * (H // G), (g + 1) * (H // G)):
                s = (q[:, hh] @ k[:, g].T) / math.sqrt(hd)
                o[:, hh] = torch.softmax(s.masked_fill_(hide, -math.inf), -1) @ v[:, g]
        x = x + o.view(T, H * hd) @ tensor(at + "attn_output.weight", fm["attn_output"], *sizes["attn_output"]).T
        h = norm(x, at + "ffn_norm.weight")
        gate, up = (h @ tensor(at + n + ".weight", fm[n], *sizes[n]).T for n in ("ffn_gate", "ffn_up"))
        x = x + (torch.nn.functional.silu(gate) * up) @ tensor(at + "ffn_down.weight", fm["ffn_down"], *sizes["ffn_down"]).T
    x = x[-1:] if case["op"] == "prompt" else x[len(first):]
    z = norm(x, "output_norm.weight") @ tensor("output.weight", _formats(case, None), p["vocab"], p["hidden"]).T
    return [r.cpu().numpy() for r in z]


def _rotation(rot, T):
    dims = rot["dims"]
    i = torch.arange(dims // 2, device="cuda", dtype=F64)
    f, mag, sc = rot["base"] ** (-2.0 * i / dims), 1.0, rot.get("scaling")
    if sc:
        def where(turns):
            return dims * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(rot["base"]))
        lo, hi = max(math.floor(where(sc["fast"])), 0), min(math.ceil(where(sc["slow"])), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f, mag = f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
    a = torch.arange(T, device="cuda", dtype=F64)[:, None] * f
    return torch.cos(a) * mag, torch.sin(a) * mag, dims


def _rotate(x, rotation, halves):
    """x [T, heads, d]: its first `dims` entries turned, in halves or in neighbouring pairs"""
    cos, sin, dims = rotation[0][:, None], rotation[1][:, None], rotation[2]
    out = x.clone()
    one, two = (slice(0, dims // 2), slice(dims // 2, dims)) if halves else (slice(0, dims, 2), slice(1, dims, 2))
    u, v = x[..., one], x[..., two]
    out[..., one], out[..., two] = u * cos - v * sin, v * cos + u * sin
    return out


def _attend(q, k, v, hide, scale, cap=0.0, sink=False):
    """q [T, H, d], k [T, G, d], v [T, G, dv]; hide [T, T]; a sink is a further key of score zero without a value"""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[2], device="cuda", dtype=F64)
    for h in range(H):
        g = h // (H // G)
        s = (q[:, h] @ k[:, g].T) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill_(hide, -math.inf)
        if sink:
            s = torch.cat([s, torch.zeros(T, 1, device="cuda", dtype=F64)], 1)
        out[:, h] = torch.softmax(s, -1)[:, :T] @ v[:, g]
    return out


def _latent(h, w, at, mx, eps, fifotar):
    T, H, dn, dr, dv, R = h.shape[0], mx["heads"], mx["dim"], mx["rot_dim"], mx["vdim"], mx["kv_rank"]
    q = _rms(h @ w(at + "dq").T, w(at + "dq.norm"), eps) @ w(at + "uq").T if "q_rank" in mx else h @ w(at + "q").T
    q = q.view(T, H, dn + dr)
    kv = h @ w(at + "dkv").T
    lat, rotation = _rms(kv[:, :R], w(at + "dkv.norm"), eps), _rotation(mx["rot"], T)
    kr = _rotate(kv[:, None, R:], rotation, fifotar)
    q = torch.cat([q[..., :dn], _rotate(q[..., dn:], rotation, fifotar)], -1)
    k = torch.cat([(lat @ w(at + "uk").T).view(T, H, dn), kr.expand(T, H, dr)], -1)
    i = torch.arange(T, device="cuda")
    hide = i[None, :] > i[:, None]
    if mx.get("mask"):
        hide = hide | (i[:, None] - i[None, :] >= mx["mask"]["size"])
    o = _attend(q, k, (lat @ w(at + "uv").T).view(T, H, dv), hide, mx["scale"])
    gate = torch.sigmoid(h @ w(at + "g").T)
    o = o * gate[..., None] if fifotar else o * gate.view(T, H, dv)
    return o.reshape(T, H * dv) @ w(at + "o").T


def _chunked(h, w, at, mx, v_first):
    T, H, G, dn, dv = h.shape[0], mx["heads"], mx["kv_heads"], mx["dim"], mx["vdim"]
    own = v = (h @ w(at + "v").T).view(T, G, dv)
    if v_first is not None:
        b = w(at + "vmix")
        v = (1.0 - b) * v + b * v_first
    i = torch.arange(T, device="cuda")
    size = mx["mask"]["size"]
    hide = (i[None, :] > i[:, None]) | (i[None, :] // size != i[:, None] // size)
    o = _attend((h @ w(at + "q").T).view(T, H, dn), (h @ w(at + "k").T).view(T, G, dn), v, hide, mx["scale"], mx["softcap"], True)
    return (o.reshape(T, H * dv) * torch.sigmoid(h @ w(at + "g").T)) @ w(at + "o").T, own


def _delta(h, w, at, mx, eps):
    T, H, G, dn, dv, taps = h.shape[0], mx["heads"], mx["kv_heads"], mx["dim"], mx["vdim"], mx["conv"]

    def conv(name):
        z, c = h @ w(at + name).T, w(at + name + ".conv")
        z = torch.cat([torch.zeros(taps - 1, z.shape[1], device="cuda", dtype=F64), z])
        return torch.nn.functional.silu(sum(c[:, j] * z[j:j + T] for j in range(taps)))

    def unit(z):
        z = z.view(T, G, dn)
        return (z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
    q, k, v = unit(conv("q")) * dn ** -0.5, unit(conv("k")), conv("v").view(T, H, dv)
    beta = torch.sigmoid(h @ w(at + "b").T)
    decay = torch.exp(-torch.exp(w(at + "A_log")) * torch.nn.functional.softplus(h @ w(at + "a").T + w(at + "dt_bias")))
    state, o = torch.zeros(H, dn, dv, device="cuda", dtype=F64), torch.empty(T, H, dv, device="cuda", dtype=F64)
    for t in range(T):
        state = state * decay[t, :, None, None]
        u = beta[t, :, None] * (v[t] - (state * k[t, :, :, None]).sum(1))
        state = state + k[t, :, :, None] * u[:, None, :]
        o[t] = (state * q[t, :, :, None]).sum(1)
    o = _rms(o, w(at + "norm"), eps).reshape(T, H * dv) * torch.nn.functional.silu(h @ w(at + "g").T)
    return o @ w(at + "o").T


def _clipped(h, w, at, limit):
    g, u = (h @ w(at + "gate").T).clamp(max=limit), (h @ w(at + "up").T).clamp(-limit, limit)
    return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(at + "down").T


def _mixture(h, w, at, ml):
    val, idx = torch.topk(torch.softmax(h @ w(at + "router").T, -1), ml["router"]["top"], -1)
    val = val / (val.sum(-1, keepdim=True) + 1e-20)
    out = torch.sigmoid(h @ w(at + "shared.sg").T) * _clipped(h, w, at + "shared.", ml["shared"]["limit"])
    for e in range(ml["router"]["experts"]):
        t, k = torch.nonzero(idx == e, as_tuple=True)
        if len(t):
            out[t] += val[t, k, None] * _clipped(h[t], w, "%se%d." % (at, e), ml["expert"]["limit"])
    return out


def _exact_folder(case, seed):
    cfg = _config(case)
    kept = dict(_weights(cfg, seed))
    eps, fifotar = cfg["norm"]["eps"], case["family"] == "fifotar"
    first, then = _tokens(case, seed)

    def w(name):
        return kept[name].to(F64)
    x = kept["embed"][torch.tensor(first + then, device="cuda")].to(F64)
    v_first = None
    if fifotar:
        x = x * cfg["embedding"]["scale"]
    for i, L in enumerate(cfg["layers"]):
        at, mx = "l%d." % i, L["mixer"]
        if not fifotar:
            y = _latent(_rms(x, 1.0 + w(at + "norm1"), eps), w, at + "mix.", mx, eps, False)
            x = x + y + _mixture(_rms(x, 1.0 + w(at + "norm2"), eps), w, at + "mlp.", L["mlp"])
            continue
        h = _rms(x, w(at + "norm1"), eps)
        if L["type"] == "attention":
            y, own = _chunked(h, w, at + "mix.", mx, v_first)
            v_first = own if v_first is None else v_first
        elif L["type"] == "delta":
            y = _delta(h, w, at + "mix.", mx, eps)
        else:
            y = _latent(h, w, at + "mix.", mx, eps, True)
        x = x + cfg["residual_mult"] * _rms(y, w(at + "norm1b"), eps)
        y = _clipped(_rms(x, w(at + "norm2"), eps), w, at + "mlp.", L["mlp"]["limit"])
        x = x + cfg["residual_mult"] * _rms(y, w(at + "norm2b"), eps)
    x = x[len(first):] if case["op"] == "decode" else x[len(first) - 1:]
    if fifotar:
        z = _rms(x, w("final.norm"), eps) @ w("embed").T
        z = cfg["logit_softcap"] * torch.tanh(z / cfg["logit_softcap"])
    else:
        z = _rms(x, 1.0 + w("final.norm"), eps) @ w("head").T
    return [r.cpu().numpy() for r in z]


def exact(case, seed):
    return _exact_gguf(case, seed) if case["kind"] == "gguf" else _exact_folder(case, seed)
