"""The work users of this framework have it do, as measurable cases.

A case is a dict of plain values.  `kind` says which public entry points one
pass goes through:

  linear     Tensor.linear: one projection of a decoder (q/k/v/o, gate/up/down,
             fc1/fc2, lm_head) on m activation rows, in every weight format.
  attention  KVCache.attention: s query rows (the cache's last s positions)
             over past + s cached keys; s = 1 is a decode step.
  prefill    Model.prefill of a prompt through the decoder runner, then
             Model.logits (what a caller that samples on the host reads).
  generate   Model.generate: prompt pass and greedy decode by graph replay.
  program    ChatDemoKVCache.generate: debug/chat_demo_with_kvcache.tl run op by
             op, one call of the tensor API per TL builtin.

Models are the two architectures the repository is configured for (llama:
hidden 2048, FFN 5632, 32/4 heads, vocab 32000, Q4_0; phi2: hidden 2560, FFN
10240, 32 heads of 80, vocab 51200, Q8_0) with 22 or fewer layers, and small
generic shapes in the drawn cases.  Weights are random: normal matrices of
gain about 1 (residual projections scaled down by the depth, as trained
models are initialised), quantised to the GGUF formats; output.weight row
next(t) is the embedding of t, so each token's successor is predicted as
confidently as a trained model predicts an easy one and the greedy tokens do
not hang on the last bit of a logit.
"""
from __future__ import annotations

import math
import os
import tempfile
import zlib

import numpy as np
import torch

import tensorlogic_amd as tl
from tensorlogic_amd.gguf import (GGML_F16, GGML_Q4_0, GGML_Q6_K, GGML_Q8_0,
                                  GGUFWriter)
from tensorlogic_amd.program import ChatDemoKVCache

DEV = "cuda" if torch.cuda.is_available() else "cpu"   # where inputs are drawn
GGML = {"f16": GGML_F16, "q4_0": GGML_Q4_0, "q8_0": GGML_Q8_0, "q6_k": GGML_Q6_K}
TL_TYPE = {"f16": tl.F16, "q4_0": tl.Q4_0, "q8_0": tl.Q8_0, "q6_k": tl.Q6_K}
BYTES = {"f16": 2.0, "q4_0": 18 / 32, "q8_0": 34 / 32, "q6_k": 210 / 256}   # per weight

LLAMA = dict(arch="llama", hidden=2048, inter=5632, heads=32, kv=4, vocab=32000, wt="q4_0", head="q4_0")
PHI2 = dict(arch="phi2", hidden=2560, inter=10240, heads=32, kv=32, vocab=51200, wt="q8_0", head="q8_0")


def listed():
    return [
        # the lm_head of one decode step, in the type llama.cpp's Q4_0 files keep it in
        dict(name="lm_head_q6k_m1", kind="linear", wt="q6_k", m=1, n=32000, k=2048, bias=False),
        # up projection of a 512-token prompt (the repository's Q8_0 linear benchmark)
        dict(name="up_q8_m512", kind="linear", wt="q8_0", m=512, n=5632, k=2048, bias=False),
        # down projection of a prompt that fills a 2048-token context
        dict(name="down_q4_m2048", kind="linear", wt="q4_0", m=2048, n=2048, k=5632, bias=False),
        # a ragged batch of rows through an unquantised square projection with bias
        dict(name="dense_f16_m333", kind="linear", wt="f16", m=333, n=2560, k=2560, bias=True),
        # attention of a prompt that fills the context; GQA heads of the llama configuration
        dict(name="attn_prefill_2048", kind="attention", s=2048, past=0, heads=32, kv=4, d=64),
        # one decode step late in a long conversation
        dict(name="attn_decode_4000", kind="attention", s=1, past=3999, heads=32, kv=4, d=64),
        # time to first token: the 46-token chat prompt of the decode benchmark, whole model
        dict(name="llama_prefill_46", kind="prefill", **LLAMA, layers=22, tokens=46),
        # a 512-token prompt through Phi-2 blocks (MHA, LayerNorm, GELU, biases)
        dict(name="phi2_prefill_512", kind="prefill", **PHI2, layers=4, tokens=512),
        # chat: prompt and greedy decode at batch 1, whole model (the headline benchmark)
        dict(name="llama_generate", kind="generate", **LLAMA, layers=22, tokens=46, decode=64),
        # Phi-2 blocks decoding after a few hundred tokens
        dict(name="phi2_generate", kind="generate", **PHI2, layers=4, tokens=300, decode=48),
        # the TL program as a script runs it, mostly prompt: a 400-token document
        dict(name="program_prompt_400", kind="program", **LLAMA, layers=2, tokens=400, decode=1),
        # the TL program as a script runs it, mostly decode: a short question
        dict(name="program_chat", kind="program", **LLAMA, layers=2, tokens=24, decode=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear"] * 4 + ["attention"] * 2 + ["prefill"] * 2 + ["generate", "program"])
    if kind == "linear":
        wt = rng.choice(["q4_0", "q4_0", "q8_0", "q8_0", "f16", "q6_k"])
        while True:
            k = 256 * _log_int(rng, 1, 40) if wt == "q6_k" else 32 * _log_int(rng, 8, 320)
            m, n = _log_int(rng, 1, 2048), _log_int(rng, 64, 32000)
            if m * n * k <= 2048 * 2048 * 5632:
                return dict(kind=kind, wt=wt, m=m, n=n, k=k, bias=rng.random() < 0.4)
    if kind == "attention":
        heads, kv, d = rng.choice([(32, 4, 64), (32, 32, 80), (32, 8, 128), (16, 16, 64)])
        s = 1 if rng.random() < 0.4 else _log_int(rng, 2, 2048)
        return dict(kind=kind, s=s, past=rng.choice([0, _log_int(rng, 1, 6000 if s == 1 else 2048)]) if s > 1 else
                    _log_int(rng, 16, 8000), heads=heads, kv=kv, d=d)
    if rng.random() < 0.5 or kind == "program":   # a small generic decoder; the full-width ones otherwise
        heads = rng.choice([4, 8, 16])
        mdl = dict(arch="llama", hidden=64 * heads, inter=32 * rng.randrange(8, 96), heads=heads,
                   kv=rng.choice([heads, heads // 2, heads // 4]), vocab=32 * rng.randrange(16, 500),
                   wt=rng.choice(["q4_0", "q8_0", "f16"]), head="q8_0")
    else:
        mdl = dict(rng.choice([LLAMA, dict(LLAMA, head="q6_k"), PHI2]))
    tokens = _log_int(rng, 2, 512)
    if kind == "prefill":
        return dict(kind=kind, **mdl, layers=rng.randrange(1, 5), tokens=tokens)
    if kind == "generate":
        return dict(kind=kind, **mdl, layers=rng.randrange(1, 5), tokens=tokens, decode=rng.randrange(1, 49))
    return dict(kind=kind, **mdl, layers=rng.randrange(1, 3), tokens=min(tokens, 400), decode=rng.randrange(0, 9))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _normal(seed, name, shape, mean=0.0, std=1.0):
    g = torch.Generator(device=DEV).manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (1 << 62))
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std + mean


def _quantise(w, wt):
    """GGUF bytes (uint8, one row per block) of the f32 matrix w."""
    if wt == "f16":
        return w.half().view(torch.uint8)
    if wt == "q4_0":   # d = the largest magnitude, signed, over -8
        b = w.reshape(-1, 32)
        top = b.gather(1, b.abs().argmax(1, keepdim=True))
        d = (top / -8).half()
        q = torch.clamp(torch.round(b / d.float()) + 8, 0, 15).to(torch.uint8)
        return torch.cat([d.view(torch.uint8), q[:, :16] | (q[:, 16:] << 4)], 1)
    if wt == "q8_0":
        b = w.reshape(-1, 32)
        d = (b.abs().amax(1, keepdim=True) / 127).half()
        q = torch.clamp(torch.round(b / d.float()), -127, 127).to(torch.int8)
        return torch.cat([d.view(torch.uint8), q.view(torch.uint8)], 1)
    b = w.reshape(-1, 16, 16)   # q6_k: 16 scaled groups of 16 per super-block
    s = b.abs().amax(2) / 31
    d = (s.amax(1, keepdim=True) / 127).half()
    sc = torch.clamp(torch.round(s / d.float()), 1, 127)
    q = torch.clamp(torch.round(b / (sc * d.float())[:, :, None]) + 32, 0, 63).to(torch.uint8).reshape(-1, 2, 4, 32)
    lo, hi = q & 15, q >> 4
    ql = torch.cat([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], 2)
    qh = hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)
    return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8), d.view(torch.uint8)], 1)


def _dequantise(blk, wt, n, k):
    """The f16 weights the GGUF bytes stand for, in 64 bits."""
    if wt == "f16":
        return blk.reshape(n, -1).view(torch.float16).double()
    if wt == "q6_k":
        ql, qh = blk[:, :128].reshape(-1, 2, 2, 32), blk[:, 128:192].reshape(-1, 2, 32)
        lo = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
        hi = torch.stack([(qh >> (2 * i)) & 3 for i in range(4)], 2)
        q = (lo | (hi << 4)).double() - 32
        sc = blk[:, 192:208].contiguous().view(torch.int8).double() * blk[:, 208:210].contiguous().view(torch.float16).double()
        w = q.reshape(-1, 16, 16) * sc[:, :, None]
    else:
        d = blk[:, :2].contiguous().view(torch.float16).double()
        if wt == "q4_0":
            q = torch.cat([blk[:, 2:] & 15, blk[:, 2:] >> 4], 1).double() - 8
        else:
            q = blk[:, 2:].contiguous().view(torch.int8).double()
        w = q * d
    return w.half().double().reshape(n, k)


def _host(t):
    return t.cpu().numpy()


def _model_tensors(case, seed):
    """(name, weight type, shape, bytes) of every tensor of the case's model, in GGUF naming."""
    h, f, v, layers, wt = case["hidden"], case["inter"], case["vocab"], case["layers"], case["wt"]
    kvd = case["kv"] * (h // case["heads"])
    llama = case["arch"] == "llama"

    def mat(name, n, k, gain=1.0, t=wt):
        return name, t, (n, k), _quantise(_normal(seed, name, (n, k), 0.0, gain / math.sqrt(k)), t)

    def vec(name, n, mean):
        return name, "f16", (n,), _normal(seed, name, (n,), mean, 0.02).half().view(torch.uint8)

    emb = _normal(seed, "token_embd.weight", (v, h)).half()
    yield "token_embd.weight", "f16", (v, h), emb.view(torch.uint8)
    down = 1.0 / math.sqrt(2 * layers)   # residual branches
    for i in range(layers):
        p = f"blk.{i}."
        yield vec(p + "attn_norm.weight", h, 1.0)
        if llama:
            for nm, n in (("attn_q", h), ("attn_k", kvd), ("attn_v", kvd)):
                yield mat(p + nm + ".weight", n, h)
            yield mat(p + "attn_output.weight", h, h, down)
            yield vec(p + "ffn_norm.weight", h, 1.0)
            yield mat(p + "ffn_gate.weight", f, h)
            yield mat(p + "ffn_up.weight", f, h)
            yield mat(p + "ffn_down.weight", h, f, down)
        else:
            yield vec(p + "attn_norm.bias", h, 0.0)
            for nm, n, k, g in (("attn_qkv", 3 * h, h, 1.0), ("attn_output", h, h, down), ("ffn_up", f, h, 1.0),
                                ("ffn_down", h, f, down)):
                yield mat(p + nm + ".weight", n, k, g)
                yield vec(p + nm + ".bias", n, 0.0)
    yield vec("output_norm.weight", h, 1.0)
    if not llama:
        yield vec("output_norm.bias", h, 0.0)
    succ = _successor(torch.arange(v, device=DEV), v)
    out = torch.empty_like(emb)
    out[succ] = emb
    yield "output.weight", case["head"], (v, h), _quantise(out.float() * (0.5 / math.sqrt(h)), case["head"])
    if not llama:
        yield vec("output.bias", v, 0.0)


def _successor(t, vocab):
    """The token a model of these cases predicts after t (a permutation)."""
    a = 97
    while math.gcd(a, vocab) > 1:
        a += 2
    return (t * a + 11) % vocab


def _write_model(case, seed, path):
    w = GGUFWriter()
    a = case["arch"]
    w.add_str("general.architecture", a)
    for key, v in (("block_count", case["layers"]), ("embedding_length", case["hidden"]),
                   ("feed_forward_length", case["inter"]), ("attention.head_count", case["heads"]),
                   ("attention.head_count_kv", case["kv"]), ("context_length", 2048),
                   ("rope.dimension_count", _rot(case))):
        w.add_u32(f"{a}.{key}", v)
    w.add_f32(f"{a}.attention.layer_norm_{'rms_' if a == 'llama' else ''}epsilon", 1e-5)
    w.add_f32(f"{a}.rope.freq_base", 10000.0)
    for name, t, shape, blk in _model_tensors(case, seed):
        w.add_tensor(name, GGML[t], shape, _host(blk))
    w.write(path)


def _rot(case):
    d = case["hidden"] // case["heads"]
    return d if case["arch"] == "llama" else min(d, 32)


def _prompt(case, seed):
    return np.random.default_rng([seed, 5]).integers(0, case["vocab"], case["tokens"], dtype=np.int32)


_device = None


def _dev():
    """One device context for the process, as a program has."""
    global _device
    if _device is None:
        _device = tl.Device(0)
    return _device


def prepare(case, seed):
    dev = _dev()
    st = {"case": case}
    if case["kind"] == "linear":
        m, n, k, wt = case["m"], case["n"], case["k"], case["wt"]
        x, w, b = _linear_inputs(case, seed)
        st["x"] = dev.tensor(_host(x))
        if wt == "f16":
            st["w"] = dev.tensor(_host(w.reshape(n, -1).view(torch.float16)))
        else:
            st["w"] = dev.quantized(_host(w), (n, k), TL_TYPE[wt])
        st["b"] = dev.tensor(_host(b)) if case["bias"] else None
    elif case["kind"] == "attention":
        q, k, v = _attention_inputs(case, seed)
        st["q"] = dev.tensor(_host(q))
        st["cache"] = tl.KVCache(dev, 1, k.shape[0], case["kv"], case["d"])
        st["cache"].set(0, dev.tensor(_host(k)), dev.tensor(_host(v)))
    else:
        st["prompt"] = _prompt(case, seed)
        fd, path = tempfile.mkstemp(suffix=".gguf")
        os.close(fd)
        try:
            _write_model(case, seed, path)
            ctx = case["tokens"] + case.get("decode", 0) + 1
            if case["kind"] == "program":
                st["prog"] = ChatDemoKVCache(dev, path, max_ctx=ctx)
            else:
                st["model"] = tl.Model(dev, path, arch=0 if case["arch"] == "llama" else 1, max_ctx=max(ctx, 128))
        finally:
            os.remove(path)
    dev.sync()
    return st


def _linear_inputs(case, seed):
    m, n, k = case["m"], case["n"], case["k"]
    return (_normal(seed, "x", (m, k)).half(), _quantise(_normal(seed, "w", (n, k), 0.0, 1 / math.sqrt(k)), case["wt"]),
            _normal(seed, "b", (n,), 0.0, 0.5).half())


def _attention_inputs(case, seed):
    j, d = case["past"] + case["s"], case["d"]
    return (_normal(seed, "q", (case["s"], case["heads"], d)).half(), _normal(seed, "k", (j, case["kv"], d)).half(),
            _normal(seed, "v", (j, case["kv"], d)).half())


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
class OnDevice(dict):
    """Outputs that stay on the device, as a program that goes on computing
    leaves them: a tensor is read back when its entry is looked at."""

    def __getitem__(self, key):
        v = super().__getitem__(key)
        return v.numpy() if isinstance(v, tl.Tensor) else v


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "linear":
        return OnDevice(y=state["x"].linear(state["w"], state["b"]))
    if kind == "attention":
        return OnDevice(out=state["cache"].attention(state["q"], 0, 1.0 / math.sqrt(case["d"])))
    if kind == "prefill":
        m = state["model"]
        m.reset()
        token = m.prefill(state["prompt"])
        return {"token": token, "logits": m.logits()}
    if kind == "generate":
        tokens = state["model"].generate(state["prompt"], case["decode"])
        return {"tokens": tokens, "logits": state["model"].logits()}
    prog = state["prog"]
    tokens = prog.generate(state["prompt"], case["decode"])
    last = prog.n_layers - 1
    return OnDevice(tokens=tokens, logits=prog.last_logits, k=prog.cache.get_k(last), v=prog.cache.get_v(last))


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    if case["kind"] == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * k * BYTES[case["wt"]] + 2 * (m * k + m * n) + (2 * n if case["bias"] else 0),
                "flops": 2.0 * m * n * k}
    if case["kind"] == "attention":
        s, past, h, d = case["s"], case["past"], case["heads"], case["d"]
        keys = s * past + s * (s + 1) / 2   # key visits, causal
        return {"bytes": 4.0 * (past + s) * case["kv"] * d + 4.0 * s * h * d, "flops": 4.0 * h * d * keys}
    h, f, v, layers, d = case["hidden"], case["inter"], case["vocab"], case["layers"], case["hidden"] // case["heads"]
    kvd = case["kv"] * d
    per_layer = (h + 2 * kvd) * h + h * h + (3 if case["arch"] == "llama" else 2) * f * h
    s, n = case["tokens"], case.get("decode", 0)
    w = per_layer * layers * BYTES[case["wt"]]
    head = v * h * BYTES[case["head"]]

    def keys(rows, past):
        return rows * past + rows * (rows + 1) / 2
    # the prompt reads the weights once and writes its K/V rows; each decode
    # step reads the weights and the K/V rows so far
    byts = (w + head) * (1 + n) + 4.0 * kvd * layers * (s + keys(n, s)) + 2.0 * h * (s + n) + 2.0 * v * (1 + n)
    flops = 2.0 * per_layer * layers * (s + n) + 2.0 * v * h * (1 + n) + 4.0 * h * layers * (keys(s, 0) + keys(n, s))
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    if case["kind"] == "linear":       # f16 results of fp32 sums: ties of the last bit
        return {"rel": 1e-3, "max": 0.02}
    if case["kind"] == "attention":    # f16 scores and probabilities
        return {"rel": 2e-3, "max": 0.04}
    # f16 activations through layers; the tokens are predicted with a wide margin
    return {"rel": 8e-3, "max": 0.08, "differ": 0.0}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "linear":
        x, w, b = _linear_inputs(case, seed)
        y = x.double() @ _dequantise(w, case["wt"], case["n"], case["k"]).T
        return {"y": y + b.double() if case["bias"] else y}
    if case["kind"] == "attention":
        q, k, v = (t.double() for t in _attention_inputs(case, seed))
        return {"out": _attend(q, k, v, case["past"], 1.0 / math.sqrt(case["d"]))}
    return _exact_model(case, seed)


def _attend(q, k, v, past, scale, causal=True):
    s, h, d = q.shape
    g = h // k.shape[1]
    k, v = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
    pos, key = torch.arange(s, device=q.device) + past, torch.arange(k.shape[0], device=q.device)
    mask = (key[None, :] > pos[:, None]) if causal else None
    out = torch.empty_like(q)
    for i in range(h):   # one head at a time: plain products
        sc = (q[:, i] @ k[:, i].T) * scale
        if mask is not None:
            sc = sc.masked_fill(mask, -math.inf)
        out[:, i] = torch.softmax(sc, -1) @ v[:, i]
    return out


def _rotate(x, pos, rot, pairs):
    """RoPE of x [s, heads, d] at positions pos, theta 10000; pairs: interleaved, else half-rotation."""
    half = rot // 2
    inv = 10000.0 ** (-torch.arange(half, device=x.device, dtype=torch.float64) * 2 / rot)
    ang = pos[:, None].double() * inv[None, :]
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    y = x.clone()
    if pairs:
        a, b = x[..., 0:rot:2], x[..., 1:rot:2]
        y[..., 0:rot:2], y[..., 1:rot:2] = a * c - b * s, a * s + b * c
    else:
        a, b = x[..., :half], x[..., half:rot]
        y[..., :half], y[..., half:rot] = a * c - b * s, a * s + b * c
    return y


def _exact_model(case, seed):
    """The model on the prompt and, one by one, its own greedy tokens: all rows
    at once, since the successor of every token is known beforehand (and is
    checked to be the largest logit)."""
    h, heads, kv, v = case["hidden"], case["heads"], case["kv"], case["vocab"]
    d, llama, n = h // heads, case["arch"] == "llama", case.get("decode", 0)
    program = case["kind"] == "program"
    prompt = _prompt(case, seed)
    ids = [int(t) for t in prompt]
    for _ in range(n + 1):
        ids.append(int(_successor(ids[-1], v)))
    tokens, ids = ids[len(prompt):], torch.tensor(ids[:-1], device=DEV)
    s = len(prompt)
    # the program as written rotates every decode row as position 0
    pos = torch.arange(len(ids), device=DEV)
    if program:
        pos = torch.where(pos < s, pos, 0)
    eps = 1e-6 if program else 1e-5
    scale = 0.125 if program else 1.0 / math.sqrt(d)
    W = {}

    def lin(x, name):
        t, shape, blk = W.pop(name + ".weight")
        y = x @ _dequantise(blk, t, *shape).T
        if name + ".bias" in W:
            y = y + vec(name + ".bias")
        return y

    def vec(name):
        return W.pop(name)[2].view(torch.float16).double()

    def norm(x, name):
        if llama:
            return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * vec(name + ".weight")
        x = x - x.mean(-1, keepdim=True)
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * vec(name + ".weight") + vec(name + ".bias")

    x, k_last, v_last = None, None, None
    per_layer = 9 if llama else 10
    for name, t, shape, blk in _model_tensors(case, seed):
        W[name] = (t, shape, blk)
        if name == "token_embd.weight":
            x = blk.reshape(v, -1).view(torch.float16)[ids].double()
            W.clear()
        elif len(W) == per_layer and name.startswith("blk."):
            p = name[:name.index(".", 4) + 1]
            a = norm(x, p + "attn_norm")
            if llama:
                q, k, val = (lin(a, p + m) for m in ("attn_q", "attn_k", "attn_v"))
            else:
                q, k, val = lin(a, p + "attn_qkv").split([h, h, h], -1)
            q = _rotate(q.reshape(-1, heads, d), pos, _rot(case), llama)
            k = _rotate(k.reshape(-1, kv, d), pos, _rot(case), llama)
            k_last, v_last = k, val.reshape(-1, kv, d)
            att = _attend(q, k_last, v_last, 0, scale).reshape(-1, h)
            if llama:
                x = x + lin(att, p + "attn_output")
                a = norm(x, p + "ffn_norm")
                x = x + lin(torch.nn.functional.silu(lin(a, p + "ffn_gate")) * lin(a, p + "ffn_up"), p + "ffn_down")
            else:
                m = torch.nn.functional.gelu(lin(a, p + "ffn_up"), approximate="tanh")
                x = x + lin(att, p + "attn_output") + lin(m, p + "ffn_down")
            assert not W
    logits = lin(norm(x[s - 1:], "output_norm"), "output")
    if logits.argmax(-1).tolist() != tokens:
        return None
    if case["kind"] == "prefill":
        return {"token": tokens[0], "logits": logits[-1]}
    if case["kind"] == "generate":
        return {"tokens": torch.tensor(tokens), "logits": logits[-1]}
    return {"tokens": torch.tensor(tokens), "logits": logits[-1:], "k": k_last, "v": v_last}
