"""Timed cases of the quantized decoder stack: single linears, SwiGLU and
attention launches through the C ABI of libbrolm_hip.so, and whole calls of
Qwen3Model (a decode step, a batched step, a prompt).

Every kind declares a range: listed() names points of it, draw() gives others.

  linear     bx_linear_f16 over `layers` matrices of one shape, as a layer
             stack runs them: one row (decode), 2..16 (batched decode), 17..127
             (chat turns, short prompts), 128..2048 (prompts; F16 from 512 rows
             on is what long passes multiply)
  swiglu     bx_linear_swiglu_f16: gate / up projections and the activation
  attention  bx_attention_decode_f16 (causal rows after `past` cached keys) or
             bx_attention_gqa_f16 (encode: every row sees every key)
  batch_attention  bx_batch_attention_f16: head norms, RoPE, cache write and
             attention of a batched step over ragged contexts
  decode     Qwen3Model.forward_last of one token after `ctx` tokens
  batch      Qwen3Model.forward_batch of `rows` sequences
  prompt     Qwen3Model.forward_last of a prompt into an empty cache

Weights and activations are random with the spread of a trained layer's (N(0,
0.02) weights as the block formats hold them, unit-variance activations); the
whole models are seeded synthetic checkpoints of the 0.6B and 1.7B shapes.
"""
import ctypes as C
import math
import os
import struct
import tempfile

import numpy as np
import torch

import brolm_amd as ba
from brolm_amd import _native

TYPES = {"F16": 1, "Q8_0": 8, "Q4_K": 12, "Q6_K": 14}
BLOCK = {"F16": (1, 2), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q6_K": (256, 210)}
MODELS = {
    "1.7b": dict(hidden=2048, intermediate=6144, tied=False, embed="Q4_K", q="Q4_K", k="Q4_K", v="Q6_K", o="Q4_K",
                 gate="Q4_K", up="Q4_K", down="Q6_K", output="Q6_K"),
    "0.6b": dict(hidden=1024, intermediate=3072, tied=True),
}
LAYERS, VOCAB, HEADS, KV_HEADS, HEAD_DIM, EPS, THETA = 28, 151936, 16, 8, 128, 1e-6, 1e6


# ------------------------------------------------------------------- cases

def listed():
    return [
        # the smallest call: one token's o projection (latency, the launch itself)
        dict(name="o-proj-1row", kind="linear", type="Q4_K", rows=1, n=2048, k=2048, layers=1),
        # the largest matrix of a decode step: the output head for one token
        dict(name="lm-head-1row", kind="linear", type="Q6_K", rows=1, n=VOCAB, k=2048, layers=1),
        # a batched step's MLP in the 0.6B's format, a few sequences in flight
        dict(name="mlp-batch6-q8", kind="swiglu", type="Q8_0", rows=6, n=3072, k=1024, layers=28),
        # a chat turn appended to a conversation: an odd count between decode batch and prompt
        dict(name="gate-turn75", kind="linear", type="Q4_K", rows=75, n=6144, k=2048, layers=14),
        # a paragraph-sized prompt, multiplied straight from the quantized blocks
        dict(name="down-prompt300", kind="linear", type="Q6_K", rows=300, n=2048, k=6144, layers=14),
        # a long prompt's MLP at the 8B widths: the matrix cores' largest call
        dict(name="mlp-prompt2048", kind="swiglu", type="F16", rows=2048, n=12288, k=4096, layers=1),
        # a long prompt's attention at the 8B head counts
        dict(name="attn-prompt2048", kind="attention", rows=2048, past=0, n_q=32, n_kv=8, causal=True),
        # an embedding model's attention over a passage (every key visible)
        dict(name="attn-encode500", kind="attention", rows=500, past=0, n_q=16, n_kv=8, causal=False),
        # serving: sixteen conversations of different lengths, one step's attention
        dict(name="attn-batch16", kind="batch_attention", rows=16, ctx=1500, n_q=16, n_kv=8),
        # single-user decode with the caller's own sampler: one token and its logits
        dict(name="decode-1.7b", kind="decode", model="1.7b", ctx=1024),
        # serving: one step of sixteen conversations and their logits
        dict(name="batch16-1.7b", kind="batch", model="1.7b", rows=16, ctx=1100),
        # time to first token of a long prompt
        dict(name="prompt-1.7b", kind="prompt", model="1.7b", rows=2000),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["swiglu"] * 3 + ["attention"] * 3 + ["batch_attention"] * 2 +
                      ["decode", "batch", "prompt", "prompt"])
    if kind in ("linear", "swiglu"):
        while True:
            t = rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q6_K", "Q8_0", "F16"])
            k = rng.choice([1024, 2048, 3072, 4096, 5120, 6144, 12288, 14336])
            n = _log_int(rng, 500, 16000)
            if kind == "linear":
                rows = _log_int(rng, 512 if t == "F16" else 1, 2048)
                if rows <= 16 and k <= 5120 and rng.random() < 0.2:
                    n = VOCAB
            else:   # the fused form's rows: decode batches and prompts
                k = min(k, 5120)
                rows = rng.randint(3, 16) if t != "F16" and rng.random() < 0.5 else _log_int(
                    rng, 512 if t == "F16" else 128, 2048)
            layers = max(1, min(28, int(1.5e8 / (n * k * BLOCK[t][1] / BLOCK[t][0]))))
            while layers > 1 and layers * rows * n * k > 2.5e11 / 4:
                layers -= 1
            if layers * rows * n * k <= 1e11:
                return dict(kind=kind, type=t, rows=rows, n=n, k=k, layers=layers)
    if kind == "attention":
        rows = _log_int(rng, 2, 2048)
        causal = rng.random() < 0.7
        past = _log_int(rng, 1, 2048) if causal and rng.random() < 0.5 else 0
        return dict(kind=kind, rows=rows, past=past, n_q=rng.choice([16, 32]), n_kv=8, causal=causal)
    if kind == "batch_attention":
        return dict(kind=kind, rows=rng.randint(1, 16), ctx=_log_int(rng, 8, 4000), n_q=rng.choice([16, 32]), n_kv=8)
    model = rng.choice(["1.7b", "0.6b"])
    if kind == "decode":
        return dict(kind=kind, model=model, ctx=_log_int(rng, 16, 3000))
    if kind == "batch":
        return dict(kind=kind, model=model, rows=rng.randint(1, 16), ctx=_log_int(rng, 16, 1500))
    return dict(kind=kind, model=model, rows=_log_int(rng, 8, 2000))


def work(case):
    kind = case["kind"]
    if kind in ("linear", "swiglu"):
        mats = 2 if kind == "swiglu" else 1
        be, bb = BLOCK[case["type"]]
        m, n, k, layers = case["rows"], case["n"], case["k"], case["layers"]
        return {"bytes": layers * (mats * n * k * bb / be + m * n * 2) + m * k * 2,
                "flops": 2.0 * layers * mats * m * n * k}
    if kind == "attention":
        m, past, nq, nkv = case["rows"], case["past"], case["n_q"], case["n_kv"]
        pairs = m * past + (m * (m + 1) / 2 if case["causal"] else m * m)
        return {"bytes": 2 * HEAD_DIM * (2 * m * nq + 2 * (m + past) * nkv), "flops": 4.0 * pairs * nq * HEAD_DIM}
    if kind == "batch_attention":
        keys = sum(_lens(case))
        return {"bytes": 2 * HEAD_DIM * (2 * keys * case["n_kv"] + case["rows"] * (2 * case["n_q"] + 2 * case["n_kv"])),
                "flops": 4.0 * keys * case["n_q"] * HEAD_DIM}
    spec = MODELS[case["model"]]
    h, f, w = spec["hidden"], spec["intermediate"], KV_HEADS * HEAD_DIM
    sizes = [("q", 2 * w * h), ("k", w * h), ("v", w * h), ("o", 2 * w * h), ("gate", f * h), ("up", f * h),
             ("down", f * h)]
    per = sum(s for _, s in sizes)
    wbytes = LAYERS * sum(s * BLOCK[spec.get(r, "Q8_0")][1] / BLOCK[spec.get(r, "Q8_0")][0] for r, s in sizes)
    wbytes += h * VOCAB * (2 if spec["tied"] else BLOCK["Q6_K"][1] / 256)
    rows = 1 if kind == "decode" else case["rows"]
    if kind == "prompt":
        pairs, kv, out = rows * (rows + 1) / 2, rows, 1
    else:
        lens = [case["ctx"]] if kind == "decode" else _lens(case)
        pairs = kv = sum(lens) + rows
        out = rows
    return {"bytes": wbytes + LAYERS * kv * 2 * w * 2 + out * VOCAB * 4,
            "flops": 2.0 * rows * LAYERS * per + 2.0 * out * h * VOCAB + 4.0 * LAYERS * pairs * HEADS * HEAD_DIM}


def tolerance(case):
    """About four times the error measured against exact(): FP16 rounding of
    the outputs (2e-4 to 3e-4) and of dequantized weights or probabilities
    where a path forms them (to 5e-4 with the activation's product), and in a
    whole model the FP16 values between its 28 layers (5e-3)."""
    return {"rel": {"linear": 1.2e-3, "swiglu": 2e-3, "attention": 1.4e-3, "batch_attention": 1.4e-3}.get(
        case["kind"], 0.02)}


# ------------------------------------------------- block formats (public ggml)

def _random_blocks(t, n, k, gen):
    """GGUF bytes of an (n, k) matrix with N(0, 0.02) values, made on the GPU."""
    dev = "cuda"
    if t == "F16":
        return (torch.randn(n, k, generator=gen, device=dev, dtype=torch.float16) * 0.02).view(torch.uint8)

    def f16_bytes(v):
        return v.to(torch.float16).view(torch.uint8).reshape(*v.shape[:-1], -1)

    def codes(shape, mean, std, lo, hi):
        return torch.randn(shape, generator=gen, device=dev, dtype=torch.float16).mul_(std).add_(mean).round_().clamp_(lo, hi)

    nb = n * k // BLOCK[t][0]
    spread = 0.8 + 0.4 * torch.rand(nb, 1, generator=gen, device=dev)
    if t == "Q8_0":
        q = codes((nb, 32), 0, 45, -127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([f16_bytes(spread * 4.4e-4), q], 1)
    if t == "Q4_K":
        sc = torch.randint(36, 61, (nb, 8), generator=gen, device=dev, dtype=torch.int32)
        mn = (sc + torch.randint(-3, 4, (nb, 8), generator=gen, device=dev, dtype=torch.int32)).clamp_(0, 63)
        lo, hi = slice(0, 4), slice(4, 8)
        scales = torch.cat([sc[:, lo] | ((sc[:, hi] >> 4) << 6), mn[:, lo] | ((mn[:, hi] >> 4) << 6),
                            (sc[:, hi] & 15) | ((mn[:, hi] & 15) << 4)], 1).to(torch.uint8)
        q = codes((nb, 4, 2, 32), 7.5, 3.2, 0, 15).to(torch.uint8)
        qs = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(nb, 128)
        return torch.cat([f16_bytes(spread * 1.17e-4), f16_bytes(spread * 8.75e-4), scales, qs], 1)
    q = codes((nb, 2, 4, 32), 32, 10, 0, 63).to(torch.uint8)
    ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
    qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
    sc = torch.randint(70, 128, (nb, 16), generator=gen, device=dev, dtype=torch.int32)
    sc = torch.where(torch.rand(nb, 16, generator=gen, device=dev) < 0.5, sc, -sc).to(torch.int8).view(torch.uint8)
    return torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), sc, f16_bytes(spread * 2e-5)], 1)


def _dequant64(t, raw, n, k):
    """The (n, k) values of GGUF bytes in 64 bits."""
    if t == "F16":
        return raw.view(torch.float16).reshape(n, k).double()
    be, bb = BLOCK[t]
    b = raw.reshape(-1, bb)
    nb = b.shape[0]

    def f16(lo):
        return b[:, lo:lo + 2].contiguous().view(torch.float16).double()

    if t == "Q8_0":
        return (f16(0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(n, k)
    if t == "Q4_K":
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = b[:, 16:].reshape(nb, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(nb, 8, 32).double()
        return ((f16(0) * sc).unsqueeze(2) * q - (f16(2) * mn).unsqueeze(2)).reshape(n, k)
    ql, qh = b[:, :128].reshape(nb, 2, 2, 32), b[:, 128:192].reshape(nb, 2, 1, 32)
    q = torch.cat([ql & 15, ql >> 4], 2) | torch.cat([((qh >> s) & 3) << 4 for s in (0, 2, 4, 6)], 2)
    q = (q.double() - 32).reshape(nb, 16, 16)
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    return ((f16(208) * sc).unsqueeze(2) * q).reshape(n, k)


# ------------------------------------------------------------------- prepare

def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _lens(case):
    """Ragged context lengths, from half of ctx to ctx, the longest first."""
    r, ctx = case["rows"], case["ctx"]
    return [max(1, ctx - (ctx // 2) * ((7 * i) % r) // r) for i in range(r)]


def _carrier(t, raw, n, k):
    if t == "F16":
        return raw
    out = torch.empty_like(raw)
    _native.bx_check(_native.hip().bx_repack_gguf_rows(TYPES[t], _ptr(raw), _ptr(out), n, k, _stream()), "repack")
    return out


def _linear_inputs(case, seed):
    gen = _gen(seed)
    mats = 2 if case["kind"] == "swiglu" else 1
    x = torch.randn(case["rows"], case["k"], generator=gen, device="cuda", dtype=torch.float16)
    return x, [[_random_blocks(case["type"], case["n"], case["k"], gen) for _ in range(mats)]
               for _ in range(case["layers"])]


def _attention_inputs(case, seed):
    gen = _gen(seed)
    keys, w = case["rows"] + case["past"], case["n_kv"] * HEAD_DIM

    def rand(rows, cols):
        return torch.randn(rows, cols, generator=gen, device="cuda", dtype=torch.float16)

    return rand(case["rows"], case["n_q"] * HEAD_DIM), rand(keys, w), rand(keys, w)


def _rope_tables(rows):
    pos = torch.arange(rows, dtype=torch.float64, device="cuda")
    ang = pos[:, None] * THETA ** (-torch.arange(0, HEAD_DIM, 2, dtype=torch.float64, device="cuda") / HEAD_DIM)
    return ang.cos().float(), ang.sin().float()


def _batch_attention_inputs(case, seed):
    gen = _gen(seed)
    rows, cap, w = case["rows"], case["ctx"] + 64, case["n_kv"] * HEAD_DIM

    def rand(*shape):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float16)

    lens = torch.tensor(_lens(case), dtype=torch.int32, device="cuda")
    base = torch.arange(rows, dtype=torch.int64, device="cuda") * cap
    gains = [1 + 0.1 * rand(HEAD_DIM) for _ in range(2)]
    return dict(q=rand(rows, case["n_q"] * HEAD_DIM), k=rand(rows, w), v=rand(rows, w), K=rand(rows * cap, w),
                V=rand(rows * cap, w), lens=lens, base=base, gains=gains, cap=cap, tables=_rope_tables(cap))


def _checkpoint(name):
    """The synthetic checkpoint's file, written once per machine."""
    path = os.path.join(tempfile.gettempdir(), "brolm_cases_%s.gguf" % name)
    if not os.path.exists(path):
        tmp = "%s.%d" % (path, os.getpid())
        ba.write_synth_qwen3(ba.SynthSpec(vocab=VOCAB, layers=LAYERS, n_q=HEADS, n_kv=KV_HEADS, head_dim=HEAD_DIM,
                                          eps=EPS, theta=THETA, **MODELS[name]), tmp)
        os.replace(tmp, path)
    return path


def _model(name):
    path = _checkpoint(name)
    ba.init()
    m = ba.Qwen3Model(ba.Qwen3Config.from_gguf(path))
    m.load_weights(path)
    return m


def _prompts(case, seed):
    """Token ids of each sequence; the last one is the step's token."""
    rng = np.random.default_rng(int(seed))
    lens = {"prompt": lambda: [case["rows"] - 1], "decode": lambda: [case["ctx"]], "batch": lambda: _lens(case)}
    return [rng.integers(0, VOCAB, n + 1).astype(np.int32) for n in lens[case["kind"]]()]


def prepare(case, seed):
    kind = case["kind"]
    hip = _native.hip()
    s = dict(case=case, stream=_stream())
    if kind in ("linear", "swiglu"):
        x, raws = _linear_inputs(case, seed)
        s["x"] = x
        s["w"] = [[_carrier(case["type"], r, case["n"], case["k"]) for r in layer] for layer in raws]
        s["y"] = torch.empty(case["layers"], case["rows"], case["n"], device="cuda", dtype=torch.float16)
        nb = int(hip.bx_linear_workspace_bytes())
        s["ws"] = torch.empty(nb, dtype=torch.uint8, device="cuda")
        s["ws_bytes"] = C.c_size_t(nb)
        _native.bx_check(hip.bx_linear_workspace_init(_ptr(s["ws"]), s["ws_bytes"], s["stream"]), "workspace")
    elif kind == "attention":
        s["q"], s["k"], s["v"] = _attention_inputs(case, seed)
        s["out"] = torch.empty_like(s["q"])
        keys = case["rows"] + case["past"]
        s["ws"] = torch.empty(int(hip.bx_attention_workspace_bytes(case["rows"], case["n_q"], HEAD_DIM, keys)),
                              dtype=torch.uint8, device="cuda")
    elif kind == "batch_attention":
        s.update(_batch_attention_inputs(case, seed))
        s["out"] = torch.empty_like(s["q"])
        nb = int(hip.bx_batch_attention_workspace_bytes(case["rows"], case["n_q"], case["n_kv"], HEAD_DIM, s["cap"]))
        s["ws"] = torch.zeros(nb, dtype=torch.uint8, device="cuda")
    else:
        m = s["model"] = _model(case["model"])
        s["ids"] = _prompts(case, seed)
        if kind == "batch":
            m.allocate_batch(case["rows"], case["ctx"] + 64)
            for i, ids in enumerate(s["ids"]):
                m.prefill_slot(i, ids[:-1])
            s["tokens"], s["slots"] = [int(i[-1]) for i in s["ids"]], list(range(case["rows"]))
        else:
            m.allocate_cache(4096)
            if kind == "decode":
                m.forward_last(s["ids"][0][:-1])
    return s


# ------------------------------------------------------------------- run

def run(s):
    case = s["case"]
    kind = case["kind"]
    hip = _native.hip()
    if kind == "linear":
        x, ws = _ptr(s["x"]), _ptr(s["ws"])
        for w, y in zip(s["w"], s["y"]):
            _native.bx_check(hip.bx_linear_f16(TYPES[case["type"]], _ptr(w[0]), None, x, _ptr(y), case["rows"],
                                               case["n"], case["k"], ws, s["ws_bytes"], s["stream"]), "linear")
        return s["y"]
    if kind == "swiglu":
        x, ws = _ptr(s["x"]), _ptr(s["ws"])
        for w, y in zip(s["w"], s["y"]):
            _native.bx_check(hip.bx_linear_swiglu_f16(TYPES[case["type"]], _ptr(w[0]), _ptr(w[1]), x, _ptr(y),
                                                      case["rows"], case["n"], case["k"], ws, s["ws_bytes"],
                                                      s["stream"]), "swiglu")
        return s["y"]
    if kind == "attention":
        q, k, v, out, ws = (_ptr(s[n]) for n in ("q", "k", "v", "out", "ws"))
        rows, keys, nq, nkv = case["rows"], case["rows"] + case["past"], case["n_q"], case["n_kv"]
        if case["causal"]:
            rc = hip.bx_attention_decode_f16(q, k, v, rows, keys, nq, nkv, HEAD_DIM, 0.0, 0, out, ws, s["stream"])
        else:
            rc = hip.bx_attention_gqa_f16(q, k, v, rows, keys, nq, nkv, HEAD_DIM, 0, out, ws, s["stream"])
        _native.bx_check(rc, "attention")
        return s["out"]
    if kind == "batch_attention":
        rc = hip.bx_batch_attention_f16(_ptr(s["q"]), _ptr(s["k"]), _ptr(s["v"]), case["rows"], HEAD_DIM, case["n_q"],
                                        case["n_kv"], _ptr(s["gains"][0]), _ptr(s["gains"][1]), EPS, _ptr(s["lens"]),
                                        _ptr(s["base"]), s["cap"], _ptr(s["tables"][0]), _ptr(s["tables"][1]),
                                        s["cap"], _ptr(s["K"]), _ptr(s["V"]), case["rows"] * s["cap"], _ptr(s["out"]),
                                        _ptr(s["ws"]), s["stream"])
        _native.bx_check(rc, "batch attention")
        return s["out"], s["K"], s["V"]
    m = s["model"]
    if kind == "prompt":
        m.reset_cache()
        return m.forward_last(s["ids"][0])
    if kind == "decode":
        m.truncate_cache(case["ctx"])
        return m.forward_last(s["ids"][0][-1:])
    for slot, ids in zip(s["slots"], s["ids"]):
        m.truncate_slot(slot, len(ids) - 1)
    return m.forward_batch(s["tokens"], s["slots"])


# ------------------------------------------------------- the same in 64 bits

def _attend64(q, k, v, n_q, n_kv, past, causal):
    """softmax(q k^T / sqrt(d)) v per head; rows of q follow `past` keys."""
    rows, keys = q.shape[0], k.shape[0]
    out = torch.empty_like(q)
    hidden = None
    if causal:
        at = torch.arange(rows, device="cuda")[:, None] + past
        hidden = torch.arange(keys, device="cuda")[None, :] > at
    for h in range(n_q):
        g, c = h // (n_q // n_kv), slice(h * HEAD_DIM, (h + 1) * HEAD_DIM)
        e = slice(g * HEAD_DIM, (g + 1) * HEAD_DIM)
        s = (q[:, c] @ k[:, e].t()) / math.sqrt(HEAD_DIM)
        if hidden is not None:
            s.masked_fill_(hidden, -math.inf)
        out[:, c] = torch.softmax(s, 1) @ v[:, e]
    return out


def _rms(x, gamma):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gamma


def _exact_batch_attention(case, seed):
    s = _batch_attention_inputs(case, seed)
    cos, sin = (t.double() for t in s["tables"])
    rows, nq, nkv = case["rows"], case["n_q"], case["n_kv"]
    pos = s["lens"].long() - 1

    def turned(x, heads, gain):
        # the kernel's cache holds (even, odd) pairs of a head side by side
        x = _rms(x.double().reshape(rows, heads, HEAD_DIM), gain.double())
        a, b, c, d = x[..., 0::2], x[..., 1::2], cos[pos][:, None], sin[pos][:, None]
        return torch.stack([a * c - b * d, a * d + b * c], -1).reshape(rows, -1)

    q, k = turned(s["q"], nq, s["gains"][0]), turned(s["k"], nkv, s["gains"][1])
    K, V = s["K"].double(), s["V"].double()
    K[s["base"] + pos], V[s["base"] + pos] = k, s["v"].double()
    out = torch.empty_like(q)
    for r, (b, n) in enumerate(zip(s["base"].tolist(), s["lens"].tolist())):
        out[r:r + 1] = _attend64(q[r:r + 1], K[b:b + n], V[b:b + n], nq, nkv, n - 1, False)
    return out, K, V


def _gguf(path):
    """{tensor name: (ggml type, rows, cols, byte offset)} of a GGUF v3 file."""
    with open(path, "rb") as f:
        def num(fmt):
            return struct.unpack("<" + fmt, f.read(struct.calcsize(fmt)))[0]

        def text():
            return f.read(num("Q")).decode("utf-8", "replace")

        fixed = {0: "B", 1: "b", 2: "H", 3: "h", 4: "I", 5: "i", 6: "f", 7: "?", 10: "Q", 11: "q", 12: "d"}

        def value(t):
            if t == 8:
                return text()
            if t == 9:
                e, n = num("I"), num("Q")
                return [value(e) for _ in range(n)]
            return num(fixed[t])

        f.read(8)
        n_tensors, n_meta = num("Q"), num("Q")
        meta = {}
        for _ in range(n_meta):
            key = text()
            meta[key] = value(num("I"))
        table = {}
        for _ in range(n_tensors):
            name = text()
            dims = [num("Q") for _ in range(num("I"))]
            table[name] = (num("I"), int(np.prod(dims[1:], dtype=np.int64)), dims[0], num("Q"))
        align = meta.get("general.alignment", 32)
        start = (f.tell() + align - 1) // align * align
    return {n: (t, r, c, start + o) for n, (t, r, c, o) in table.items()}


def _exact_logits(case, seed):
    """The causal decoder over whole sequences, logits of each one's last token."""
    path = _checkpoint(case["model"])
    table = _gguf(path)
    data = np.memmap(path, np.uint8, "r")
    names = {v: n for n, v in TYPES.items()}

    def weight(name):
        t, n, k, at = table[name]
        if t == 0:
            return torch.from_numpy(np.array(data[at:at + 4 * n * k])).cuda().view(torch.float32).double().reshape(n, k)
        be, bb = BLOCK[names[t]]
        return _dequant64(names[t], torch.from_numpy(np.array(data[at:at + n * k // be * bb])).cuda(), n, k)

    seqs = _prompts(case, seed)
    ids = torch.from_numpy(np.concatenate(seqs).astype(np.int64)).cuda()
    ends = np.cumsum([len(x) for x in seqs])
    pos = torch.cat([torch.arange(len(x), device="cuda") for x in seqs])
    ang = pos.double()[:, None] * THETA ** (-torch.arange(0, HEAD_DIM, 2, dtype=torch.float64, device="cuda") / HEAD_DIM)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def heads(x, n, gain):
        x = _rms(x.reshape(-1, n, HEAD_DIM), gain)
        a, b = x.chunk(2, -1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1).reshape(-1, n * HEAD_DIM)

    emb = weight("token_embd.weight")
    h = emb[ids]
    if not MODELS[case["model"]]["tied"]:
        del emb
    for layer in range(LAYERS):
        def w(role):
            return weight("blk.%d.%s.weight" % (layer, role))

        x = _rms(h, w("attn_norm").reshape(-1))
        q = heads(x @ w("attn_q").t(), HEADS, w("attn_q_norm").reshape(-1))
        k = heads(x @ w("attn_k").t(), KV_HEADS, w("attn_k_norm").reshape(-1))
        v = x @ w("attn_v").t()
        a = torch.cat([_attend64(q[e - len(x_):e], k[e - len(x_):e], v[e - len(x_):e], HEADS, KV_HEADS, 0, True)
                       for e, x_ in zip(ends.tolist(), seqs)])
        h = h + a @ w("attn_output").t()
        x = _rms(h, w("ffn_norm").reshape(-1))
        h = h + (torch.nn.functional.silu(x @ w("ffn_gate").t()) * (x @ w("ffn_up").t())) @ w("ffn_down").t()
    last = _rms(h[torch.from_numpy(ends - 1).cuda()], weight("output_norm.weight").reshape(-1))
    logits = last @ (emb if MODELS[case["model"]]["tied"] else weight("output.weight")).t()
    logits = logits.cpu().numpy()
    return logits if case["kind"] == "batch" else logits[0]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear", "swiglu"):
        x, raws = _linear_inputs(case, seed)
        x = x.double()
        out = torch.empty(case["layers"], case["rows"], case["n"], device="cuda", dtype=torch.float64)
        for i, layer in enumerate(raws):
            y = [x @ _dequant64(case["type"], r, case["n"], case["k"]).t() for r in layer]
            out[i] = y[0] if kind == "linear" else torch.nn.functional.silu(y[0]) * y[1]
        return out
    if kind == "attention":
        q, k, v = (t.double() for t in _attention_inputs(case, seed))
        return _attend64(q, k, v, case["n_q"], case["n_kv"], case["past"], case["causal"])
    if kind == "batch_attention":
        return _exact_batch_attention(case, seed)
    return _exact_logits(case, seed)
