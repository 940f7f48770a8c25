"""The work a user of this library has it do, as measurable cases.

Two groups:

* single operations of the forward path through the C ABI (`yl_quantize`,
  `yl_rmsnorm_quantize`, `yl_swiglu_quantize`, `yl_matmul`, `yl_matmul_f32`,
  `yl_attention_noalloc`), on device buffers, as a program that builds its own
  pipeline calls them: one decoded token, a chat turn of some tens of tokens,
  a long prompt;
* whole calls of the model API (`Transformer.forward_x` on a session):
  one decode step, and a conversation's first prompt (reset, then prefill),
  on the SmolLM2-135M-shaped and Llama-3.2-1B-shaped models.

Every result of these entry points is specified to the bit (each sum in the
reference's operation order, each product and sum rounded on its own), so
`tolerance` is "exact".
"""
import ctypes
import math

import numpy as np
import torch

import yallma3_mini_inference_amd as Y
from yallma3_mini_inference_amd import synth
from yallma3_mini_inference_amd.weight_type import QuantizedWeight, WeightFormat

FMT = {"q8": WeightFormat.Q8_0, "q4": WeightFormat.Q4_0}
VALUE_BYTES = {"q8": 1.0, "q4": 0.5}   # weight bytes per element, scales apart
EPS = 1e-5
DEV = "cuda"


def listed():
    return [
        # one token's activation row at dim 2048, ahead of a projection: the smallest call
        dict(name="quantize_row", op="quantize", fmt="q8", n=2048),
        # a prompt's rows before the QKV or gate/up projection
        dict(name="norm_prompt", op="norm", fmt="q8", batch=500, size=2048),
        # a chat turn's FFN activations at hidden 8192, for a Q4_0 down projection
        dict(name="swiglu_turn", op="swiglu", fmt="q4", batch=77, hidden=8192),
        # one decoded token through a gate or up projection of the 1B shape
        dict(name="matmul_row_q8", op="matmul", fmt="q8", batch=1, o=8192, n=2048),
        # a chat turn through an output projection of the 8B shape
        dict(name="matmul_turn_q4", op="matmul", fmt="q4", batch=24, o=4096, n=4096),
        # a long prompt, not a multiple of any tile, through a gate or up projection of the 1B shape
        dict(name="matmul_prompt_q8", op="matmul", fmt="q8", batch=1000, o=8192, n=2048),
        # a prompt through an F16 model's output projection
        dict(name="matmul_f16_prompt", op="matmul_f16", batch=190, o=2048, n=2048),
        # a second chat turn: 45 tokens onto a conversation of 1200, 1B head layout
        dict(name="attention_turn", op="attention", batch=45, start=1200, heads=32, kv_heads=8, hd=64),
        # one decoded token at a context of 8192, 8B head layout
        dict(name="attention_decode_long", op="attention", batch=1, start=8191, heads=32, kv_heads=8, hd=128),
        # one decode step of the 1B model in a conversation of some 600 positions, logits to the host
        dict(name="decode_1b", op="decode", model="llama32_1b", start=600),
        # the first turn of a conversation: system text and a question
        dict(name="turn_1b", op="prompt", model="llama32_1b", tokens=41),
        # a document as the prompt
        dict(name="prefill_1b", op="prompt", model="llama32_1b", tokens=2000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the operation by its share of the list, sizes over the
    whole range (by their logarithm), the widths those of the repository's
    configurations or odd ones."""
    op = rng.choice(["quantize", "norm", "swiglu", "matmul", "matmul", "matmul", "matmul_f16", "attention", "attention",
                     "decode", "prompt", "prompt"])
    widths = [576, 1536, 2048, 4096, 8192, 32 * rng.randint(4, 256)]
    fmt = rng.choice(["q8", "q4"])
    if op == "quantize":
        return dict(op=op, fmt=fmt, n=32 * _log_int(rng, 1, 131072))
    if op == "norm":
        return dict(op=op, fmt=fmt, batch=_log_int(rng, 1, 2048), size=rng.choice(widths))
    if op == "swiglu":
        return dict(op=op, fmt=fmt, batch=_log_int(rng, 1, 1024), hidden=rng.choice([1536, 8192, 14336, 32 * rng.randint(4, 400)]))
    if op == "matmul":
        # (n: the shapes of the configurations, or any number of 32-blocks; o any)
        n = rng.choice([576, 1536, 2048, 4096, 8192, 32 * rng.randint(2, 256)])
        o = rng.choice([576, 2048, 3072, 4096, 8192, rng.randint(33, 8192)])
        return dict(op=op, fmt=fmt, batch=_log_int(rng, 1, 1000), o=o, n=n)
    if op == "matmul_f16":
        n = rng.choice([576, 2048, 8192, 32 * rng.randint(2, 128)])
        return dict(op=op, batch=_log_int(rng, 1, 512), o=rng.choice([576, 2048, 3072, rng.randint(33, 8192)]), n=n)
    if op == "attention":
        heads, kv_heads, hd = rng.choice([(32, 8, 64), (32, 8, 128), (9, 3, 64), (8, 8, 64)])
        if rng.random() < 0.4:
            return dict(op=op, batch=1, start=_log_int(rng, 1, 8000), heads=heads, kv_heads=kv_heads, hd=hd)
        # (within the call's fixed scratch: keys and scores below 64 MiB)
        batch = _log_int(rng, 2, 200)
        return dict(op=op, batch=batch, start=_log_int(rng, 1, 1400), heads=heads, kv_heads=kv_heads, hd=hd)
    model = rng.choice(["smollm2_135m", "llama32_1b"])
    if op == "decode":
        return dict(op=op, model=model, start=_log_int(rng, 2, 1700))
    return dict(op=op, model=model, tokens=_log_int(rng, 2, 2000))


# ---------------------------------------------------------------- inputs

def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000 + salt)
    return g


def _normal(seed, salt, *shape):
    return torch.randn(*shape, generator=_gen(seed, salt), device=DEV, dtype=torch.float32)


def _weights(fmt, seed, o, n):
    """A quantized [o][n] matrix of N(0, 0.02) weights: integer values (Q4_0:
    nibbles 0..15, the value itself, no offset) and f16 block scales."""
    w = _normal(seed, 1, o, n // 32, 32) * 0.02
    top = w.abs().amax(-1, keepdim=True)
    if fmt == "q8":
        d = (top / 127).half()
        q = (w / d.float()).round().clamp(-127, 127).to(torch.int8)
    else:
        d = (top / 8).half()
        q = ((w / d.float()).round() + 8).clamp(0, 15).to(torch.int8)
    return q, d


def _gguf_blocks(fmt, q, d):
    """GGUF blocks: the f16 scale, then 32 int8 or 16 bytes (element 2j the low nibble of byte j)."""
    body = q.view(torch.uint8) if fmt == "q8" else (q[..., 0::2] | (q[..., 1::2] << 4)).view(torch.uint8)
    return torch.cat([d.view(torch.uint8), body], -1).contiguous().cpu().numpy()


def _activations(fmt, seed, batch, n):
    """Rows of N(0, 1) quantized in blocks of 32: int8 values and f32 scales."""
    x = _normal(seed, 2, batch, n // 32, 32)
    s = x.abs().amax(-1, keepdim=True) / (127 if fmt == "q8" else 7)
    lim = 127 if fmt == "q8" else 7
    q = (x / s).round().clamp(-lim, lim).to(torch.int8)
    return q.reshape(batch, n).contiguous(), s.reshape(batch, n // 32).contiguous()


_models = {}


def _model(name):
    """The model a program has loaded (its file is written on first use)."""
    if name not in _models:
        _models[name] = Y.Transformer(synth.ensure(name))
    return _models[name]


def _fill_cache(session, seed, positions):
    """K and V of the conversation so far: N(0, 1) below `positions`, zeros after."""
    m = session.model
    sh = m.shape
    kv, ld = sh.n_kv_heads * sh.head_size, (sh.ctx_len + 3) & ~3
    k = torch.zeros(sh.n_layers, kv, ld, device=DEV)   # keys are held transposed
    v = torch.zeros(sh.n_layers, ld, kv, device=DEV)
    k[:, :, :positions] = _normal(seed, 3, sh.n_layers, kv, positions)
    v[:, :positions] = _normal(seed, 4, sh.n_layers, positions, kv)
    torch.cuda.synchronize()
    kp, vp, floats = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    L = Y.lib()
    _ok(L.yl_session_kv(session._h, ctypes.byref(kp), ctypes.byref(vp), ctypes.byref(floats)))
    _ok(L.yl_memcpy_d2d(kp, k.data_ptr(), 4 * k.numel()))
    _ok(L.yl_memcpy_d2d(vp, v.data_ptr(), 4 * v.numel()))


def _ok(status):
    if status != 0:
        raise RuntimeError("yallma3: %d: %s" % (status, Y.lib().yl_last_error().decode()))


DECODE_STEPS = 256   # positions a decode case walks before it starts over


def prepare(case, seed):
    op = case["op"]
    s = {"op": op, "case": case}
    if op in ("quantize", "norm", "swiglu"):
        rows, width = (1, case["n"]) if op == "quantize" else (case["batch"], case.get("size") or case.get("hidden"))
        s["x"] = _normal(seed, 5, rows, width)
        if op == "norm":
            s["w"] = 1.0 + 0.1 * _normal(seed, 6, width)
        if op == "swiglu":
            s["up"] = _normal(seed, 6, rows, width)
        s["q"] = torch.empty(rows, width, device=DEV, dtype=torch.int8)
        s["scale"] = torch.empty(rows, width // 32, device=DEV)
    elif op == "matmul":
        fmt, b, o, n = case["fmt"], case["batch"], case["o"], case["n"]
        s["w"] = QuantizedWeight.upload_gguf(FMT[fmt], _gguf_blocks(fmt, *_weights(fmt, seed, o, n)), o, n)
        s["xq"], s["xs"] = _activations(fmt, seed, b, n)
        s["out"] = torch.empty(b, o, device=DEV)
    elif op == "matmul_f16":
        b, o, n = case["batch"], case["o"], case["n"]
        s["w"] = QuantizedWeight.upload_f16((_normal(seed, 1, o, n) * 0.02).half().cpu().numpy(), o, n)
        s["x"] = _normal(seed, 2, b, n)
        s["out"] = torch.empty(b, o, device=DEV)
    elif op == "attention":
        seq, kv = case["start"] + case["batch"], case["kv_heads"] * case["hd"]
        s["q"] = _normal(seed, 1, case["batch"], case["heads"] * case["hd"])
        s["k"] = _normal(seed, 2, seq, kv)
        s["v"] = _normal(seed, 3, seq, kv)
        s["out"] = torch.empty_like(s["q"])
    else:
        m = _model(case["model"])
        s["model"], s["session"] = m, m.create_session()
        rng = np.random.default_rng(seed)
        if op == "decode":
            _fill_cache(s["session"], seed, case["start"])
            s["token"] = int(rng.integers(0, m.vocab_size()))
            s["step"] = 0
        else:
            s["tokens"] = rng.integers(0, m.vocab_size(), case["tokens"]).astype(np.uint32)
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    c, op, L = s["case"], s["op"], Y.lib()
    if op == "quantize":
        _ok(L.yl_quantize(int(FMT[c["fmt"]]), s["q"].data_ptr(), s["scale"].data_ptr(), s["x"].data_ptr(), c["n"], 32, None))
        return s["q"], s["scale"]
    if op == "norm":
        _ok(L.yl_rmsnorm_quantize(s["x"].data_ptr(), s["w"].data_ptr(), c["size"], EPS, c["batch"], None,
                                  int(FMT[c["fmt"]]), s["q"].data_ptr(), s["scale"].data_ptr(), None))
        return s["q"], s["scale"]
    if op == "swiglu":
        _ok(L.yl_swiglu_quantize(s["x"].data_ptr(), s["up"].data_ptr(), c["hidden"], c["batch"], None,
                                 int(FMT[c["fmt"]]), s["q"].data_ptr(), s["scale"].data_ptr(), None))
        return s["q"], s["scale"]
    if op == "matmul":
        s["out"].zero_()   # the columns accumulate onto `out`
        _ok(L.yl_matmul(s["out"].data_ptr(), int(FMT[c["fmt"]]), s["xq"].data_ptr(), s["xs"].data_ptr(), c["batch"],
                        s["w"]._h, c["n"], c["o"], 32, None))
        return s["out"]
    if op == "matmul_f16":
        _ok(L.yl_matmul_f32(s["out"].data_ptr(), s["x"].data_ptr(), c["batch"], s["w"]._h, c["n"], c["o"], None))
        return s["out"]
    if op == "attention":
        _ok(L.yl_attention_noalloc(s["out"].data_ptr(), s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                                   c["batch"], c["start"], c["heads"], c["kv_heads"], c["hd"], 1.0 / math.sqrt(c["hd"]), None))
        return s["out"]
    if op == "decode":
        # one step of a greedy loop on the host: the logits, and the token fed to the next step
        logits = s["model"].forward_x([s["token"]], c["start"] + s["step"], s["session"])
        s["step"] = (s["step"] + 1) % DECODE_STEPS
        s["token"] = int(logits.argmax())
        return logits
    # a new conversation in a kept session
    s["session"].reset()
    return s["model"].forward_x(s["tokens"], 0, s["session"])


# ---------------------------------------------------------------- what it takes

def _attended(batch, start):
    """(query, position) pairs of a causal batch."""
    return batch * start + batch * (batch + 1) // 2


def work(case):
    op = case["op"]
    if op == "quantize":
        n = case["n"]
        return {"bytes": 4 * n + n + n // 8, "flops": 4 * n}
    if op == "norm":
        b, n = case["batch"], case["size"]
        return {"bytes": b * (4 * n + n + n // 8) + 4 * n, "flops": 8 * b * n}
    if op == "swiglu":
        b, n = case["batch"], case["hidden"]
        return {"bytes": b * (8 * n + n + n // 8), "flops": 10 * b * n}
    if op == "matmul":
        b, o, n = case["batch"], case["o"], case["n"]
        return {"bytes": o * n * VALUE_BYTES[case["fmt"]] + o * n // 16 + b * (n + n // 8) + 4 * b * o, "flops": 2 * b * o * n}
    if op == "matmul_f16":
        b, o, n = case["batch"], case["o"], case["n"]
        return {"bytes": 2 * o * n + 4 * b * (n + o), "flops": 2 * b * o * n}
    if op == "attention":
        h, kvh, hd, b, start = case["heads"], case["kv_heads"], case["hd"], case["batch"], case["start"]
        return {"bytes": 8 * b * h * hd + 8 * (start + b) * kvh * hd, "flops": 4 * _attended(b, start) * h * hd}
    c = synth.CONFIGS[case["model"]]
    b, start = (1, case["start"]) if op == "decode" else (case["tokens"], 0)
    hd = c.dim // c.n_heads
    kv = c.n_kv_heads * hd
    params = c.n_layers * (c.dim * (2 * c.dim + 2 * kv) + 3 * c.dim * c.hidden)
    # weights once, the tied table once (logits), K and V of the attended positions, the logits
    return {"bytes": (params + c.vocab * c.dim) * 34 // 32 + 8 * c.n_layers * (start + b) * kv + 4 * c.vocab,
            "flops": 2 * b * params + 2 * c.vocab * c.dim + 4 * c.n_layers * _attended(b, start) * c.dim}


def tolerance(case):
    return "exact"


# ---------------------------------------------------------------- in 64 bits

def _quantized_scales(rows, fmt):
    """Block scales of float64 rows (the integers have no 64-bit value of their own)."""
    return rows.reshape(rows.shape[0], -1, 32).abs().amax(-1) / (127 if fmt == "q8" else 7)


def exact(case, seed):
    op = case["op"]
    if op in ("decode", "prompt"):
        # a whole quantized model: one activation rounded the other way moves
        # every layer that follows, so a 64-bit pass says nothing about a result
        return None
    if op in ("quantize", "norm", "swiglu"):
        s = prepare(case, seed)
        x = s["x"].double()
        if op == "norm":
            x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * s["w"].double()
        if op == "swiglu":
            x = x * torch.sigmoid(x) * s["up"].double()
        return None, _quantized_scales(x, case["fmt"])
    if op == "matmul":
        fmt, b, o, n = case["fmt"], case["batch"], case["o"], case["n"]
        q, d = _weights(fmt, seed, o, n)
        xq, xs = _activations(fmt, seed, b, n)
        w = (q.double() * d.double()).reshape(o, n)
        x = (xq.double().reshape(b, n // 32, 32) * xs.double()[..., None]).reshape(b, n)
        return x @ w.t().contiguous()
    if op == "matmul_f16":
        b, o, n = case["batch"], case["o"], case["n"]
        return _normal(seed, 2, b, n).double() @ (_normal(seed, 1, o, n) * 0.02).half().double().t().contiguous()
    h, kvh, hd, b, start = case["heads"], case["kv_heads"], case["hd"], case["batch"], case["start"]
    seq = start + b
    q = _normal(seed, 1, b, h, hd).double()
    k = _normal(seed, 2, seq, kvh, hd).double()
    v = _normal(seed, 3, seq, kvh, hd).double()
    masked = torch.arange(seq, device=DEV)[None, :] > start + torch.arange(b, device=DEV)[:, None]
    out = torch.empty(b, h, hd, device=DEV, dtype=torch.float64)
    for i in range(h):
        j = i // (h // kvh)
        score = (q[:, i].contiguous() @ k[:, j].t().contiguous()) / math.sqrt(hd)
        out[:, i] = torch.softmax(score.masked_fill(masked, -math.inf), -1) @ v[:, j].contiguous()
    return out.reshape(b, h * hd)
