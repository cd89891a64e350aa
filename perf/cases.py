"""Performance cases of the quantized-matmul path: what a program that links
librce_qmm has it do, through the Python mirror of the C ABI.

Five kinds of work:

* ``host``    the drop-in operator on host arrays (``mm_1d`` / ``mm_batched``),
              as the reference's dispatcher calls it, result on the host;
* ``linear``  one weight on device buffers (``mm_batched_dev``): decode
              (EXACT and Q8, one to a few dozen tokens) and prefill
              (F16_MFMA, a short prompt to several thousand tokens);
* ``moe``     the grouped experts (``moe_ffn_dev`` / ``moe_swiglu_dev``) at
              prefill and decode sizes;
* ``decode``  a Llama-shaped decoder fed a sequence of tokens one by one from
              an empty cache (``TinyLlamaRuntime.forward_token_dev``).

Weights are N(0, 0.02) quantized on the GPU by plain torch below,
activations N(0, 1).  Every pass runs on the one context (and stream) a
program keeps.
"""
import math

import numpy as np
import torch

import rce_amd
from rce_amd import GgufDtype, Mode

DTYPES = {"f16": GgufDtype.F16, "bf16": GgufDtype.BF16, "q4_0": GgufDtype.Q4_0, "q8_0": GgufDtype.Q8_0,
          "q4_k": GgufDtype.Q4K, "q6_k": GgufDtype.Q6K}
MODES = {"exact": Mode.EXACT, "q8": Mode.Q8, "mfma": Mode.F16_MFMA}

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = rce_amd.Context(0)
    return _context


# ---- the cases -----------------------------------------------------------------

def listed():
    return [
        # the smallest call: the operator as the reference's dispatcher makes it, one small projection, host arrays
        {"name": "host_1024", "kind": "host", "dtype": "q8_0", "n": 1024, "k": 1024, "t": 1},
        # one decode step's FFN-up projection of a 7B model, in the reference's order
        {"name": "gemv_exact", "kind": "linear", "mode": "exact", "dtype": "q4_0", "n": 11008, "k": 4096, "t": 1, "act": "f32"},
        # the same for eight sequences decoded together
        {"name": "batch8_exact", "kind": "linear", "mode": "exact", "dtype": "q4_0", "n": 11008, "k": 4096, "t": 8, "act": "f32"},
        # a serving batch of 32 sequences on a K-quant projection, 8-bit activations
        {"name": "batch32_q8", "kind": "linear", "mode": "q8", "dtype": "q4_k", "n": 14336, "k": 4096, "t": 32, "act": "f32"},
        # an ordinary prompt
        {"name": "prefill_512", "kind": "linear", "mode": "mfma", "dtype": "q4_k", "n": 4096, "k": 4096, "t": 512, "act": "f16"},
        # a long prompt (or several packed together) through the widest projection
        {"name": "prefill_4096", "kind": "linear", "mode": "mfma", "dtype": "q4_k", "n": 14336, "k": 4096, "t": 4096, "act": "f16"},
        # a short, ragged prompt with f32 activations on a Q6_K down projection
        {"name": "prefill_77", "kind": "linear", "mode": "mfma", "dtype": "q6_k", "n": 2048, "k": 5632, "t": 77, "act": "f32"},
        # an unquantized layer at an odd prompt length
        {"name": "prefill_f16", "kind": "linear", "mode": "mfma", "dtype": "f16", "n": 6912, "k": 2560, "t": 333, "act": "f16"},
        # Mixtral-shaped experts, a prompt of 256 tokens
        {"name": "moe_256", "kind": "moe", "mode": "mfma", "dtype": "q4_0", "dtype2": "q4_0", "experts": 8, "top_k": 2,
         "d_model": 4096, "d_ff": 14336, "t": 256, "swiglu": False},
        # SwiGLU experts of a Q4_K_M file, six sequences decoded together
        {"name": "moe_decode", "kind": "moe", "mode": "q8", "dtype": "q4_k", "dtype2": "q6_k", "experts": 8, "top_k": 2,
         "d_model": 2048, "d_ff": 5632, "t": 6, "swiglu": True},
        # a whole TinyLlama-shaped model answering a short question, 8-bit activations
        {"name": "decode_64", "kind": "decode", "mode": "q8", "layers": 22, "tokens": 64, "d_model": 2048, "heads": 32,
         "kv_heads": 4, "d_ff": 5632, "vocab": 32000, "dtype": "q4_k", "head": "q6_k"},
        # a long context on eight of its layers, in the reference's order
        {"name": "decode_1024", "kind": "decode", "mode": "exact", "layers": 8, "tokens": 1024, "d_model": 2048, "heads": 32,
         "kv_heads": 4, "d_ff": 5632, "vocab": 32000, "dtype": "q4_k", "head": "q6_k"},
    ]


def _log(rng, lo, hi, step=1):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["host", "decode_linear", "decode_linear", "prefill", "prefill", "prefill", "moe", "moe", "decode"])
    quant = ["q4_0", "q8_0", "q4_k", "q6_k"]
    if kind == "host":
        return {"kind": "host", "dtype": rng.choice(quant), "n": _log(rng, 64, 4096), "k": _log(rng, 256, 4096, 256),
                "t": rng.choice([1, 1, 1, 2, 5])}
    if kind == "decode_linear":
        mode = rng.choice(["exact", "q8"])
        return {"kind": "linear", "mode": mode, "dtype": rng.choice(quant), "n": _log(rng, 256, 14336),
                "k": _log(rng, 512, 14336, 256), "t": 1 if rng.random() < 0.3 else _log(rng, 2, 16 if mode == "exact" else 64),
                "act": rng.choice(["f32", "f32", "f16"])}
    if kind == "prefill":
        dtype = rng.choice(quant + quant + ["f16", "bf16", "q8_0"])
        step = 64 if dtype in ("f16", "bf16") else 256
        c = {"kind": "linear", "mode": "mfma", "dtype": dtype, "n": _log(rng, 512, 14336), "k": _log(rng, 512, 14336, step),
             "t": _log(rng, 16, 4096), "act": rng.choice(["f16", "f16", "f32"])}
        while 2 * c["n"] * c["k"] * c["t"] > 2 * 14336 * 4096 * 4096:
            c["t"] = (c["t"] + 1) // 2
        return c
    if kind == "moe":
        mode = rng.choice(["mfma", "mfma", "q8", "exact"])
        experts = rng.choice([4, 8, 16])
        d1 = rng.choice(quant)
        return {"kind": "moe", "mode": mode, "dtype": d1, "dtype2": rng.choice([d1, d1, "q6_k"]), "experts": experts,
                "top_k": rng.choice([1, 2, 4]), "d_model": _log(rng, 768, 4096, 256),
                "d_ff": _log(rng, 768, 14336 if experts <= 8 else 4096, 256),
                "t": _log(rng, 1, 512 if mode == "mfma" else 24), "swiglu": rng.random() < 0.5}
    d_model = rng.choice([512, 1024, 2048])
    return {"kind": "decode", "mode": rng.choice(["exact", "q8"]), "layers": rng.randint(1, 6), "tokens": _log(rng, 16, 768),
            "d_model": d_model, "heads": d_model // 64, "kv_heads": rng.choice([2, 4, d_model // 64]),
            "d_ff": _log(rng, 1024, 5632, 256), "vocab": _log(rng, 4000, 32000), "dtype": rng.choice(["q4_0", "q4_k", "q8_0"]),
            "head": rng.choice(["q6_k", "q8_0"])}


# ---- GGUF weights made on the GPU -----------------------------------------------

def _f16_bytes(x):
    """[..., m] f16 values as [..., 2m] bytes."""
    return x.to(torch.float16).contiguous().view(torch.uint8)


def _make(gen, dtype, n, k):
    """N(0, 0.02) weights [n, k] in `dtype`: (bytes [n, row bytes], the fields
    they hold)."""
    w = torch.randn(n, k, device="cuda", generator=gen) * 0.02
    if dtype == "f16":
        w = w.half()
        return w.view(torch.uint8), (w,)
    if dtype == "bf16":
        w = w.bfloat16()
        return w.view(torch.uint8), (w,)
    if dtype in ("q4_0", "q8_0"):
        b = w.view(n, k // 32, 32)
        if dtype == "q8_0":
            d = (b.abs().amax(-1, keepdim=True) / 127).half()
            q = (b / d.float()).round().clamp(-127, 127).to(torch.int8)
            raw = torch.cat([_f16_bytes(d), q.view(torch.uint8)], -1)
        else:
            at = b.abs().argmax(-1, keepdim=True)
            d = (b.gather(-1, at) / -8).half()
            u = (b / d.float() + 8).round().clamp(0, 15).to(torch.uint8)
            q = u.to(torch.int8) - 8
            raw = torch.cat([_f16_bytes(d), u[..., :16] | (u[..., 16:] << 4)], -1)
        return raw.view(n, -1), (d, q)
    if dtype == "q4_k":
        b = w.view(n, k // 256, 8, 32)
        lo = (-b.amin(-1)).clamp_min(0)
        hi = (b.amax(-1) + lo) / 15
        d, dm = (hi.amax(-1, keepdim=True) / 63).half(), (lo.amax(-1, keepdim=True) / 63).half()
        sc = (hi / d.float()).round().clamp(1, 63).to(torch.uint8)
        mn = (lo / dm.float()).round().clamp(0, 63).to(torch.uint8)
        q = ((b + (dm.float() * mn).unsqueeze(-1)) / (d.float() * sc).unsqueeze(-1)).round().clamp(0, 15).to(torch.uint8)
        packed = torch.cat([(sc[..., :4] & 63) | ((sc[..., 4:] >> 4) << 6), (mn[..., :4] & 63) | ((mn[..., 4:] >> 4) << 6),
                            (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)
        qs = (q[..., 0::2, :] | (q[..., 1::2, :] << 4)).reshape(n, k // 256, 128)
        raw = torch.cat([_f16_bytes(d), _f16_bytes(dm), packed, qs], -1)
        return raw.view(n, -1), (d, dm, sc, mn, q)
    b = w.view(n, k // 256, 16, 16)  # q6_k
    top = b.gather(-1, b.abs().argmax(-1, keepdim=True)).squeeze(-1) / -32
    d = (top.abs().amax(-1, keepdim=True) / 127).half()
    sc = (top / d.float()).round().clamp(-127, 127)
    sc = torch.where(sc == 0, torch.ones_like(sc), sc).to(torch.int8)
    q = (b / (d.float() * sc).unsqueeze(-1)).round().clamp(-32, 31)
    u = (q + 32).to(torch.uint8).reshape(n, k // 256, 2, 4, 32)  # half, quarter, position
    ql = (u[..., 0:2, :] & 15) | ((u[..., 2:4, :] & 15) << 4)
    qh = (u[..., 0, :] >> 4) | ((u[..., 1, :] >> 4) << 2) | ((u[..., 2, :] >> 4) << 4) | ((u[..., 3, :] >> 4) << 6)
    raw = torch.cat([ql.reshape(n, k // 256, 128), qh.reshape(n, k // 256, 64), sc.view(torch.uint8), _f16_bytes(d)], -1)
    return raw.view(n, -1), (d, sc, q.to(torch.int8))


def _values(dtype, fields, n, k):
    """The float64 values [n, k] of _make's fields."""
    if dtype in ("f16", "bf16"):
        return fields[0].double()
    if dtype in ("q4_0", "q8_0"):
        return (fields[0].double() * fields[1]).view(n, k)
    if dtype == "q4_k":
        d, dm, sc, mn, q = fields
        return ((d.double() * sc).unsqueeze(-1) * q - (dm.double() * mn).unsqueeze(-1)).view(n, k)
    d, sc, q = fields
    return ((d.double() * sc).unsqueeze(-1) * q).view(n, k)


def _weight(gen, dtype, n, k):
    raw, _ = _make(gen, dtype, n, k)
    return rce_amd.QuantWeight.from_owned_bytes(_ctx(), raw.cpu().numpy(), DTYPES[dtype], n, k)


def _exact_weight(gen, dtype, n, k):
    return _values(dtype, _make(gen, dtype, n, k)[1], n, k)


def _q8(x):
    """Activations [.., k] as the Q8 mode holds them: f32 blocks of 32, d =
    amax / 127, integers rounded half away from zero, d kept in binary16."""
    b = x.float().reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    v = b * torch.where(d == 0, d, 1 / d)
    q = torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v))
    return (d.half().double() * q).reshape(x.shape)


# ---- preparing and running -------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _activations(gen, case):
    a = torch.randn(case["t"], case["k"], device="cuda", generator=gen)
    return a.half() if case.get("act") == "f16" else a


def _routing(gen, case):
    """Top-k of N(0, 1) router logits, softmax weights renormalized over them."""
    logits = torch.randn(case["t"], case["experts"], device="cuda", generator=gen)
    p, ids = torch.topk(torch.softmax(logits, -1), min(case["top_k"], case["experts"]), -1)
    return ids.to(torch.int32).contiguous(), (p / p.sum(-1, keepdim=True)).float().contiguous()


def _moe_shapes(case):
    one = [(case["dtype"], case["d_ff"], case["d_model"])] * (2 if case["swiglu"] else 1)
    return one + [(case["dtype2"], case["d_model"], case["d_ff"])]


def _decoder_shapes(case):
    d, ff, kv = case["d_model"], case["d_ff"], case["kv_heads"] * 64
    return {"wq": (d, d), "wk": (kv, d), "wv": (kv, d), "wo": (d, d), "ffn_gate": (ff, d), "ffn_up": (ff, d),
            "ffn_down": (d, ff)}


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = {"case": case}
    if kind in ("host", "linear"):
        s["w"] = _weight(g, case["dtype"], case["n"], case["k"])
        a = _activations(g, case)
        if kind == "host":
            s["a"], s["out"] = a.cpu().numpy(), np.empty((case["t"], case["n"]), np.float32)
        else:
            s["a"], s["out"] = a, torch.empty(case["t"], case["n"], device="cuda")
    elif kind == "moe":
        s["w"] = [[_weight(g, *shape) for _ in range(case["experts"])] for shape in _moe_shapes(case)]
        s["x"] = torch.randn(case["t"], case["d_model"], device="cuda", generator=g)
        s["ids"], s["weights"] = _routing(g, case)
        s["out"] = torch.empty_like(s["x"])
    else:
        cfg = rce_amd.TinyLlamaConfig(
            d_model=case["d_model"], vocab=case["vocab"], n_layers=case["layers"], n_q_heads=case["heads"],
            n_kv_heads=case["kv_heads"], d_head=64, rope_dim=64, rope_freq_base=10000.0, d_ff=case["d_ff"],
            context_length=case["tokens"], eps=1e-5)
        ones = np.ones(case["d_model"], np.float32)
        embd = _weight(g, case["dtype"], case["vocab"], case["d_model"])
        head = _weight(g, case["head"], case["vocab"], case["d_model"])
        blocks = [rce_amd.TinyLlamaBlock(attn_norm=ones, ffn_norm=ones, **{
            name: _weight(g, case["dtype"], n, k) for name, (n, k) in _decoder_shapes(case).items()})
            for _ in range(case["layers"])]
        s["rt"] = rce_amd.TinyLlamaRuntime(_ctx(), cfg, rce_amd.TinyLlamaWeights(embd, ones, head, blocks), MODES[case["mode"]])
        s["tokens"] = torch.randint(0, case["vocab"], (case["tokens"],), device="cuda", generator=g, dtype=torch.int32)
        s["logits"] = torch.empty(case["tokens"], case["vocab"], device="cuda")
    torch.cuda.synchronize()  # the inputs are made on torch's stream, the passes run on the context's
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "host":
        if case["t"] == 1:
            return rce_amd.mm_1d(state["a"], state["w"], state["out"][0])
        return rce_amd.mm_batched(state["a"], case["t"], state["w"], state["out"].reshape(-1))
    if kind == "linear":
        a = state["a"]
        rce_amd.mm_batched_dev(_ctx(), a.data_ptr(), GgufDtype.F16 if a.dtype == torch.float16 else GgufDtype.F32, case["t"],
                               state["w"], state["out"].data_ptr(), MODES[case["mode"]])
        return state["out"]
    if kind == "moe":
        call = rce_amd.moe_swiglu_dev if case["swiglu"] else rce_amd.moe_ffn_dev
        call(_ctx(), *state["w"], state["x"].data_ptr(), case["t"], state["ids"].data_ptr(), state["weights"].data_ptr(),
             state["ids"].shape[1], state["out"].data_ptr(), MODES[case["mode"]])
        return state["out"]
    rt, tokens, logits = state["rt"], state["tokens"].data_ptr(), state["logits"].data_ptr()
    rt.new_state()
    for i in range(case["tokens"]):
        rt.forward_token_dev(tokens + 4 * i, logits + 4 * i * case["vocab"])
    return state["logits"]


# ---- what a pass cannot do without -------------------------------------------------

def _row_bytes(dtype, k):
    return rce_amd.row_bytes(DTYPES[dtype], k)


def work(case):
    kind = case["kind"]
    if kind in ("host", "linear"):
        n, k, t = case["n"], case["k"], case["t"]
        return {"bytes": n * _row_bytes(case["dtype"], k) + t * k * (2 if case.get("act") == "f16" else 4) + 4 * t * n,
                "flops": 2 * n * k * t}
    if kind == "moe":
        e, pairs = case["experts"], case["t"] * min(case["top_k"], case["experts"])
        used = e * (1 - (1 - min(case["top_k"], e) / e) ** case["t"])  # experts that get a token
        shapes = _moe_shapes(case)
        return {"bytes": used * sum(n * _row_bytes(d, k) for d, n, k in shapes) + 8 * case["t"] * case["d_model"] + 8 * pairs,
                "flops": 2 * pairs * sum(n * k for _, n, k in shapes)}
    shapes, steps, kv = _decoder_shapes(case).values(), case["tokens"], case["kv_heads"] * 64
    per_step = case["layers"] * sum(n * _row_bytes(case["dtype"], k) for n, k in shapes)
    per_step += case["vocab"] * _row_bytes(case["head"], case["d_model"]) + 4 * case["vocab"] + _row_bytes(case["dtype"], case["d_model"])
    cache = case["layers"] * 8 * kv * (steps * (steps + 1) // 2)  # every step reads k and v of the positions so far
    flops = 2 * steps * (case["layers"] * sum(n * k for n, k in shapes) + case["vocab"] * case["d_model"])
    return {"bytes": steps * per_step + cache,
            "flops": flops + 4 * case["layers"] * case["heads"] * 64 * (steps * (steps + 1) // 2)}


def tolerance(case):
    """EXACT and Q8 fix the order of every rounding, so another correct build
    gives the same bits; a decoder's attention and norms may be summed in
    another order (in Q8 a last bit then flips an activation's rounding here
    and there, and 22 layers carry that on).  F16_MFMA rounds weights and
    activations to 11 bits: about four times its distance from 64 bits as
    measured (Q4_K 6.7e-4, Q6_K 3.4e-4, Q4_0 / Q8_0 2e-4, F16 / BF16 weights
    2e-7 with f16 activations and 2e-4 with rounded f32 ones), at most the
    ABI's budgets (2e-3, grouped experts 3e-3)."""
    mode = case.get("mode", "exact")
    if case["kind"] == "decode":
        return {"rel": 0.03, "max": 0.5} if mode == "q8" else {"rel": 5e-5, "max": 1e-3}
    if mode != "mfma":
        return "exact"
    coarse = {"q4_k": 2e-3, "q6_k": 1.4e-3, "q4_0": 8e-4, "q8_0": 8e-4}
    if case["kind"] == "moe":
        return {"rel": min(3e-3, 2 * max(coarse[case["dtype"]], coarse[case["dtype2"]]))}
    return {"rel": coarse.get(case["dtype"], 1e-5 if case["act"] == "f16" else 1e-3)}


# ---- the same in 64 bits -------------------------------------------------------------

def _linear64(x, w, mode):
    return (_q8(x) if mode == "q8" else x.double()) @ w.t()


def exact(case, seed):
    g, kind, mode = _gen(seed), case["kind"], case.get("mode", "exact")
    if kind in ("host", "linear"):
        w = _exact_weight(g, case["dtype"], case["n"], case["k"])
        y = _linear64(_activations(g, case), w, mode if case["dtype"] not in ("f16", "bf16") else "exact")
        return y.cpu().numpy()[0] if kind == "host" and case["t"] == 1 else \
            y.cpu().numpy().reshape(-1) if kind == "host" else y
    if kind == "moe":
        fields = [[(shape, _make(g, *shape)[1]) for _ in range(case["experts"])] for shape in _moe_shapes(case)]
        x = torch.randn(case["t"], case["d_model"], device="cuda", generator=g)
        ids, gates = _routing(g, case)
        out = torch.zeros(case["t"], case["d_model"], device="cuda", dtype=torch.float64)
        for e in range(case["experts"]):
            tok, j = (ids == e).nonzero(as_tuple=True)
            if not len(tok):
                continue
            w = [_values(shape[0], f, *shape[1:]) for shape, f in (m[e] for m in fields)]
            h = torch.nn.functional.silu(_linear64(x[tok], w[0], mode))
            if case["swiglu"]:
                h = h * _linear64(x[tok], w[1], mode)
            out.index_add_(0, tok, gates[tok, j].double().unsqueeze(-1) * _linear64(h, w[-1], mode))
        return out
    if mode == "q8":  # a rounding that flips in one layer travels on: 64 bits say nothing about the last bits
        return None
    d, t, kvh, heads = case["d_model"], case["tokens"], case["kv_heads"], case["heads"]
    embd = _exact_weight(g, case["dtype"], case["vocab"], d)
    head = _exact_weight(g, case["head"], case["vocab"], d)
    blocks = [{name: _make(g, case["dtype"], n, k)[1] for name, (n, k) in _decoder_shapes(case).items()}
              for _ in range(case["layers"])]
    x = embd[torch.randint(0, case["vocab"], (t,), device="cuda", generator=g, dtype=torch.int32).long()]
    del embd
    angle = torch.arange(t, device="cuda", dtype=torch.float64)[:, None] * \
        10000.0 ** (-torch.arange(32, device="cuda", dtype=torch.float64) / 32)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    causal = torch.full((t, t), -math.inf, device="cuda", dtype=torch.float64).triu(1)

    def norm(v):
        return v * (v.square().mean(-1, keepdim=True) + 1e-5).rsqrt()

    def rope(v):
        a, b = v[..., :32], v[..., 32:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    for fields in blocks:
        w = {name: _values(case["dtype"], fields[name], n, k) for name, (n, k) in _decoder_shapes(case).items()}
        h = norm(x)
        q, key, v = (h @ w[name].t() for name in ("wq", "wk", "wv"))
        q, key, v = rope(q.view(t, heads, 64)), rope(key.view(t, kvh, 64)), v.view(t, kvh, 64)
        att = torch.empty_like(q)
        for i in range(heads):
            kv = i // (heads // kvh)
            att[:, i] = torch.softmax(q[:, i] @ key[:, kv].t() / 8 + causal, -1) @ v[:, kv]
        x = x + att.reshape(t, d) @ w["wo"].t()
        h = norm(x)
        x = x + (torch.nn.functional.silu(h @ w["ffn_gate"].t()) * (h @ w["ffn_up"].t())) @ w["ffn_down"].t()
    return norm(x) @ head.t()
