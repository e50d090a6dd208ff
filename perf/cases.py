"""The work that users of this framework have it do, as measurable cases.

Kinds:
  operators  the kernel-level API (``ops``) composed as the reference's decode step, the way a program that keeps the
             reference's operator layer calls it;
  decode     one step of a model whose context is there (``LlamaModel.forward`` / ``forward_batch``);
  prompt     time to first token: ``prefill`` of a prompt, one step, its logits;
  predict    ``predict`` / ``predict_batch``: prompts in, greedy tokens out;
  stack      a block-stack model serving several prompts as one batch, then decode passes (``StackModel.feed``).

Shapes are the package's presets and the block stacks that ``bench.py --design`` times. Weights are the engine's seeded
synthetic ones; ``exact`` restates their generator and every model in float64 torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from simplellminference_amd import ops
from simplellminference_amd.model import LlamaModel, preset
from simplellminference_amd.stack import BlockSpec, StackModel, StackSpec


def listed() -> list[dict]:
    return [
        # the smallest: the reference's tiny shape in its own numerics, 4 prompt tokens and 32 greedy ones
        dict(name="predict_tiny_f32", kind="predict", model="tiny-gqa", w="f32", kv="f32", batch=1, prompt=4, spread=0,
             length=36),
        # operator by operator in the reference's numerics, two layers and the output head of a 7B model
        dict(name="operators_7b_f32", kind="operators", model="llama2-7b", w="f32", layers=2, pos=777),
        # one token of a chat at a nearly full context: the headline benchmark's shape
        dict(name="decode_7b_f16", kind="decode", model="llama2-7b", w="f16", kv="f16", batch=1, ctx=2048, pos=2047),
        # the same model served in int8, an ordinary context
        dict(name="decode_7b_i8", kind="decode", model="llama2-7b", w="i8", kv="f16", batch=1, ctx=2048, pos=1301),
        # eight chats in lockstep on a grouped-query model, ragged contexts up to 4096
        dict(name="decode_8b_f16_b8", kind="decode", model="llama3-8b", w="f16", kv="f16", batch=8, ctx=4096, pos=4095),
        # a short question to an int8 model
        dict(name="prompt_7b_i8_45", kind="prompt", model="llama2-7b", w="i8", kv="f16", ctx=2048, length=45),
        # an ordinary prompt: the length bench.py times
        dict(name="prompt_7b_f16_512", kind="prompt", model="llama2-7b", w="f16", kv="f16", ctx=2048, length=512),
        # a document, odd length, grouped-query model
        dict(name="prompt_8b_f16_3777", kind="prompt", model="llama3-8b", w="f16", kv="f16", ctx=4096, length=3777),
        # the reference's own call in its own numerics: a prompt and a short answer, fp32 weights and cache
        dict(name="predict_7b_f32", kind="predict", model="llama2-7b", w="f32", kv="f32", batch=1, prompt=75, spread=0,
             length=96),
        # eight ragged prompts scored and answered in lockstep
        dict(name="predict_8b_f16_b8", kind="predict", model="llama3-8b", w="f16", kv="f16", batch=8, prompt=121,
             spread=7, length=128),
        # block stack, one prompt of about a thousand tokens
        dict(name="stack_7b_1025", kind="stack", size="7b", slots=1, longest=1025, shortest=1025, steps=1),
        # block stack, six ragged prompts as one batch and four decode passes
        dict(name="stack_1b_b6", kind="stack", size="1b", slots=6, longest=300, shortest=17, steps=4),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng) -> dict:
    kind = rng.choice(["operators", "decode", "decode", "prompt", "prompt", "prompt", "predict", "predict", "stack"])
    if kind == "operators":
        model = rng.choice(["tiny-gqa", "small-h128-gqa", "llama2-7b", "llama3-8b"])
        return dict(kind=kind, model=model, w=rng.choice(["f32", "f16"]), layers=rng.randint(1, 2),
                    pos=_log_int(rng, 1, preset(model).max_length - 1))
    if kind == "decode":
        model, w = rng.choice([("llama2-7b", "f16"), ("llama2-7b", "i8"), ("llama3-8b", "f16"), ("llama3-8b", "i8"),
                               ("llama2-7b", "f32")])
        ctx = {"llama2-7b": 2048, "llama3-8b": 4096}[model]
        return dict(kind=kind, model=model, w=w, kv="f32" if w == "f32" else "f16",
                    batch=rng.randint(1, 8) if w == "f16" else 1, ctx=ctx, pos=_log_int(rng, 16, ctx - 1))
    if kind == "prompt":
        model, w = rng.choice([("llama2-7b", "f16"), ("llama2-7b", "i8"), ("llama3-8b", "f16"), ("llama3-8b", "i8")])
        ctx = {"llama2-7b": 2048, "llama3-8b": 4096}[model]
        return dict(kind=kind, model=model, w=w, kv="f16", ctx=ctx, length=_log_int(rng, 9, min(3777, ctx - 1)))
    if kind == "predict":
        model, w, batch = rng.choice([("tiny-gqa", "f32", 1), ("tiny-gqa", "f16", 1), ("llama2-7b", "f32", 1),
                                      ("llama3-8b", "f16", 8)])
        if batch > 1:
            batch, prompt, spread = rng.randint(2, 8), _log_int(rng, 9, 121), rng.randint(0, 7)
            return dict(kind=kind, model=model, w=w, kv="f16", batch=batch, prompt=prompt, spread=spread,
                        length=prompt + spread)
        top = 36 if model == "tiny-gqa" else 75
        prompt = _log_int(rng, 2, top)
        return dict(kind=kind, model=model, w=w, kv=w, batch=1, prompt=prompt, spread=0,
                    length=prompt + _log_int(rng, 2, 21))
    slots = rng.randint(1, 8)
    longest = _log_int(rng, 33, 1000 // slots if slots > 1 else 2000)
    return dict(kind="stack", size="1b", slots=slots, longest=longest, shortest=_log_int(rng, 1, longest),
                steps=rng.randint(0, 4))


# ---------------------------------------------------------------- inputs
def _rng(seed: int):
    return np.random.default_rng(1000003 + seed)


def _config(case):
    if "ctx" in case:
        return preset(case["model"], max_length=case["ctx"])
    return preset(case["model"])


def _decode_inputs(case, seed):
    """Token and position of every sequence: the last one at case["pos"], the others anywhere below it."""
    r, B, p = _rng(seed), case["batch"], case["pos"]
    pos = [int(v) for v in r.integers(max(1, p // 4), p + 1, B - 1)] + [p]
    return [int(v) for v in r.integers(0, _config(case).vocab_size, B)], pos


def _prompts(case, seed):
    r, V = _rng(seed), _config(case).vocab_size
    lens = [case["prompt"] + (case["spread"] * (case["batch"] - 1 - b)) // max(1, case["batch"] - 1)
            for b in range(case["batch"])]
    return [r.integers(0, V, n).astype(np.int32) for n in lens]


def _stack_inputs(case, seed):
    """Prompt of every slot and the tokens of the decode passes [steps][slots]."""
    r, n, V = _rng(seed), case["slots"], 32000
    lens = [case["longest"] - ((case["longest"] - case["shortest"]) * i) // max(1, n - 1) for i in range(n)]
    return ([r.integers(0, V, k).astype(np.int32) for k in lens],
            [[int(v) for v in r.integers(0, V, n)] for _ in range(case["steps"])])


def _stack_spec(case) -> StackSpec:
    """Retention (width / 256 heads) alternating with attention, feed-forward in every block (bench.py --design)."""
    D, ff, hd, heads, kvh, n = {"1b": (2048, 8192, 64, 32, 8, 16), "7b": (4096, 11008, 128, 32, 32, 32)}[case["size"]]
    rh = D // 256
    at = BlockSpec("attention", heads, hd, hd, kv_heads=kvh, scale=hd ** -0.5, ff=ff, ff_limit=7.0)
    rt = BlockSpec("retention", rh, 128, 256, decay=tuple(1 - 2.0 ** (-5 - 4 * i / rh) for i in range(rh)), rot_dims=128,
                   rot_base=1e4, ff=ff, ff_limit=7.0)
    return StackSpec(32000, D, (rt, at) * (n // 2), taps=4, eps=1e-6, residual_mult=0.3, max_length=2048)


def _op_tensors(case, seed, device):
    c = preset(case["model"])
    g = torch.Generator(device=device).manual_seed(seed)
    D, KV, I, V, T = c.hidden_size, c.kv_hidden_size, c.intermediate_size, c.vocab_size, c.max_length
    wd = torch.float16 if case["w"] == "f16" else torch.float32

    def rand(*shape, std, dtype=wd):
        return (torch.randn(*shape, generator=g, device=device) * std).to(dtype)
    t = {"emb": rand(V, D, std=0.02), "final": 1 + rand(D, std=0.1, dtype=torch.float32), "layers": []}
    for _ in range(case["layers"]):
        t["layers"].append({
            "n1": 1 + rand(D, std=0.1, dtype=torch.float32), "n2": 1 + rand(D, std=0.1, dtype=torch.float32),
            "q": rand(D, D, std=D ** -0.5), "k": rand(KV, D, std=D ** -0.5), "v": rand(KV, D, std=D ** -0.5),
            "o": rand(D, D, std=D ** -0.5), "up": rand(I, D, std=D ** -0.5), "gate": rand(I, D, std=D ** -0.5),
            "down": rand(D, I, std=I ** -0.5)})
    L = case["layers"]
    t["kc"] = rand(L, T, KV, std=1.0, dtype=torch.float32)
    t["vc"] = rand(L, T, KV, std=1.0, dtype=torch.float32)
    return t


def prepare(case, seed):
    kind = case["kind"]
    if kind == "operators":
        c = preset(case["model"])
        s = {"case": case, "c": c, "t": _op_tensors(case, seed, "cuda"), "token": int(_rng(seed).integers(0, c.vocab_size))}
        s["sin"], s["cos"] = ops.rope_cache(c.head_dim, c.max_length, c.rope_theta)
        return s
    if kind == "stack":
        m = StackModel(_stack_spec(case), dtype="bfloat16", batch=case["slots"], seed=seed).init()
        prompts, steps = _stack_inputs(case, seed)
        return {"case": case, "m": m, "prompts": prompts, "steps": steps}
    m = LlamaModel(config=_config(case), w_dtype=case["w"], kv_dtype=case["kv"], seed=seed, batch=case.get("batch", 1)).init()
    s = {"case": case, "m": m}
    if kind == "decode":
        s["tokens"], s["pos"] = _decode_inputs(case, seed)
        m.fill_kv_synthetic(seed, case["pos"])
    elif kind == "prompt":
        s["ids"] = _rng(seed).integers(0, _config(case).vocab_size, case["length"]).astype(np.int32)
    else:
        s["prompts"] = _prompts(case, seed)
    return s


# ---------------------------------------------------------------- one pass
def _run_operators(s):
    c, t, pos = s["c"], s["t"], s["case"]["pos"]
    x = ops.embedding(s["token"], t["emb"])
    for l, w in enumerate(t["layers"]):
        k, v = t["kc"][l, pos], t["vc"][l, pos]
        h = ops.rmsnorm(x, w["n1"], c.rms_norm_eps)
        q = ops.matmul(h, w["q"])
        ops.matmul(h, w["k"], y=k)
        ops.matmul(h, w["v"], y=v)
        ops.rope(q, k, pos, s["sin"], s["cos"], c.head_dim)
        o = ops.mha(q, t["kc"], t["vc"], l, pos, c.max_length, c.head_dim, c.num_attention_heads, c.num_key_value_heads)
        x = ops.add(x, ops.matmul(o, w["o"]))
        h = ops.rmsnorm(x, w["n2"], c.rms_norm_eps)
        a = ops.swiglu(ops.matmul(h, w["up"]), ops.matmul(h, w["gate"]))
        x = ops.add(ops.matmul(a, w["down"]), x)
    logits = ops.matmul(ops.rmsnorm(x, t["final"], c.rms_norm_eps), t["emb"])
    return {"x": x, "logits": logits, "k": t["kc"][:, pos], "v": t["vc"][:, pos], "token": ops.argmax(logits)}


def run(s):
    kind = s["case"]["kind"]
    if kind == "operators":
        return _run_operators(s)
    m = s["m"]
    if kind == "decode":
        if s["case"]["batch"] == 1:
            return {"logits": m.forward(s["tokens"][0], s["pos"][0])}
        return {"logits": m.forward_batch(s["tokens"], s["pos"])}
    if kind == "prompt":
        m.prefill(s["ids"])
        m.step()
        return {"logits": m.logits()[0]}
    if kind == "predict":
        if s["case"]["batch"] == 1:
            tokens = m.predict(s["prompts"][0], s["case"]["length"])
        else:
            tokens = m.predict_batch(s["prompts"], s["case"]["length"])
        return {"tokens": tokens, "logits": m.logits()[0]}
    lens, n = [len(p) for p in s["prompts"]], len(s["prompts"])
    out = [m.feed(range(n), [0] * n, s["prompts"], [[k - 1] for k in lens])]
    for j, toks in enumerate(s["steps"]):
        out.append(m.feed(range(n), [k + j for k in lens], [[t] for t in toks], [[0]] * n))
    return {"logits": out}


# ---------------------------------------------------------------- what a pass cannot do without
_WBYTES = {"f32": 4, "f16": 2, "i8": 1}


def work(case):
    kind = case["kind"]
    if kind == "stack":
        sp = _stack_spec(case)
        prompts, steps = _stack_inputs(case, 0)
        D, n, tok = sp.width, case["slots"], sum(len(p) for p in prompts)
        w = sum(D * (2 * b.heads * b.dim + 2 * b.heads * b.vdim + b.heads * b.vdim if b.mixer == "retention" else
                     b.heads * b.dim + b.kv_heads * (b.dim + b.vdim) + b.heads * b.vdim) + 3 * D * b.ff for b in sp.blocks)
        head, rows = sp.vocab_size * D, n * (1 + len(steps))
        att = sum(b.heads * (b.dim + b.vdim) * (len(p) + 1) * len(p) if b.mixer == "attention" else
                  4 * b.heads * b.dim * b.vdim * len(p) for b in sp.blocks for p in prompts)
        kv = sum(2 * b.kv_heads * (b.dim + b.vdim) * (tok + len(steps) * tok) for b in sp.blocks if b.mixer == "attention")
        kv += sum(8 * n * b.heads * b.dim * b.vdim * (1 + len(steps)) for b in sp.blocks if b.mixer == "retention")
        return {"bytes": 2 * (w + head) * (1 + len(steps)) + kv + 4 * rows * sp.vocab_size,
                "flops": 2 * w * (tok + n * len(steps)) + 2 * head * rows + att}
    c, wb = _config(case), _WBYTES[case["w"]]
    D, KV, I, V, hq = c.hidden_size, c.kv_hidden_size, c.intermediate_size, c.vocab_size, c.num_attention_heads * c.head_dim
    layer = D * (hq + 2 * KV) + hq * D + 3 * D * I
    L = case.get("layers", c.num_hidden_layers)
    if kind in ("operators", "decode"):
        pos = [case["pos"]] if kind == "operators" else _decode_inputs(case, 0)[1]
        kb = 4 if case.get("kv", "f32") == "f32" else 2
        ctx = sum(p + 1 for p in pos)
        return {"bytes": wb * (L * layer + V * D) + 2 * kb * L * KV * ctx + 4 * V * len(pos),
                "flops": 2 * (L * layer + V * D) * len(pos) + 4 * L * hq * ctx}
    kb = 4 if case["kv"] == "f32" else 2
    if kind == "prompt":
        n, B, gen = case["length"], 1, 1
        tok, ctx2 = n, n * (n + 1) // 2
    else:
        lens = [len(p) for p in _prompts(case, 0)]
        n, B = case["length"], case["batch"]
        tok, ctx2, gen = n * B, B * n * (n + 1) // 2, n - min(lens) + 1
    # the prompt needs the weights once, every token made after it needs them again with its context
    return {"bytes": wb * (L * layer * gen + V * D * gen) + 2 * kb * L * KV * B * (n + sum(range(n - gen + 1, n + 1))) +
            4 * B * V, "flops": 2 * L * layer * tok + 2 * V * D * B * gen + 4 * L * hq * ctx2}


def tolerance(case):
    """Four times the largest error seen against ``exact`` over the listed and some drawn cases, rounded up."""
    if case["kind"] == "stack":  # prompt rows are fp16: 1.0e-3 of the norm, 9.4e-3 of the root mean square
        return {"rel": 4e-3, "max": 4e-2}
    if case["kind"] == "operators" or case["w"] == "f32":  # fp32 throughout: 4.8e-7, 2.3e-6
        return {"rel": 2e-6, "max": 1e-5}
    # the cache rounds K and V to fp16, and a rounding may fall either way: 1.7e-4, 1.4e-3
    return {"rel": 8e-4, "max": 6e-3, "differ": 0.01}


# ---------------------------------------------------------------- float64
_M32 = 0xFFFFFFFF


def _hash32(x):
    x = x ^ (x >> 16)
    x = (x * 0x7FEB352D) & _M32
    x = x ^ (x >> 15)
    x = (x * 0x846CA68B) & _M32
    return x ^ (x >> 16)


def _normal(seed, kind, index, i0, n, std, dev):
    """Elements i0 .. i0 + n - 1 of a synthetic Llama tensor (include/sli_synth.h), fp32."""
    h0 = _hash32(((seed * 0x9E3779B9) & _M32) ^ _hash32(((kind << 16 | index) + 0x632BE5AB) & _M32))

    def u32(i):
        return _hash32(_hash32((i & _M32) ^ h0) ^ (i >> 32) ^ 0x85EBCA6B)
    i = torch.arange(i0, i0 + n, dtype=torch.int64, device=dev) * 2
    a, b = u32(i), u32(i + 1)
    s = (a & 0xFFFF) + (a >> 16) + (b & 0xFFFF) + (b >> 16) - 131070
    return s.to(torch.float32) * float(np.float32(std * 1.7320508075688772 / 65536.0))


class _Weight:
    """A matrix as the engine stores it; rows(x) = x @ W.T in float64, W widened a block of rows at a time."""

    def __init__(self, seed, kind, index, rows, cols, std, w, dev):
        self.q = torch.empty(rows, cols, dtype={"f32": torch.float32, "f16": torch.float16, "i8": torch.int8}[w], device=dev)
        self.s = torch.ones(rows, dtype=torch.float64, device=dev) if w == "i8" else None
        self.step = max(1, (1 << 25) // cols)
        for r in range(0, rows, self.step):
            n = min(self.step, rows - r)
            v = _normal(seed, kind, index, r * cols, n * cols, std, dev).view(n, cols)
            if w == "i8":
                sc = v.abs().amax(1) / 127.0
                v = torch.clamp(torch.round(v / sc[:, None]), -127, 127)
                self.s[r:r + n] = sc.double()
            self.q[r:r + n] = v.to(self.q.dtype)

    def pick(self, ids):
        e = self.q[ids].double()
        return e * self.s[ids][:, None] if self.s is not None else e

    def rows(self, x):
        out = torch.empty(x.shape[0], self.q.shape[0], dtype=torch.float64, device=x.device)
        for r in range(0, self.q.shape[0], self.step):
            out[:, r:r + self.step] = x @ self.q[r:r + self.step].double().t()
        return out * self.s if self.s is not None else out


def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _attend(q, k, v, scale, pos, bias=None, sink=None):
    """q [n][H][d] at positions pos, k / v [ctx][Hkv][d]: causal softmax attention, one kv head at a time."""
    n, H, d = q.shape
    g, ctx = H // k.shape[1], k.shape[0]
    out = torch.empty(n, H, v.shape[2], dtype=torch.float64, device=q.device)
    dist = pos[:, None] - torch.arange(ctx, device=q.device)[None, :]
    for h in range(H):
        s = q[:, h] @ k[:, h // g].t() * scale
        if bias is not None:
            s = s - bias[0][h] * torch.log1p(bias[1][h] * dist.clamp(min=0))
        s = s.masked_fill(dist < 0, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(n, 1)], 1)
        out[:, h] = torch.softmax(s, 1)[:, :ctx] @ v[:, h // g]
    return out


def _rope_tables(hd, theta, T, dev):
    """The model's fp32 sin / cos tables (part of its definition, as the weights are)."""
    f = (1.0 / (theta ** ((2 * np.arange(hd // 2)).astype(np.float32) / np.float32(hd)).astype(np.float64)).astype(np.float32)
         ).astype(np.float32)
    val = (f[None, :] * np.arange(T, dtype=np.float32)[:, None]).astype(np.float64)
    return [torch.tensor(t(val).astype(np.float32).astype(np.float64), device=dev) for t in (np.sin, np.cos)]


def _turn(x, sn, cs):
    a, b = x.chunk(2, -1)
    return torch.cat([a * cs[:, None] - b * sn[:, None], b * cs[:, None] + a * sn[:, None]], -1)


class _Llama:
    def __init__(self, case, seed, dev):
        c = self.c = _config(case)
        self.seed, self.dev, w = seed, dev, case["w"]
        self.kv = torch.float32 if case["kv"] == "f32" else torch.float16
        D, KV, I = c.hidden_size, c.kv_hidden_size, c.intermediate_size
        self.emb = _Weight(seed, 1, 0, c.vocab_size, D, 0.02, w, dev)
        self.norms = [(1.0 + _normal(seed, 2, i, 0, D, 0.1, dev)).double() for i in range(2 * c.num_hidden_layers + 1)]
        std = 1 / math.sqrt(D)
        self.layers = [{n: _Weight(seed, k, l, r, cc, sd, w, dev) for n, k, r, cc, sd in (
            ("q", 3, D, D, std), ("k", 4, KV, D, std), ("v", 5, KV, D, std), ("o", 6, D, D, std), ("up", 7, I, D, std),
            ("gate", 8, I, D, std), ("down", 9, D, I, 1 / math.sqrt(I)))} for l in range(c.num_hidden_layers)]
        self.sin, self.cos = _rope_tables(c.head_dim, c.rope_theta, c.max_length, dev)
        self.cache = {}

    def fill(self, l, b, upto):
        KV = self.c.kv_hidden_size
        return [_normal(self.seed + b, k, l, 0, upto * KV, 1.0, self.dev).view(upto, KV).to(self.kv).double() for k in (10, 11)]

    def rows(self, tokens, spans, context=0):
        """Rows of several sequences in order, spans = [(sequence, first position, rows)]; context: positions below each
        sequence's own that hold the synthetic fill. Returns the residual rows after the last norm."""
        c, hd = self.c, self.c.head_dim
        pos = torch.cat([torch.arange(p, p + n, device=self.dev) for _, p, n in spans])
        x = self.emb.pick(torch.as_tensor(np.asarray(tokens), device=self.dev).long())
        sn, cs = self.sin[pos], self.cos[pos]
        for l, w in enumerate(self.layers):
            h = _rms(x, self.norms[2 * l], c.rms_norm_eps)
            q = _turn(w["q"].rows(h).view(len(pos), -1, hd), sn, cs)
            k = _turn(w["k"].rows(h).view(len(pos), -1, hd), sn, cs).to(self.kv).double()
            v = w["v"].rows(h).view(len(pos), -1, hd).to(self.kv).double()
            o, r = [], 0
            for b, p, n in spans:
                kk, vv = k[r:r + n], v[r:r + n]
                if context and p:
                    fk, fv = self.fill(l, b, p)
                    kk, vv = torch.cat([fk.view(p, -1, hd), kk]), torch.cat([fv.view(p, -1, hd), vv])
                elif (l, b) in self.cache:
                    kk, vv = [torch.cat([a.double(), z]) for a, z in zip(self.cache[l, b], (kk, vv))]
                if not context:
                    self.cache[l, b] = kk.to(self.kv), vv.to(self.kv)
                o.append(_attend(q[r:r + n], kk, vv, hd ** -0.5, pos[r:r + n]))
                r += n
            x = x + w["o"].rows(torch.cat(o).view(len(pos), -1))
            h = _rms(x, self.norms[2 * l + 1], c.rms_norm_eps)
            x = x + w["down"].rows(torch.sigmoid(w["gate"].rows(h)) * w["up"].rows(h))
        return _rms(x, self.norms[-1], c.rms_norm_eps)


def _exact_llama(case, seed, dev):
    m = _Llama(case, seed, dev)
    if case["kind"] == "decode":
        toks, pos = _decode_inputs(case, seed)
        lg = m.emb.rows(m.rows(toks, [(b, p, 1) for b, p in enumerate(pos)], context=1)).cpu().numpy()
        return {"logits": lg[0] if case["batch"] == 1 else lg}
    if case["kind"] == "prompt":
        n = case["length"]
        ids = _rng(seed).integers(0, m.c.vocab_size, n).astype(np.int32)
        return {"logits": m.emb.rows(m.rows(ids, [(0, 0, n)])[-1:]).cpu().numpy()[0]}
    prompts, B, N = _prompts(case, seed), case["batch"], case["length"]
    toks = np.zeros((B, N), np.int32)
    for b, p in enumerate(prompts):
        toks[b, :min(N, len(p))] = p[:N]
    n0 = min(min(len(p) for p in prompts), N)
    x = m.rows(toks[:, :n0].reshape(-1), [(b, 0, n0) for b in range(B)])[n0 - 1::n0]
    for t in range(n0, N):
        best = m.emb.rows(x).argmax(1).cpu().numpy()
        for b, p in enumerate(prompts):
            if t >= len(p):
                toks[b, t] = best[b]
        x = m.rows(toks[:, t], [(b, t, 1) for b in range(B)])
    lg = m.emb.rows(x).cpu().numpy()
    return {"tokens": toks[0] if B == 1 else toks, "logits": lg[0] if B == 1 else lg}


def _exact_operators(case, seed, dev):
    c, t, pos = preset(case["model"]), _op_tensors(case, seed, dev), case["pos"]
    sin, cos = _rope_tables(c.head_dim, c.rope_theta, c.max_length, dev)
    at, hd = torch.tensor([pos], device=dev), c.head_dim
    tok = int(_rng(seed).integers(0, c.vocab_size))
    x, ks, vs = t["emb"][tok].double()[None], [], []
    for l, w in enumerate(t["layers"]):
        w = {n: a.double() for n, a in w.items()}
        h = _rms(x, w["n1"], c.rms_norm_eps)
        q = _turn((h @ w["q"].t()).view(1, -1, hd), sin[at], cos[at])
        k = _turn((h @ w["k"].t()).view(1, -1, hd), sin[at], cos[at])
        v = (h @ w["v"].t()).view(1, -1, hd)
        kk = torch.cat([t["kc"][l, :pos].double().view(pos, -1, hd), k])
        vv = torch.cat([t["vc"][l, :pos].double().view(pos, -1, hd), v])
        x = x + _attend(q, kk, vv, hd ** -0.5, at).view(1, -1) @ w["o"].t()
        h = _rms(x, w["n2"], c.rms_norm_eps)
        x = x + (torch.sigmoid(h @ w["gate"].t()) * (h @ w["up"].t())) @ w["down"].t()
        ks.append(k.flatten())
        vs.append(v.flatten())
    lg = (_rms(x, t["final"].double(), c.rms_norm_eps) @ t["emb"].double().t())[0]
    return {"x": x[0], "logits": lg, "k": torch.stack(ks), "v": torch.stack(vs), "token": lg.argmax()[None].int()}


def _stack_tensors(sp: StackSpec, seed, dev):
    """The engine's synthetic block-stack weights by name: matrices in fp16, vectors and convolutions fp32."""
    D, shapes = sp.width, {}
    for i, b in enumerate(sp.blocks):
        kv = b.kv_heads if b.mixer == "attention" else b.heads
        leaf = {"norm1": (1, 1), "norm2": (1, 1), "canon1": (D, sp.taps), "canon2": (D, sp.taps),
                "mix.q": (b.heads * b.dim, D), "mix.k": (kv * b.dim, D), "mix.v": (kv * b.vdim, D),
                "mix.o": (D, b.heads * b.vdim), "mlp.gate": (b.ff, D), "mlp.up": (b.ff, D), "mlp.down": (D, b.ff)}
        leaf.update({n: (1, b.heads) for n in ("mix.r1", "mix.r2", "mix.sink")} if b.mixer == "attention" else
                    {"mix.g": (b.heads * b.vdim, D)})
        shapes.update({f"l{i}.{n}": s for n, s in leaf.items()})
    shapes.update(embed=(sp.vocab_size, D), head=(sp.vocab_size, D))
    shapes["final.norm"] = (1, 1)
    f32, M64, out = np.float32, (1 << 64) - 1, {}
    for i, (name, (r, k)) in enumerate(sorted(shapes.items())):
        s = ((seed * 0x9E3779B9) ^ ((i + 1) * 0x85EBCA6B)) & _M32
        leaf = name.split(".", 1)[-1]
        conv, gain = leaf in ("canon1", "canon2"), "norm" in leaf
        if r > 1 and not conv:
            amp = 1.0 if name == "embed" else float(f32(1.5) / np.sqrt(f32(k)))
            w = torch.empty(r * k, dtype=torch.float16, device=dev)
            for e in range(0, r * k, 1 << 25):
                n = torch.arange(e, min(r * k, e + (1 << 25)), dtype=torch.int64, device=dev)
                h = _hash32(((n & _M32) * 2654435761 & _M32) ^ ((n >> 32) * 0x9E3779B9 & _M32) ^ s)
                w[e:e + n.numel()] = (((h >> 8).float() / 8388608.0 - 1.0) * amp).half()
            out[name] = w.view(r, k)
            continue
        amp = f32(0.1 if gain else 0.2 if leaf == "mix.r2" else 0.3 if conv else 1.0)
        off = f32(1.0 if gain else 0.25 if leaf == "mix.r2" else 0.0 if conv else 1.0)
        x, v = (0x9E3779B97F4A7C15 * (s + 1)) & M64, []
        for _ in range(r * k):
            x ^= x >> 12
            x ^= (x << 25) & M64
            x ^= x >> 27
            v.append(((x * 0x2545F4914F6CDD1D & M64) >> 40) / 8388608.0 - 1.0)
        out[name] = torch.tensor((off + amp * np.array(v, f32)).astype(np.float64), device=dev).view(r, k)
    return out


def _exact_stack(case, seed, dev):
    sp = _stack_spec(case)
    t = _stack_tensors(sp, seed, dev)
    prompts, steps = _stack_inputs(case, seed)
    seqs = [np.concatenate([p, [s[i] for s in steps]]).astype(np.int64) for i, p in enumerate(prompts)]
    cut = np.cumsum([0] + [len(s) for s in seqs])
    at = [torch.arange(len(s), device=dev) for s in seqs]

    def conv(h, w):
        y = torch.zeros_like(h)
        for a, b in zip(cut, cut[1:]):
            for j in range(sp.taps):  # tap j multiplies the row taps - 1 - j back
                d = sp.taps - 1 - j
                y[a + d:b] += h[a:b - d] * w[:, j] if d < b - a else 0.0
        return h + y
    x = t["embed"][torch.tensor(np.concatenate(seqs), device=dev)].double() * sp.emb_scale
    for i, b in enumerate(sp.blocks):
        w = {n[len(f"l{i}."):]: v.double() for n, v in t.items() if n.startswith(f"l{i}.")}
        h = conv(_rms(x, w["norm1"][0, 0], sp.eps), w["canon1"])
        n, att = len(x), b.mixer == "attention"
        kvh = b.kv_heads if att else b.heads
        q, k = (h @ w["mix.q"].t()).view(n, b.heads, b.dim), (h @ w["mix.k"].t()).view(n, kvh, b.dim)
        v, o = (h @ w["mix.v"].t()).view(n, kvh, b.vdim), []
        for s, (lo, hi) in enumerate(zip(cut, cut[1:])):
            p = at[s]
            if att:
                o.append(_attend(q[lo:hi], k[lo:hi].half().double(), v[lo:hi].half().double(), b.scale, p,
                                 (w["mix.r1"][0], w["mix.r2"][0]), w["mix.sink"][0]))
                continue
            ang = p[:, None] * float(b.rot_base) ** (-2.0 * torch.arange(b.rot_dims // 2, device=dev).double() / b.rot_dims)
            qq, kk = _turn(q[lo:hi], ang.sin(), ang.cos()), _turn(k[lo:hi], ang.sin(), ang.cos()) * b.dim ** -0.5
            oo = torch.empty(hi - lo, b.heads, b.vdim, dtype=torch.float64, device=dev)
            for hh in range(b.heads):
                dist = (p[:, None] - p[None, :]).double()
                dec = float(np.float32(b.decay[hh])) ** dist.clamp(min=0) * (dist >= 0)
                oo[:, hh] = ((qq[:, hh] @ kk[:, hh].t()) * dec) @ v[lo:hi, hh]
            o.append(oo)
        o = torch.cat(o)
        if not att:
            g = (h @ w["mix.g"].t()).view(n, b.heads, b.vdim)
            o = _rms(o, 1.0, sp.eps) * g * torch.sigmoid(g)
        y = o.reshape(n, -1) @ w["mix.o"].t()
        h = conv(_rms(x, w["norm2"][0, 0], sp.eps), w["canon2"])
        g, u = (h @ w["mlp.gate"].t()).clamp(max=b.ff_limit), (h @ w["mlp.up"].t()).clamp(-b.ff_limit, b.ff_limit)
        x = x + sp.residual_mult * (y + (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w["mlp.down"].t())
    want = [torch.tensor([a + len(p) - 1 + j for a, p in zip(cut, prompts)], device=dev) for j in range(1 + len(steps))]
    head = t["head"].double()
    return {"logits": [(_rms(x[r], t["final.norm"][0, 0], sp.eps) @ head.t()).cpu().numpy() for r in want]}


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    with torch.no_grad():
        if case["kind"] == "operators":
            return _exact_operators(case, seed, dev)
        return (_exact_stack if case["kind"] == "stack" else _exact_llama)(case, seed, dev)
