"""The work that programs built on this library have it do, as cases that can be timed and checked.

A case is one pass through the public entry points (the Python binding of the C ABI): a quantized linear layer, an
attention layer over the paged cache or over contiguous tensors, the language-model head with its sampler's selection,
and a whole model call.  listed() holds fixed sizes, draw() others from the ranges that they stand for.
"""
import math
import os
import random
import sys

import numpy as np
import torch

_PACKAGE = os.path.join(os.getcwd(), "cuda-llm-inference-engine_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import ie_amd as ie  # noqa: E402

DEV = "cuda"
EPILOGUES = {"plain": ie.EPI_PLAIN, "bias": ie.EPI_BIAS, "gelu": ie.EPI_BIAS_GELU, "residual": ie.EPI_BIAS_RESIDUAL}


def listed():
    return [
        # the QKV projection of one decoded token at GPT-2 Small's widths: launches and latency
        _linear("linear-token", M=1, K=768, N=2304, epilogue="bias"),
        # an output projection with the residual stream for a decode batch, at a width that is not GPT-2 Small's
        _linear("linear-batch16-4096", M=16, K=4096, N=4096, epilogue="residual"),
        # a wide layer for a small decode batch: 235 MB of weights streamed once
        _linear("linear-batch4-wide", M=4, K=8192, N=28672, epilogue="plain"),
        # residual add, LayerNorm, quantizer and the FFN-up layer with GELU for a prompt's rows
        _linear("linear-prompt512-ffn", M=512, K=768, N=3072, epilogue="gelu", norm=True),
        # a prompt's rows at widths that no tile divides
        _linear("linear-prompt-ragged", M=300, K=1600, N=4801, epilogue="bias"),
        # the largest product the benchmark names
        _linear("linear-8192-cube", M=8192, K=8192, N=8192, epilogue="plain"),
        # a decode step's attention for a batch of GPT-2-like sequences, full fp32 cache
        _decode("decode-attn-mha-1k", B=8, H_kv=12, G=1, d=64, ctx=1024, bf16=False, ragged=False),
        # grouped-query decode attention over long ragged contexts in a bf16 cache
        _decode("decode-attn-gqa-8k", B=32, H_kv=8, G=4, d=128, ctx=8192, bf16=True, ragged=True),
        # a batch of prompts: their K/V rows into the paged cache, then causal attention over it
        _prompt("prompt-attn-512", B=4, P=512, start=0, H_kv=12, G=1, d=64, bf16=False),
        # attention over contiguous tensors at a long sequence length
        _flash("flash-attn-2k", B=1, H=16, N=2048, d=128, causal=True),
        # fp32 language-model head of a decode batch and the sampler's top-k of each row
        _head("lm-head-topk", rows=8, d=768, V=50257, k=40),
        # a whole model: GPT-2 Small reads a batch of prompts and decodes eight tokens each
        _engine("engine-gpt2-small", B=4, P=128, steps=8, layers=12, d=768, V=50257, bf16=False, head8=False),
    ]


def draw(rng):
    kind = rng.choice(("token", "token", "rows", "rows", "decode", "decode", "prompt", "prompt", "flash", "head", "engine"))
    if kind == "token":  # decode-sized linear layers
        K = _width(rng, 256, 8192)
        return _linear(None, M=rng.randint(1, 16), K=K, N=_log(rng, 256, 50257), epilogue=rng.choice(sorted(EPILOGUES)),
                       norm=rng.random() < 0.25)
    if kind == "rows":  # prompt-sized ones
        while True:
            M, K, N = _log(rng, 17, 4096), _width(rng, 256, 8192), _log(rng, 256, 16384)
            if M * K * N <= (1 << 36 if K % 16 == 0 else 1 << 31):
                return _linear(None, M=M, K=K, N=N, epilogue=rng.choice(sorted(EPILOGUES)), norm=rng.random() < 0.25)
    if kind == "decode":
        while True:
            c = _decode(None, B=_log(rng, 1, 64), H_kv=rng.choice((4, 8, 12, 16)), G=rng.choice((1, 1, 2, 4, 8)),
                        d=rng.choice((64, 128)), ctx=_log(rng, 16, 8192), bf16=rng.random() < 0.5,
                        ragged=rng.random() < 0.5)
            if _decode_kv_bytes(c) <= 800e6:
                return c
    if kind == "prompt":
        while True:
            c = _prompt(None, B=_log(rng, 1, 8), P=_log(rng, 17, 1024), start=rng.choice((0, 0, rng.randint(1, 512))),
                        H_kv=rng.choice((4, 8, 12, 16)), G=rng.choice((1, 1, 2, 4)), d=rng.choice((64, 128)),
                        bf16=rng.random() < 0.5)
            if work(c)["flops"] <= 2e10:
                return c
    if kind == "flash":
        while True:
            c = _flash(None, B=_log(rng, 1, 8), H=rng.choice((4, 8, 12, 16, 32)), N=_log(rng, 33, 4096),
                       d=rng.choice((64, 128)), causal=rng.random() < 0.75)
            if work(c)["flops"] <= 2e10:
                return c
    if kind == "head":
        return _head(None, rows=rng.randint(1, 16), d=_width(rng, 256, 2048), V=_log(rng, 1000, 50257),
                     k=_log(rng, 1, 100))
    return _engine(None, B=_log(rng, 1, 16), P=_log(rng, 8, 256), steps=rng.randint(1, 8), layers=rng.randint(2, 12),
                   d=rng.choice((512, 768, 768, 1024)), V=_log(rng, 5000, 50257), bf16=rng.random() < 0.5,
                   head8=rng.random() < 0.25)


def prepare(case, seed):
    return _OPS[case["op"]].prepare(case, seed)


def run(state):
    return state["run"](state)


def work(case):
    return _OPS[case["op"]].work(case)


def tolerance(case):
    return _OPS[case["op"]].tolerance(case)


def exact(case, seed):
    return _OPS[case["op"]].exact(case, seed)


# ------------------------------------------------------------------ sizes and inputs
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly a multiple of 128, at times only of 16, at times only of 4 (what the quantizer asks for)."""
    step = rng.choice((128, 128, 128, 128, 128, 16, 16, 4))
    return max(step, _log(rng, lo, hi) // step * step)


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(shape, device=DEV, generator=g)


def _quantize_rows(x):
    """Symmetric int8 per row in fp32, the layers' own definition: scale = max|x| / 127, q = rint(x * (1 / scale))."""
    m = x.abs().amax(dim=1)
    one = torch.ones_like(m)  # a divisor that is a plain number would become a multiplication
    scale = torch.where(m > 0, m / (127.0 * one), one)
    return (x * (one / scale)[:, None]).round_().clamp_(-128, 127).to(torch.int8), scale


def _activations(g, rows, cols):
    """Rows as a residual stream has them: near-normal, their sizes spread, a few wide channels."""
    x = _normal(g, rows, cols) * torch.exp(0.3 * _normal(g, rows, 1))
    wide = torch.where(torch.rand(cols, device=DEV, generator=g) < 0.01, 6.0, 1.0)
    return x * wide


# ------------------------------------------------------------------ a quantized linear layer
def _linear(name, M, K, N, epilogue, norm=False):
    c = dict(op="linear", M=M, K=K, N=N, epilogue=epilogue, norm=norm)
    return dict(c, name=name) if name else c


class _Linear:
    @staticmethod
    def inputs(case, seed):
        g, M, K, N = _generator(seed), case["M"], case["K"], case["N"]
        v = {"x": _activations(g, M, K)}
        v["w"], v["w_scale"] = _quantize_rows(0.02 * _normal(g, N, K))
        v["bias"] = 0.02 * _normal(g, N)
        if case["epilogue"] == "residual":
            v["residual"] = _activations(g, M, N)
        if case["norm"]:
            v["skip"] = _activations(g, M, K)
            v["gamma"] = 1.0 + 0.1 * _normal(g, K)
            v["beta"] = 0.1 * _normal(g, K)
        return v

    @staticmethod
    def prepare(case, seed):
        M, K, N = case["M"], case["K"], case["N"]
        s = _Linear.inputs(case, seed)
        s["w"] = s["w"].view(torch.int32)  # four values a word, as the weight files hold them
        s["packed"] = torch.empty(M, K // 4, dtype=torch.int32, device=DEV)
        s["scales"] = torch.empty(M, device=DEV)
        s["out"] = torch.empty(M, N, device=DEV)
        if case["norm"]:
            s["hidden"], s["normed"] = torch.empty(M, K, device=DEV), torch.empty(M, K, device=DEV)
        s["epilogue"] = EPILOGUES[case["epilogue"]]
        if case["epilogue"] == "plain":
            s["bias"] = None
        s["run"] = _Linear.run_norm if case["norm"] else _Linear.run
        return s

    @staticmethod
    def run(s):
        ie.quantize(s["x"], s["packed"], s["scales"])
        return ie.int8_gemm(s["packed"], s["w"], s["scales"], s["w_scale"], s["epilogue"], s["bias"], s.get("residual"),
                            s["out"])

    @staticmethod
    def run_norm(s):
        ie.layernorm_residual(s["x"], s["skip"], s["gamma"], s["beta"], s["normed"], s["hidden"])
        ie.quantize(s["normed"], s["packed"], s["scales"])
        ie.int8_gemm(s["packed"], s["w"], s["scales"], s["w_scale"], s["epilogue"], s["bias"], s.get("residual"), s["out"])
        return s["out"], s["hidden"]

    @staticmethod
    def work(case):
        M, K, N = case["M"], case["K"], case["N"]
        b = N * K + 4 * M * K + 4 * N + 4 * M * N
        b += 4 * N if case["epilogue"] != "plain" else 0
        b += 4 * M * N if case["epilogue"] == "residual" else 0
        b += 8 * M * K + 8 * K if case["norm"] else 0
        return {"bytes": b, "flops": 2 * M * N * K}

    @staticmethod
    def tolerance(case):
        # int32 sums are exact, so only the fp32 dequantization (and tanh) rounds: 6e-8 and 5e-7 against 64 bits; a
        # scale or a LayerNorm one bit apart moves some values to the next int8 step: 4e-5 and 5e-3
        return {"rel": 2e-4, "max": 2e-2} if case["norm"] else {"rel": 2.5e-7, "max": 2e-6}

    @staticmethod
    def exact(case, seed):
        v = _Linear.inputs(case, seed)
        x, hidden = v["x"], None
        if case["norm"]:
            h = hidden = x.double() + v["skip"].double()
            mean = h.mean(dim=1, keepdim=True)
            var = (h * h).mean(dim=1, keepdim=True) - mean * mean
            x = ((h - mean) * torch.rsqrt(var + 1e-5) * v["gamma"].double() + v["beta"].double()).float()
        q, scale = _quantize_rows(x)
        out = torch.empty(case["M"], case["N"], dtype=torch.float64, device=DEV)
        qd = q.double()
        for n in range(0, case["N"], 8192):
            out[:, n:n + 8192] = qd @ v["w"][n:n + 8192].double().t().contiguous()
        out *= scale.double()[:, None]
        out *= v["w_scale"].double()[None, :]
        if case["epilogue"] != "plain":
            out += v["bias"].double()
        if case["epilogue"] == "gelu":
            out = 0.5 * out * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (out + 0.044715 * out**3)))
        if case["epilogue"] == "residual":
            out += v["residual"].double()
        return (out, hidden) if case["norm"] else out


# ------------------------------------------------------------------ the paged cache
def _paged(g, lens, H_kv, d, bf16, block):
    """Caches whose sequences' blocks lie scattered, and the block table."""
    nb = [(n + block - 1) // block for n in lens]
    total = sum(nb)
    kind = torch.bfloat16 if bf16 else torch.float32
    k = (_normal(g, total, block, H_kv, d) + 0.5 * _normal(g, H_kv, d)).to(kind)
    v = _normal(g, total, block, H_kv, d).to(kind)
    order = torch.randperm(total, device=DEV, generator=g).to(torch.int32)
    table = torch.zeros(len(lens), max(nb), dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(nb):
        table[b, :n] = order[at:at + n]
        at += n
    return k, v, table


def _gathered(cache, table, b, n, block):
    """The first n tokens of sequence b as [H_kv, n, d] in 64 bits."""
    rows = cache[table[b, :(n + block - 1) // block].long()].reshape(-1, *cache.shape[2:])[:n]
    return rows.double().permute(1, 0, 2).contiguous()


def _attention(q, k, v, mask=None):
    """softmax(q k^T / sqrt(d)) v in 64 bits: q [H, t, d], k and v [H, n, d]."""
    s = (q @ k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
    if mask is not None:
        s = s.masked_fill(~mask, -math.inf)
    return torch.softmax(s, dim=-1) @ v


# ------------------------------------------------------------------ decode attention
def _decode(name, B, H_kv, G, d, ctx, bf16, ragged):
    c = dict(op="decode", B=B, H_kv=H_kv, G=G, d=d, ctx=ctx, bf16=bf16, ragged=ragged)
    return dict(c, name=name) if name else c


def _decode_lens(case):
    """Context lengths: all ctx, or spread over its upper half."""
    if not case["ragged"]:
        return [case["ctx"]] * case["B"]
    r = random.Random(case["ctx"])
    return [r.randint((case["ctx"] + 1) // 2, case["ctx"]) for _ in range(case["B"])]


def _decode_kv_bytes(case):
    return sum(_decode_lens(case)) * case["H_kv"] * case["d"] * 2 * (2 if case["bf16"] else 4)


class _Decode:
    BLOCK = 16

    @staticmethod
    def inputs(case, seed):
        g, lens = _generator(seed), _decode_lens(case)
        k, v, table = _paged(g, lens, case["H_kv"], case["d"], case["bf16"], _Decode.BLOCK)
        return _normal(g, case["B"], case["H_kv"] * case["G"], case["d"]), k, v, table, lens

    @staticmethod
    def prepare(case, seed):
        q, k, v, table, lens = _Decode.inputs(case, seed)
        B, H, d = q.shape
        top = max(lens)
        need = ie.workspace_bytes(B, H, d, ie.num_splits(top, _Decode.BLOCK))
        return {"run": _Decode.run, "q": q, "k": k, "v": v, "table": table, "top": top, "H_kv": case["H_kv"],
                "lens": torch.tensor(lens, dtype=torch.int32, device=DEV), "out": torch.empty_like(q),
                "kind": ie.KV_BF16 if case["bf16"] else ie.KV_F32,
                "workspace": torch.empty(max(need // 4, 1), device=DEV)}

    @staticmethod
    def run(s):
        return ie.decode_attn(s["q"], s["k"], s["v"], s["table"], s["lens"], s["top"], _Decode.BLOCK, s["H_kv"],
                              kv_dtype=s["kind"], out=s["out"], workspace=s["workspace"])

    @staticmethod
    def work(case):
        n, H = sum(_decode_lens(case)), case["H_kv"] * case["G"]
        return {"bytes": _decode_kv_bytes(case) + 8 * case["B"] * H * case["d"] + n // 4 + 4 * case["B"],
                "flops": 4 * n * H * case["d"]}

    @staticmethod
    def tolerance(case):
        return {"rel": 1.5e-6, "max": 4e-5}  # fp32 sums: up to 3.7e-7 and 1e-5 against 64 bits

    @staticmethod
    def exact(case, seed):
        q, k, v, table, lens = _Decode.inputs(case, seed)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b, n in enumerate(lens):
            qb = q[b].double().reshape(case["H_kv"], case["G"], case["d"])
            out[b] = _attention(qb, _gathered(k, table, b, n, 16), _gathered(v, table, b, n, 16)).reshape(q.shape[1:])
        return out


# ------------------------------------------------------------------ prompt attention over the paged cache
def _prompt(name, B, P, start, H_kv, G, d, bf16):
    c = dict(op="prompt", B=B, P=P, start=start, H_kv=H_kv, G=G, d=d, bf16=bf16)
    return dict(c, name=name) if name else c


class _Prompt:
    BLOCK = 16

    @staticmethod
    def inputs(case, seed):
        g, B, P, d = _generator(seed), case["B"], case["P"], case["d"]
        k, v, table = _paged(g, [case["start"] + P] * B, case["H_kv"], d, case["bf16"], _Prompt.BLOCK)
        q = _normal(g, B, P, case["H_kv"] * case["G"], d)
        return q, k, v, table, _normal(g, B, P, case["H_kv"], d), _normal(g, B, P, case["H_kv"], d)

    @staticmethod
    def prepare(case, seed):
        q, k, v, table, new_k, new_v = _Prompt.inputs(case, seed)
        return {"run": _Prompt.run, "q": q, "k": k, "v": v, "table": table, "new": list(zip(new_k, new_v, table)),
                "start": case["start"], "H_kv": case["H_kv"], "out": torch.empty_like(q),
                "kind": ie.KV_BF16 if case["bf16"] else ie.KV_F32}

    @staticmethod
    def run(s):
        for new_k, new_v, row in s["new"]:
            ie.kv_cache_write(new_k, new_v, s["k"], s["v"], row, s["start"], _Prompt.BLOCK, s["kind"])
        out = ie.prefill_attn(s["q"], s["k"], s["v"], s["table"], s["start"], _Prompt.BLOCK, s["H_kv"],
                              kv_dtype=s["kind"], out=s["out"])
        return out, s["k"], s["v"]

    @staticmethod
    def work(case):
        B, P, start, d, size = case["B"], case["P"], case["start"], case["d"], 2 if case["bf16"] else 4
        rows, H = B * P, case["H_kv"] * case["G"]
        return {"bytes": 8 * rows * H * d + 8 * rows * case["H_kv"] * d + 2 * size * B * (start + P) * case["H_kv"] * d,
                "flops": 4 * B * H * d * (P * start + P * (P + 1) // 2)}

    @staticmethod
    def tolerance(case):
        return {"rel": 1.5e-6, "max": 4e-5}  # fp32 sums: up to 3.7e-7 and 1e-5 against 64 bits

    @staticmethod
    def exact(case, seed):
        q, k, v, table, new_k, new_v = _Prompt.inputs(case, seed)
        B, P, start, G = case["B"], case["P"], case["start"], case["G"]
        pos = torch.arange(start, start + P, device=DEV)
        mask = torch.arange(start + P, device=DEV)[None, :] <= pos[:, None]
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b in range(B):
            slot = table[b, (pos // _Prompt.BLOCK)].long()
            k[slot, pos % _Prompt.BLOCK] = new_k[b].to(k.dtype)
            v[slot, pos % _Prompt.BLOCK] = new_v[b].to(v.dtype)
            kb, vb = (_gathered(c, table, b, start + P, _Prompt.BLOCK) for c in (k, v))
            for h in range(case["H_kv"]):
                qh = q[b, :, h * G:(h + 1) * G].double().permute(1, 0, 2).contiguous()
                o = _attention(qh, kb[h].expand(G, -1, -1).contiguous(), vb[h].expand(G, -1, -1).contiguous(), mask)
                out[b, :, h * G:(h + 1) * G] = o.permute(1, 0, 2)
        return out, k.double(), v.double()


# ------------------------------------------------------------------ attention over contiguous tensors
def _flash(name, B, H, N, d, causal):
    c = dict(op="flash", B=B, H=H, N=N, d=d, causal=causal)
    return dict(c, name=name) if name else c


class _Flash:
    @staticmethod
    def inputs(case, seed):
        g, shape = _generator(seed), (case["B"], case["H"], case["N"], case["d"])
        return _normal(g, *shape), _normal(g, *shape) + 0.5 * _normal(g, 1, case["H"], 1, case["d"]), _normal(g, *shape)

    @staticmethod
    def prepare(case, seed):
        q, k, v = _Flash.inputs(case, seed)
        return {"run": _Flash.run, "q": q, "k": k, "v": v, "causal": case["causal"], "out": torch.empty_like(q)}

    @staticmethod
    def run(s):
        return ie.flash_attn(s["q"], s["k"], s["v"], s["causal"], s["out"])

    @staticmethod
    def work(case):
        B, H, N, d = case["B"], case["H"], case["N"], case["d"]
        return {"bytes": 16 * B * H * N * d, "flops": 4 * B * H * d * (N * (N + 1) // 2 if case["causal"] else N * N)}

    @staticmethod
    def tolerance(case):
        return {"rel": 1.5e-6, "max": 4e-5}  # fp32 sums: up to 3.7e-7 and 1e-5 against 64 bits

    @staticmethod
    def exact(case, seed):
        q, k, v = _Flash.inputs(case, seed)
        N = case["N"]
        mask = torch.ones(N, N, dtype=torch.bool, device=DEV).tril() if case["causal"] else None
        return torch.stack([torch.cat([_attention(q[b, h:h + 1].double(), k[b, h:h + 1].double(), v[b, h:h + 1].double(),
                                                  mask) for h in range(case["H"])]) for b in range(case["B"])])


# ------------------------------------------------------------------ language-model head and top-k
def _head(name, rows, d, V, k):
    c = dict(op="head", rows=rows, d=d, V=V, k=k)
    return dict(c, name=name) if name else c


class _Head:
    @staticmethod
    def inputs(case, seed):
        g = _generator(seed)
        return _normal(g, case["rows"], case["d"]), 0.02 * _normal(g, case["V"], case["d"])

    @staticmethod
    def prepare(case, seed):
        h, wte = _Head.inputs(case, seed)
        return {"run": _Head.run, "h": h, "wte": wte, "k": case["k"],
                "logits": torch.empty(case["rows"], case["V"], device=DEV)}

    @staticmethod
    def run(s):
        ie.vocab_proj(s["h"], s["wte"], s["logits"])
        values, indices = ie.topk(s["logits"], s["k"])
        return s["logits"], values, indices

    @staticmethod
    def work(case):
        rows, d, V = case["rows"], case["d"], case["V"]
        return {"bytes": 4 * V * d + 4 * rows * (d + V) + 8 * rows * case["k"], "flops": 2 * rows * V * d}

    @staticmethod
    def tolerance(case):
        # fp32 sums: 1.7e-7 and 1e-6 against 64 bits; two logits a rounding apart may change places
        return {"rel": 7e-7, "max": 4e-6, "differ": 0.01}

    @staticmethod
    def exact(case, seed):
        h, wte = _Head.inputs(case, seed)
        logits = h.double() @ wte.double().t().contiguous()
        return logits, torch.topk(logits, case["k"], dim=1).values, None


# ------------------------------------------------------------------ a whole model
def _engine(name, B, P, steps, layers, d, V, bf16, head8):
    c = dict(op="engine", B=B, P=P, steps=steps, layers=layers, d=d, V=V, bf16=bf16, head8=head8)
    return dict(c, name=name) if name else c


class _Engine:
    @staticmethod
    def prepare(case, seed):
        B, P, steps = case["B"], case["P"], case["steps"]
        e = ie.Engine(seed=seed, max_batch=B, kv_dtype=ie.KV_BF16 if case["bf16"] else ie.KV_F32,
                      int8_lm_head=case["head8"], n_layers=case["layers"], n_heads=case["d"] // 64, d_model=case["d"],
                      d_ff=4 * case["d"], vocab_size=case["V"], max_seq_len=512)
        ids = np.random.default_rng(seed).integers(0, case["V"], (B, P + steps), dtype=np.int32)
        return {"run": _Engine.run, "engine": e, "prompt": np.ascontiguousarray(ids[:, :P]),
                "next": [np.ascontiguousarray(ids[:, P + i]) for i in range(steps)]}

    @staticmethod
    def run(s):
        s["engine"].reset()
        return [s["engine"].prefill(s["prompt"])] + [s["engine"].step(t) for t in s["next"]]

    @staticmethod
    def work(case):
        B, P, steps, d = case["B"], case["P"], case["steps"], case["d"]
        layers = case["layers"] * 12 * d * d
        head = case["V"] * d
        kv = case["layers"] * 2 * d * (2 if case["bf16"] else 4)  # bytes a token
        reads = sum(P + i for i in range(1, steps + 1)) * kv * B
        return {"bytes": (1 + steps) * (layers + head * (1 if case["head8"] else 4) + 4 * B * case["V"]) + reads
                + (P + steps) * B * kv,
                "flops": 2 * B * ((P + steps) * layers + (1 + steps) * head) + 2 * case["layers"] * d * B * P * (P + 1)}

    @staticmethod
    def tolerance(case):
        # a last-bit difference in an attention output can move an activation to the next int8 step, and every later
        # layer then sees another input: the prompt fed token by token, whose attention adds in another order, gives
        # logits 2e-2 and 1e-1 away
        return {"rel": 8e-2, "max": 4e-1}

    @staticmethod
    def exact(case, seed):
        return None  # the weights are the engine's own random ones


_OPS = {"linear": _Linear, "decode": _Decode, "prompt": _Prompt, "flash": _Flash, "head": _Head, "engine": _Engine}
