"""What the framework's users have it do, as cases that can be timed and compared.

    qgemv        one quantised matrix times one activation row (fk_qgemv)
    projections  the fused calls of one layer at batch 1: RMSNorm + q / k / v, RMSNorm + gate / up + SwiGLU,
                 down projection + residual
    attention    rotary position + cache append + attention of one token over a long cache (bf16 or quantised)
    decode       greedy decode of a dense model: a chunk of tokens from the captured graph
    prompt       prompt processing of a dense model, several rows a pass
    moe_decode   greedy decode of the mixture-of-experts model
    moe_rows     several active rows of the mixture-of-experts model in one pass

A case is a dict of plain values; listed() gives the fixed ones, draw() more of the same ranges.  Models are random-init.
The embedding is about as large as what all layers together add to it and, where the model has a head of its own, the head
is the embedding with its rows in another order: the next token then stands well clear of the others, as it does in a
trained model, so that the greedy token does not hang on the last bit of a logit.  Caches are filled with N(0, 1) values.
"""
import math

import numpy as np
import torch

import fusekit_amd.native as fk
from fusekit_amd.decoder import DENSE_4B, QWEN25_05B_LIKE, DecoderConfig, DecoderRuntime, DecoderWeights, quantize_on_device
from fusekit_amd.moe_decoder import MoeConfig, MoeRuntime, MoeWeights

# dense shapes: the two that the package names and two generic ones, a small and a wide one
MODELS = {
    "05b": dict(QWEN25_05B_LIKE),
    "4b": dict(DENSE_4B),
    "small": dict(n_layers=12, hidden=1024, n_heads=16, n_kv=8, head_dim=64, inter=3072, vocab=32000),
    "wide": dict(n_layers=16, hidden=4096, n_heads=32, n_kv=8, head_dim=128, inter=14336, vocab=65536),
}
GROUP = 64
EMBED_STD = 8.0


def listed():
    return [
        # a single int4 matrix-vector product of the 0.5B class: launch latency and the host's call are all of it
        {"name": "qgemv-4864x896-q4", "kind": "qgemv", "n": 4864, "k": 896, "bits": 4},
        # the fused calls of one 0.5B-class layer, made one by one by a program that keeps its own loop
        {"name": "projections-05b-q4", "kind": "projections", "hidden": 896, "inter": 4864, "n_q": 896, "n_kv": 128, "bits": 4},
        # one layer's attention deep in a long conversation
        {"name": "attention-32768", "kind": "attention", "length": 32768, "n_heads": 32, "n_kv": 8, "head_dim": 128, "kv_bits": 0},
        # a small assistant: two KV heads, projection biases, one launch per task
        {"name": "decode-05b-q4", "kind": "decode", "model": "05b", "layers": 24, "bits": 4, "kv_bits": 0, "context": 480, "tokens": 64},
        # the headline: 4B class, int4, around context 512
        {"name": "decode-4b-q4", "kind": "decode", "model": "4b", "layers": 36, "bits": 4, "kv_bits": 0, "context": 480, "tokens": 64},
        # the same model unquantised
        {"name": "decode-4b-bf16", "kind": "decode", "model": "4b", "layers": 36, "bits": 16, "kv_bits": 0, "context": 480, "tokens": 32},
        # a long conversation that keeps its cache in 8 bits
        {"name": "decode-4b-q4-kv8-long", "kind": "decode", "model": "4b", "layers": 36, "bits": 4, "kv_bits": 8, "context": 12000,
         "tokens": 16},
        # mixture of experts, one user
        {"name": "decode-moe-q4", "kind": "moe_decode", "layers": 27, "context": 480, "tokens": 64},
        # a chat turn of a few words (37 rows: no tile's multiple)
        {"name": "prompt-05b-q4-37", "kind": "prompt", "model": "05b", "layers": 24, "bits": 4, "kv_bits": 0, "start": 0, "rows": 37},
        # an ordinary prompt
        {"name": "prompt-4b-q4-512", "kind": "prompt", "model": "4b", "layers": 36, "bits": 4, "kv_bits": 0, "start": 0, "rows": 512},
        # a document
        {"name": "prompt-4b-q4-4096", "kind": "prompt", "model": "4b", "layers": 36, "bits": 4, "kv_bits": 0, "start": 0, "rows": 4096},
        # eight active rows of the mixture-of-experts model: several drafts checked in one pass
        {"name": "rows-moe-q4-8", "kind": "moe_rows", "layers": 27, "start": 480, "rows": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("qgemv", "projections", "attention", "decode", "decode", "prompt", "prompt", "moe_decode", "moe_rows"))
    if kind == "qgemv":
        k = GROUP * _log(rng, 8, 128)
        return {"kind": kind, "n": _log(rng, 256, min(152000, 400_000_000 // k)), "k": k, "bits": rng.choice((4, 8, 16))}
    if kind == "projections":
        hidden, dim = 128 * rng.randint(4, 32), rng.choice((64, 128))
        n_kv = dim * rng.choice((2, 4, 8))
        return {"kind": kind, "hidden": hidden, "inter": GROUP * rng.randint(2 * hidden // GROUP, 6 * hidden // GROUP),
                "n_q": n_kv * rng.choice((1, 2, 4)), "n_kv": n_kv, "bits": rng.choice((4, 8, 16))}
    if kind == "attention":
        n_kv, ratio = rng.choice((2, 4, 8)), rng.choice((1, 2, 4, 7))
        return {"kind": kind, "length": _log(rng, 64, 32768), "n_heads": n_kv * ratio, "n_kv": n_kv, "head_dim": rng.choice((64, 128)),
                "kv_bits": rng.choice((0, 0, 8, 4))}
    if kind == "decode":
        model = rng.choice(("05b", "4b", "small", "wide"))
        layers = MODELS[model]["n_layers"]
        return {"kind": kind, "model": model, "layers": rng.randint(max(6, layers // 2), layers), "bits": rng.choice((4, 4, 8, 16)),
                "kv_bits": rng.choice((0, 0, 8, 4)), "context": _log(rng, 16, 12000), "tokens": rng.randint(4, 24)}
    if kind == "prompt":
        model = rng.choice(("05b", "4b", "small", "wide"))
        layers = MODELS[model]["n_layers"]
        return {"kind": kind, "model": model, "layers": rng.randint(max(6, layers // 2), layers), "bits": rng.choice((4, 4, 8, 16)),
                "kv_bits": rng.choice((0, 0, 0, 8)), "start": rng.choice((0, 0, rng.randint(1, 3000))), "rows": _log(rng, 9, 3000)}
    if kind == "moe_decode":
        return {"kind": kind, "layers": rng.randint(10, 27), "context": _log(rng, 16, 3000), "tokens": rng.randint(4, 24)}
    return {"kind": "moe_rows", "layers": rng.randint(10, 27), "start": _log(rng, 16, 1500), "rows": _log(rng, 2, 96)}


# ---------------------------------------------------------------- inputs

_TYPES = {"bf16": (torch.bfloat16, 2, "<i2"), "f32": (torch.float32, 4, "<f4"), "u8": (torch.uint8, 1, "|u1")}


class _Memory:
    def __init__(self, buf, kind):
        _, size, code = _TYPES[kind]
        self.owner = buf
        self.__cuda_array_interface__ = {"shape": (buf.nbytes // size,), "typestr": code, "data": (buf.ptr, False), "version": 2}


def _view(buf, kind, *shape):
    """A tensor over a device buffer's own memory."""
    t = torch.as_tensor(_Memory(buf, kind), device="cuda").view(_TYPES[kind][0])
    return t.view(*shape) if shape else t


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, mean=0.0, std=1.0, dtype=torch.bfloat16):
    return torch.empty(*shape, dtype=dtype, device="cuda").normal_(mean, std, generator=g)


def _weight(g, n, k, bits):
    """N(0, 0.02^2), quantised as the framework quantises."""
    if bits == 16:
        W = fk.DeviceWeight.__new__(fk.DeviceWeight)
        W.n, W.k, W.bits, W.group, W.scales, W.biases = n, k, 16, 0, None, None
        W.w = fk.DeviceBuffer(n * k * 2)
        _view(W.w, "bf16").normal_(0.0, 0.02, generator=g)
        return W
    w = fk.DeviceBuffer(n * k * 4)
    _view(w, "f32").normal_(0.0, 0.02, generator=g)
    torch.cuda.synchronize()
    W = quantize_on_device(w, n, k, bits, GROUP)
    fk.sync()
    return W


def _fill_quant_cache(cache, g):
    """Codes of every value, scales and biases that spread them as N(0, 1) values are spread."""
    top = (1 << cache.bits) - 1
    _view(cache.packed, "u8").random_(0, 256, generator=g)
    _view(cache.scales, "bf16").normal_(3.5 / top, 0.3 / top, generator=g)
    _view(cache.biases, "bf16").normal_(-1.75, 0.15, generator=g)


def _dense(case, seed, capacity):
    shape = dict(MODELS[case["model"]], n_layers=case["layers"])
    cfg = DecoderConfig(**shape, bits=case["bits"], kv_bits=case["kv_bits"], capacity=capacity, swiglu_variant=1)
    W = DecoderWeights.random_init(cfg, seed=seed % 100003)
    g = _gen(seed)
    table = _view(W.mats["embed_tokens"].w, "bf16", cfg.vocab, cfg.hidden).normal_(0.0, EMBED_STD, generator=g)
    follows = torch.randperm(cfg.vocab, generator=g, device="cuda")
    head = fk.DeviceWeight.__new__(fk.DeviceWeight)
    head.n, head.k, head.bits, head.group, head.scales, head.biases = cfg.vocab, cfg.hidden, 16, 0, None, None
    head.w = fk.DeviceBuffer(cfg.vocab * cfg.hidden * 2)
    _view(head.w, "bf16", cfg.vocab, cfg.hidden).copy_(table[follows])
    W.mats["lm_head"] = head
    rt = DecoderRuntime(cfg, W)
    return cfg, rt, g


def _cache_rows(buffers, heads, capacity, dim, first, count):
    return [_view(b, "bf16", heads, capacity, dim)[:, first:first + count] for b in buffers]


def _written_rows(cfg, rt, first, count):
    """The cache rows that a pass writes: of every layer, or where that is more than 60 buffers K of every even and V of
    every odd layer.  Of a quantised cache the scales and biases (a code next to a rounding boundary may fall either side)."""
    if cfg.kv_bits:
        per = cfg.head_dim // GROUP
        part = {0: lambda c: c.scales, 1: lambda c: c.biases}
        pairs = [(rt.cache_k if l % 2 == 0 else rt.cache_v)[l] for l in range(cfg.n_layers)]
        return _cache_rows([part[(l // 2) % 2](c) for l, c in enumerate(pairs)], cfg.n_kv, cfg.capacity, per, first, count)
    if 2 * cfg.n_layers <= 60:
        bufs = list(rt.cache_k) + list(rt.cache_v)
    else:
        bufs = [(rt.cache_k if l % 2 == 0 else rt.cache_v)[l] for l in range(cfg.n_layers)]
    return _cache_rows(bufs, cfg.n_kv, cfg.capacity, cfg.head_dim, first, count)


def _fill_caches(cfg, rt, g):
    for c in list(rt.cache_k) + list(rt.cache_v):
        if cfg.kv_bits:
            _fill_quant_cache(c, g)
        else:
            _view(c, "bf16").normal_(0.0, 1.0, generator=g)


def _moe(case, seed, capacity):
    cfg = MoeConfig(n_layers=case["layers"], capacity=capacity)
    W = MoeWeights.random_init(cfg, seed=seed % 100003)
    g = _gen(seed)
    # one table serves as embedding and head: tokens come in pairs whose rows agree in one half and are opposite in the
    # other, and the final norm turns the second half's sign, so that each token is followed by the other of its pair
    half = cfg.hidden // 2
    table = _view(W.mats["embed_tokens"].w, "bf16", cfg.vocab // 2, 2, 2, half)
    base = _normal(g, cfg.vocab // 2, 2, half, std=EMBED_STD)
    table[:, 0].copy_(base)
    table[:, 1, 0].copy_(base[:, 0])
    table[:, 1, 1].copy_(-base[:, 1])
    norm = _view(W.vecs["final_norm"], "bf16")
    norm[half:].mul_(-1)
    rt = MoeRuntime(cfg, W)
    for c in list(rt.cache_k) + list(rt.cache_v):
        _view(c, "bf16").normal_(0.0, 1.0, generator=g)
    return cfg, rt


def _moe_written(cfg, rt, first, count):
    return (_cache_rows(rt.cache_k, cfg.n_heads, cfg.capacity, cfg.qk_dim, first, count)
            + _cache_rows(rt.cache_v, cfg.n_heads, cfg.capacity, cfg.v_dim, first, count))


def _capacity(positions):
    return max(256, 256 * -(-positions // 256))


def _tokens(seed, count, vocab):
    return np.random.Generator(np.random.PCG64(seed)).integers(0, vocab, count).tolist()


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "qgemv":
        g = _gen(seed)
        s.update(W=_weight(g, case["n"], case["k"], case["bits"]), x=_normal(g, case["k"]),
                 y=torch.empty(case["n"], dtype=torch.bfloat16, device="cuda"))
    elif kind == "projections":
        g = _gen(seed)
        h, inter, n_q, n_kv, bits = (case[n] for n in ("hidden", "inter", "n_q", "n_kv", "bits"))
        s.update(Wq=_weight(g, n_q, h, bits), Wk=_weight(g, n_kv, h, bits), Wv=_weight(g, n_kv, h, bits),
                 Wg=_weight(g, inter, h, bits), Wu=_weight(g, inter, h, bits), Wd=_weight(g, h, inter, bits),
                 n1=_normal(g, h, mean=1.0, std=0.1), n2=_normal(g, h, mean=1.0, std=0.1), x=_normal(g, h),
                 bias=[_normal(g, n, std=0.5) for n in (n_q, n_kv, n_kv)])
        for name, n in (("q", n_q), ("k", n_kv), ("v", n_kv), ("mid", inter), ("y", h)):
            s[name] = torch.empty(n, dtype=torch.bfloat16, device="cuda")
    elif kind == "attention":
        g = _gen(seed)
        length, nh, nk, d, kvb = (case[n] for n in ("length", "n_heads", "n_kv", "head_dim", "kv_bits"))
        s.update(q=_normal(g, nh * d), k=_normal(g, nk * d), v=_normal(g, nk * d), out=torch.empty(nh * d, dtype=torch.bfloat16, device="cuda"),
                 scale=1.0 / math.sqrt(d))
        pb, cb = fk.sdpa_workspace_bytes(nh, nk, d, d, length)
        s.update(parts=fk.DeviceBuffer(max(pb, 4)), counters=fk.zeros(max(cb, 4)))
        if kvb:
            s["K"], s["V"] = (fk.QuantKvCache(nk, length, d, kvb, GROUP) for _ in range(2))
            for c in (s["K"], s["V"]):
                _fill_quant_cache(c, g)
            s["rows"] = [_view(b, "bf16", nk, length, d // GROUP)[:, length - 1:] for c in (s["K"], s["V"]) for b in (c.scales, c.biases)]
        else:
            s["K"], s["V"] = (_normal(g, nk, length, d) for _ in range(2))
            s["rows"] = [s["K"][:, length - 1:], s["V"][:, length - 1:]]
    elif kind == "decode":
        first, count = case["context"], case["tokens"]
        cfg, rt, g = _dense(case, seed, _capacity(first + count))
        _fill_caches(cfg, rt, g)
        s.update(rt=rt, rows=_written_rows(cfg, rt, first, count), logits=_view(rt.logits, "bf16"), token=_tokens(seed, 1, cfg.vocab)[0])
    elif kind == "prompt":
        first, count = case["start"], case["rows"]
        cfg, rt, g = _dense(case, seed, _capacity(first + count))
        _fill_caches(cfg, rt, g)
        s.update(rt=rt, rows=_written_rows(cfg, rt, first, count), logits=_view(rt.logits, "bf16"),
                 prompt=_tokens(seed, count, cfg.vocab))
    elif kind == "moe_decode":
        first, count = case["context"], case["tokens"]
        cfg, rt = _moe(case, seed, _capacity(first + count))
        s.update(rt=rt, rows=_moe_written(cfg, rt, first, count), logits=_view(rt.logits, "bf16"), token=_tokens(seed, 1, cfg.vocab)[0])
    else:
        first, count = case["start"], case["rows"]
        cfg, rt = _moe(case, seed, _capacity(first + count))
        s.update(rt=rt, rows=_moe_written(cfg, rt, first, count), logits=_view(rt.logits, "bf16"), prompt=_tokens(seed, count, cfg.vocab))
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "qgemv":
        fk.qgemv(s["W"], s["x"].data_ptr(), None, s["y"].data_ptr())
        return s["y"]
    if kind == "projections":
        bq, bk, bv = (b.data_ptr() for b in s["bias"])
        x, q, k, v, mid, y = (s[n].data_ptr() for n in ("x", "q", "k", "v", "mid", "y"))
        fk.rmsnorm_qkv(x, s["n1"].data_ptr(), 1e-6, s["Wq"], s["Wk"], s["Wv"], bq, bk, bv, q, k, v)
        fk.gateup_swiglu(x, s["n2"].data_ptr(), 1e-6, s["Wg"], s["Wu"], 1, mid)
        fk.linear_residual(s["Wd"], mid, x, None, y)
        return {n: s[n] for n in ("q", "k", "v", "mid", "y")}
    if kind == "attention":
        length, nh, nk, d = (case[n] for n in ("length", "n_heads", "n_kv", "head_dim"))
        q, k, v, out = (s[n].data_ptr() for n in ("q", "k", "v", "out"))
        if case["kv_bits"]:     # q comes rotated
            fk.kv_cache_store_quant(k, v, None, nk, d, d, 1e6, 1e-6, None, length - 1, 1, s["K"], s["V"])
            fk.sdpa_decode_quant(q, s["K"], s["V"], out, None, length, length, 1, nh, s["scale"], s["parts"], s["counters"])
        else:
            fk.rope_store_sdpa_decode(q, k, v, None, None, s["K"].data_ptr(), s["V"].data_ptr(), out, None, length, length, nh, nk, d, d,
                                      1e6, 1e-6, length, s["scale"], None, s["parts"], s["counters"])
        return {"out": s["out"], "rows": s["rows"]}
    rt = s["rt"]
    if kind in ("decode", "moe_decode"):
        tokens, _ = rt.d.decode_chunk(rt.graph, rt.uniforms, case["context"], s["token"], case["tokens"])
        return {"tokens": np.array(tokens, np.int64), "logits": s["logits"], "rows": s["rows"]}
    if kind == "prompt":
        nxt = rt.prefill_rows(s["prompt"], case["start"])
    else:
        nxt = rt.forward_rows(s["prompt"], case["start"])
    return {"next": nxt, "logits": s["logits"], "rows": s["rows"]}


# ---------------------------------------------------------------- what a pass cannot do without

def _per_weight(bits):
    return bits / 8 + (0 if bits == 16 else 4 / GROUP)


def _per_value(kv_bits):
    return kv_bits / 8 + 4 / GROUP if kv_bits else 2.0


def work(case):
    kind = case["kind"]
    if kind == "qgemv":
        n, k = case["n"], case["k"]
        return {"bytes": n * k * _per_weight(case["bits"]) + 2 * (n + k), "flops": 2.0 * n * k}
    if kind == "projections":
        h, inter, n_q, n_kv = (case[n] for n in ("hidden", "inter", "n_q", "n_kv"))
        p = h * (n_q + 2 * n_kv) + 3 * h * inter
        return {"bytes": p * _per_weight(case["bits"]) + 2 * (5 * h + 2 * (n_q + 2 * n_kv) + 2 * inter), "flops": 2.0 * p}
    if kind == "attention":
        length, nh, nk, d = (case[n] for n in ("length", "n_heads", "n_kv", "head_dim"))
        return {"bytes": 2 * nk * d * length * _per_value(case["kv_bits"]) + 4 * nh * d, "flops": 4.0 * nh * d * length}
    if kind in ("decode", "prompt"):
        m = MODELS[case["model"]]
        h, d, nh, nk = m["hidden"], m["head_dim"], m["n_heads"], m["n_kv"]
        p = case["layers"] * (h * (nh + 2 * nk) * d + nh * d * h + 3 * h * m["inter"])
        head = m["vocab"] * h
        kv_row = case["layers"] * 2 * nk * d * _per_value(case["kv_bits"])
        if kind == "decode":
            t, first = case["tokens"], case["context"]
            seen = t * first + t * (t + 1) // 2
            return {"bytes": t * (p * _per_weight(case["bits"]) + 2 * head) + kv_row * seen,
                    "flops": t * 2.0 * (p + head) + 4.0 * case["layers"] * nh * d * seen}
        r, first = case["rows"], case["start"]
        seen = r * first + r * (r + 1) // 2
        return {"bytes": p * _per_weight(case["bits"]) + 2 * head + kv_row * (first + r) + 2 * r * h,
                "flops": 2.0 * (r * p + head) + 4.0 * case["layers"] * nh * d * seen}
    c = MoeConfig(n_layers=case["layers"])
    attn = c.hidden * (c.n_heads * c.qk_dim + c.kv_lora_rank + c.rope_dim) + c.kv_lora_rank * c.n_heads * (c.nope_dim + c.v_dim) \
        + c.n_heads * c.v_dim * c.hidden
    expert, n_moe = 3 * c.hidden * c.moe_inter, c.n_layers - c.first_dense
    fixed = c.n_layers * attn + n_moe * c.n_shared * expert + c.first_dense * 3 * c.hidden * c.dense_inter
    router, head = n_moe * c.n_experts * c.hidden, c.vocab * c.hidden
    kv_row = c.n_layers * c.n_heads * (c.qk_dim + c.v_dim) * 2
    once = fixed + n_moe * c.top_k * expert
    if kind == "moe_decode":
        t, first = case["tokens"], case["context"]
        seen = t * first + t * (t + 1) // 2
        return {"bytes": t * (once * _per_weight(4) + 2 * (router + head)) + kv_row * seen,
                "flops": t * 2.0 * (once + router + head) + 2.0 * c.n_layers * c.n_heads * (c.qk_dim + c.v_dim) * seen}
    r, first = case["rows"], case["start"]
    seen = r * first + r * (r + 1) // 2
    touched = c.n_experts * (1 - (1 - c.top_k / c.n_experts) ** r)   # distinct experts of r rows
    return {"bytes": (fixed + n_moe * touched * expert) * _per_weight(4) + 2 * (router + head) + kv_row * (first + r) + 2 * r * c.hidden,
            "flops": 2.0 * (r * (once + router) + head) + 2.0 * c.n_layers * c.n_heads * (c.qk_dim + c.v_dim) * seen}


def tolerance(case):
    """bf16 activations with fp32 accumulation: one call is good to some 2e-3; in a model the roundings of every layer add
    up, about 2.5e-3 times the square root of the number of layers between two forms of the same layer."""
    if case["kind"] in ("qgemv", "projections", "attention"):
        return {"rel": 5e-3, "max": 0.1}
    return {"rel": round(0.0035 * math.sqrt(case["layers"]), 4), "max": 0.2, "differ": 0.0}
