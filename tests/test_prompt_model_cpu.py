"""What a prompt pass points to: the model that a runtime keeps for its prompts follows the buffers that the caller puts in place of
others, and keeps alive what it points to.  No device: the buffers are stand-ins and the native call is recorded."""
import gc
import itertools
import weakref

import numpy as np
import pytest

import fusekit_amd.decoder as decoder
import fusekit_amd.native as native
from fusekit_amd.decoder import DecoderConfig, DecoderRuntime, DecoderWeights

_addresses = itertools.count(4096, 256)


class Buffer(native.DeviceBuffer):
    def __init__(self, nbytes=16):
        self.nbytes, self.ptr = nbytes, next(_addresses)

    def free(self):
        self.ptr = None


def _matrix(n, k, bits):
    W = native.DeviceWeight.__new__(native.DeviceWeight)
    W.n, W.k, W.bits, W.group = n, k, bits, 0 if bits == 16 else 64
    W.w, W.scales, W.biases = Buffer(), *((None, None) if bits == 16 else (Buffer(), Buffer()))
    return W


def _runtime(kv_bits=0):
    c = DecoderConfig(n_layers=2, hidden=512, n_heads=4, n_kv=2, head_dim=64, inter=1024, vocab=100, capacity=256, qk_norm=True, kv_bits=kv_bits)
    w = DecoderWeights(c)
    for l in range(c.n_layers):
        for n in ("self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj", "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj"):
            w.mats[f"layers.{l}.{n}"] = _matrix(64, 512, 4)
        for n in ("input_layernorm", "post_attention_layernorm", "self_attn.q_norm", "self_attn.k_norm"):
            w.vecs[f"layers.{l}.{n}"] = Buffer()
    w.mats["embed_tokens"], w.vecs["final_norm"] = _matrix(100, 512, 16), Buffer()
    rt = DecoderRuntime.__new__(DecoderRuntime)
    rt.cfg, rt.w = c, w
    rt._rows, rt._rows_R = {n: Buffer() for n in ("tok", "x", "x2", "xn", "q", "k", "v", "att", "mid", "ws", "part", "cnt", "rope", "kdq", "vdq")}, 4096
    rt._prompt_models, rt._bf16_weights = {}, {}
    rt._prompt_held, rt._prompt_buffers, rt._prompt_assigned, rt._bf16_sources = [], [], -1, {}
    def cache():
        if not kv_bits:
            return Buffer()
        C = native.QuantKvCache.__new__(native.QuantKvCache)
        C.packed, C.scales, C.biases = Buffer(), Buffer(), Buffer()
        return C
    rt.cache_k, rt.cache_v = ([cache() for _ in range(c.n_layers)] for _ in range(2))
    rt.logits, rt.token, rt.argmax_ws, rt.step_counter = Buffer(), Buffer(), Buffer(), Buffer()
    return rt, cache


def _pointers(model, kv_bits):
    """Every address in the model."""
    out = {n: getattr(model, n) for n in ("final_norm", "logits", "token", "argmax_workspace", "step_counter")}
    for name in ("embed", "head"):
        out[name] = getattr(model, name).w
    for l in range(model.n_layers):
        L = model.layers[l]
        for name in ("q", "k", "v", "o", "gate", "up", "down"):
            W = getattr(L, name)
            out[l, name] = (W.w, W.scales, W.biases, W.n, W.k, W.bits)
        for name in ("input_norm", "post_norm", "q_norm", "k_norm", "cache_k", "cache_v"):
            out[l, name] = getattr(L, name)
        if kv_bits:
            for name in ("cache_kq", "cache_vq"):
                out[l, name] = tuple(getattr(getattr(L, name), f) for f, _ in getattr(L, name)._fields_)
    return out


def _replace_matrix(rt, cache):
    rt.w.mats["layers.1.self_attn.o_proj"] = _matrix(512, 256, 4)


def _replace_codes(rt, cache):
    rt.w.mats["layers.0.mlp.up_proj"].scales = Buffer()


def _replace_vector(rt, cache):
    rt.w.vecs["layers.1.post_attention_layernorm"] = Buffer()


def _replace_cache(rt, cache):
    rt.cache_k[1], rt.cache_v[0] = cache(), cache()


def _add_head(rt, cache):
    rt.w.mats["lm_head"] = _matrix(100, 512, 16)


def _replace_logits(rt, cache):
    rt.logits = Buffer()


@pytest.mark.parametrize("kv_bits", [0, 8])
@pytest.mark.parametrize("replace", [_replace_matrix, _replace_codes, _replace_vector, _replace_cache, _add_head, _replace_logits])
def test_a_prompt_reads_what_is_in_place_now(monkeypatch, replace, kv_bits):
    seen = []
    monkeypatch.setattr(decoder.native, "prompt_run", lambda model, *a: seen.append((model, _pointers(model, kv_bits))) or 7)
    rt, cache = _runtime(kv_bits)
    assert rt.prefill_rows([1, 2, 3]) == 7 and rt.prefill_rows([1, 2, 3]) == 7
    assert seen[0][1] == seen[1][1] and seen[0][0].layers[0].q.w == seen[1][0].layers[0].q.w
    replace(rt, cache)
    gc.collect()
    rt.prefill_rows([1, 2, 3])
    assert seen[2][1] != seen[1][1]
    fresh, _ = _runtime(kv_bits)
    fresh.w, fresh._rows, fresh.cache_k, fresh.cache_v = rt.w, rt._rows, rt.cache_k, rt.cache_v
    fresh.logits, fresh.token, fresh.argmax_ws, fresh.step_counter = rt.logits, rt.token, rt.argmax_ws, rt.step_counter
    fresh.prefill_rows([1, 2, 3])
    assert seen[3][1] == seen[2][1]


def test_what_the_kept_model_points_to_lives_as_long(monkeypatch):
    monkeypatch.setattr(decoder.native, "prompt_run", lambda *a: 7)
    rt, _ = _runtime()
    rt.prefill_rows([1, 2, 3])
    W = rt.w.mats["layers.0.mlp.up_proj"]
    old = [weakref.ref(b) for b in (rt.cache_k[0], W.w, W.scales, rt.w.vecs["layers.0.input_layernorm"])]
    rt.cache_k[0], W.w, W.scales, rt.w.vecs["layers.0.input_layernorm"] = Buffer(), Buffer(), Buffer(), Buffer()
    gc.collect()
    assert all(r() is not None for r in old)           # still what the kept model would read
    rt.prefill_rows([1, 2, 3])
    gc.collect()
    assert all(r() is None for r in old)


def test_the_model_is_kept_while_nothing_changes(monkeypatch):
    seen = []
    monkeypatch.setattr(decoder.native, "prompt_run", lambda model, *a: seen.append(model) or 7)
    monkeypatch.setattr(decoder.native, "gemm_library_available", lambda: True)
    monkeypatch.setattr(decoder.native, "dequantize_bf16", lambda W: _matrix(W.n, W.k, 16))
    rt, _ = _runtime()
    rt.cfg.capacity = 4096
    for keep in (True, False):          # (the copies themselves assign buffers)
        for _ in range(3):
            rt.prefill_rows(list(range(300)), keep_bf16_weights=keep)
    assert all(m is seen[0] for m in seen[:3]) and all(m is seen[3] for m in seen[3:])


def test_a_replaced_matrix_gets_a_new_bf16_copy(monkeypatch):
    monkeypatch.setattr(decoder.native, "prompt_run", lambda *a: 7)
    monkeypatch.setattr(decoder.native, "gemm_library_available", lambda: True)
    monkeypatch.setattr(decoder.native, "dequantize_bf16", lambda W: _matrix(W.n, W.k, 16))
    rt, cache = _runtime()
    prompt = np.arange(256).tolist()
    rt.cfg.capacity = 4096
    rt.prefill_rows(prompt, keep_bf16_weights=True)
    kept = dict(rt._bf16_weights)
    _replace_matrix(rt, cache)
    _replace_codes(rt, cache)
    rt.prefill_rows(prompt, keep_bf16_weights=True)
    assert sorted(n for n in kept if rt._bf16_weights[n] is not kept[n]) == ["layers.0.mlp.up_proj", "layers.1.self_attn.o_proj"]
