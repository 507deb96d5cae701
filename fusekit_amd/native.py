"""ctypes binding of libfusekit_hip.so (the C ABI in include/fusekit_hip.h).

Mirrors how the reference's Python runtime talks to `_fusekit_runtime_native`
(reference python/fusekit_runtime/dispatch.py -> python_runtime/src/lib.rs):
Python owns no arithmetic, only pointers and sizes.  bf16 tensors travel as
numpy uint16 bit patterns.  Loading fails loudly when the library is missing;
there is no fallback path.
"""
from __future__ import annotations

import ctypes as C
import os

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("FUSEKIT_HIP_LIB") or os.path.join(_HERE, "libfusekit_hip.so")

FK_OK, FK_ERR_INVALID, FK_ERR_IO, FK_ERR_NOT_FOUND, FK_ERR_HIP, FK_ERR_UNSUPPORTED = range(6)


class FusekitError(RuntimeError):
    def __init__(self, status: int, message: str):
        super().__init__(f"[fk_status {status}] {message}")
        self.status = status


class InvalidArgument(FusekitError, ValueError):
    """FK_ERR_INVALID: what the reference raises as PyValueError."""


def _load() -> C.CDLL:
    if not os.path.exists(LIB_PATH):
        raise ImportError(
            f"{LIB_PATH} is missing: build it with `python -c 'import __graft_entry__ as g; g.build()'` "
            "(hipcc, gfx950). fusekit_amd has no CPU fallback."
        )
    return C.CDLL(LIB_PATH)


lib = _load()
lib.fk_last_error.restype = C.c_char_p
lib.fk_version.restype = C.c_char_p


def check(status: int) -> None:
    if status != FK_OK:
        msg = lib.fk_last_error().decode("utf-8", "replace")
        if status == FK_ERR_INVALID:
            raise InvalidArgument(status, msg)
        raise FusekitError(status, msg)


def version() -> str:
    return lib.fk_version().decode()


class DeviceProps(C.Structure):
    _fields_ = [
        ("name", C.c_char * 128), ("arch", C.c_char * 32), ("compute_units", C.c_int), ("wavefront", C.c_int),
        ("lds_bytes_per_block", C.c_int), ("l2_bytes", C.c_int), ("hbm_bytes", C.c_uint64), ("clock_khz", C.c_int),
    ]


class Target(C.Structure):
    """fk_target: the gfx950 entry of the reference's ChipModel / Budgets table."""
    _fields_ = [("arch", C.c_char * 32), ("from_device", C.c_uint32), ("compute_units", C.c_uint32),
                ("xcds", C.c_uint32), ("wave_size", C.c_uint32), ("simds_per_cu", C.c_uint32),
                ("vgprs_per_lane", C.c_uint32), ("lds_bytes_per_cu", C.c_uint32), ("workgroup_threads", C.c_uint32),
                ("gemm_min_rows", C.c_uint32), ("gemm_rows_per_pass", C.c_uint32), ("hbm_bytes", C.c_uint64),
                ("hbm_peak_bytes_per_s", C.c_double), ("mfma_bf16_peak_flops", C.c_double)]


def target_describe() -> Target:
    t = Target()
    check(lib.fk_target_describe(C.byref(t)))
    return t


def device_props() -> DeviceProps:
    p = DeviceProps()
    check(lib.fk_device_props_get(C.byref(p)))
    return p


def mem_info():
    """(free, total) device memory in bytes."""
    a, b = C.c_size_t(), C.c_size_t()
    check(lib.fk_mem_info(C.byref(a), C.byref(b)))
    return a.value, b.value


def has_device() -> bool:
    p = DeviceProps()
    return lib.fk_device_props_get(C.byref(p)) == FK_OK


class Weight(C.Structure):
    """`fk_weight`."""

    _fields_ = [
        ("w", C.c_void_p), ("scales", C.c_void_p), ("biases", C.c_void_p),
        ("n", C.c_uint32), ("k", C.c_uint32), ("bits", C.c_uint32), ("group", C.c_uint32),
    ]


class DeviceBuffer:
    """One device allocation owned through fk_alloc / fk_free."""

    def __init__(self, nbytes: int):
        self.nbytes = int(nbytes)
        p = C.c_void_p()
        check(lib.fk_alloc(C.c_size_t(max(self.nbytes, 1)), C.byref(p)))
        self.ptr = p.value

    @classmethod
    def from_numpy(cls, a: np.ndarray) -> "DeviceBuffer":
        a = np.ascontiguousarray(a)
        b = cls(a.nbytes)
        if a.nbytes:
            check(lib.fk_upload(C.c_void_p(b.ptr), a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes)))
        return b

    def upload(self, a: np.ndarray, offset: int = 0) -> None:
        a = np.ascontiguousarray(a)
        assert offset + a.nbytes <= self.nbytes
        check(lib.fk_upload(C.c_void_p(self.ptr + offset), a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes)))

    def to_numpy(self, dtype, shape=None, offset: int = 0) -> np.ndarray:
        dtype = np.dtype(dtype)
        if shape is None:
            shape = ((self.nbytes - offset) // dtype.itemsize,)
        out = np.empty(shape, dtype=dtype)
        assert offset + out.nbytes <= self.nbytes
        if out.nbytes:
            check(lib.fk_download(out.ctypes.data_as(C.c_void_p), C.c_void_p(self.ptr + offset),
                                  C.c_size_t(out.nbytes)))
        return out

    def free(self) -> None:
        if getattr(self, "ptr", None):
            lib.fk_free(C.c_void_p(self.ptr))
            self.ptr = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class DeviceWeight:
    """A weight matrix resident in HBM (packed + scales + biases, or dense bf16)."""

    assigned = 0   # how often a buffer of any matrix has been assigned: unchanged, no matrix has been given another buffer

    _c = None      # the operators' struct and the addresses it holds

    def __setattr__(self, name: str, value) -> None:
        object.__setattr__(self, name, value)
        self.__dict__.pop("_c", None)
        if name in ("w", "scales", "biases"):
            DeviceWeight.assigned += 1

    def __init__(self, w: np.ndarray, scales, biases, n: int, k: int, bits: int, group: int = 64):
        self.n, self.k, self.bits, self.group = int(n), int(k), int(bits), int(group)
        self.w = DeviceBuffer.from_numpy(w)
        self.scales = None if scales is None else DeviceBuffer.from_numpy(np.asarray(scales, dtype=np.uint16))
        self.biases = None if biases is None else DeviceBuffer.from_numpy(np.asarray(biases, dtype=np.uint16))

    @property
    def c(self) -> Weight:
        """fk_weight, the caller's own."""
        scales, biases = self.scales, self.biases
        return Weight(self.w.ptr, scales.ptr if scales else None, biases.ptr if biases else None, self.n, self.k, self.bits, self.group)

    @property
    def nbytes(self) -> int:
        return self.w.nbytes + (self.scales.nbytes + self.biases.nbytes if self.scales else 0)


def _addr(b):
    """A device address as the declared signatures (_SIGNATURES) take it: an int or None."""
    if b is None or b.__class__ is int:
        return b
    return b.ptr if isinstance(b, DeviceBuffer) else int(b)


def _w(W):
    """An fk_weight operand (a call copies what it needs): of a DeviceWeight made when an attribute has been set or a buffer's address is
    another.  Nothing else holds that one: what a caller does with W.c must not change the next call."""
    if W.__class__ is not DeviceWeight:
        return W.c
    scales, biases = W.scales, W.biases
    at = (W.w.ptr, scales.ptr if scales else None, biases.ptr if biases else None)
    kept = W._c
    if kept is None or kept[0] != at:
        kept = (at, Weight(*at, W.n, W.k, W.bits, W.group))
        W.__dict__["_c"] = kept
    return kept[1]


def _ptr(b) -> C.c_void_p:
    if b is None:
        return C.c_void_p(None)
    if isinstance(b, DeviceBuffer):
        return C.c_void_p(b.ptr)
    return C.c_void_p(int(b))


# ---------------------------------------------------------------- operators

def qgemv(W: DeviceWeight, x, bias, y, stream=None) -> None:
    check(lib.fk_qgemv(_w(W), _addr(x), _addr(bias), _addr(y), _addr(stream)))


def linear_residual(W: DeviceWeight, x, res, res2, y, stream=None) -> None:
    check(lib.fk_linear_residual(_w(W), _addr(x), _addr(res), _addr(res2), _addr(y), _addr(stream)))


def rmsnorm_qkv(x, norm_w, eps, Wq, Wk, Wv, bq, bk, bv, q, k, v, stream=None) -> None:
    check(lib.fk_rmsnorm_qkv(_addr(x), _addr(norm_w), eps, _w(Wq), _w(Wk), _w(Wv), _addr(bq), _addr(bk), _addr(bv), _addr(q),
                             _addr(k), _addr(v), _addr(stream)))


def gateup_swiglu_rows(x, rows, norm_w, eps, Wg, Wu, variant, out, stream=None) -> None:
    """fk_gateup_swiglu_rows: RMSNorm + gate / up + SwiGLU of 2..8 token rows in one launch."""
    check(lib.fk_gateup_swiglu_rows(_addr(x), rows, _addr(norm_w), eps, _w(Wg), _w(Wu), variant, _addr(out), _addr(stream)))


def rmsnorm_qkv_rows(x, rows, x_row_stride, norm_w, eps, Wq, Wk, Wv, q, q_row_stride, k=None, k_row_stride=0, v=None,
                     v_row_stride=0, stream=None) -> None:
    """fk_rmsnorm_qkv_rows: RMSNorm + one to three projections of 2..8 token rows in one launch."""
    wk = _w(Wk) if Wk is not None else None
    wv = _w(Wv) if Wv is not None else None
    check(lib.fk_rmsnorm_qkv_rows(_addr(x), rows, x_row_stride, _addr(norm_w), eps, _w(Wq), wk, wv, _addr(q), q_row_stride,
                                  _addr(k), k_row_stride, _addr(v), v_row_stride, _addr(stream)))


def gateup_swiglu(x, norm_w, eps, Wg, Wu, variant, out, stream=None) -> None:
    check(lib.fk_gateup_swiglu(_addr(x), _addr(norm_w), eps, _w(Wg), _w(Wu), variant, _addr(out), _addr(stream)))


def routed_qmv_swiglu(x, n_x_rows, Wg, Wu, n_experts, row_idx, expert_idx, route_weight, n_routes, out0,
                      stream=None) -> None:
    """Wg / Wu: DeviceWeight whose arrays are stacked [E, n, ...] and whose n, k describe one expert."""
    check(lib.fk_routed_qmv_swiglu(_addr(x), n_x_rows, _w(Wg), _w(Wu), n_experts, _addr(row_idx), _addr(expert_idx),
                                   _addr(route_weight), n_routes, _addr(out0), _addr(stream)))


def routed_qmv_swiglu_shared(x, Wg, Wu, n_experts, expert_idx, route_weight, n_routes, out0, Sg, Su, shared_out,
                             stream=None) -> None:
    """One token: the routed gate/up + SwiGLU with the shared experts' pair as further routes of the same launch."""
    check(lib.fk_routed_qmv_swiglu_shared(_addr(x), _w(Wg), _w(Wu), n_experts, _addr(expert_idx), _addr(route_weight), n_routes,
                                          _addr(out0), _w(Sg), _w(Su), _addr(shared_out), _addr(stream)))


def routed_qmv_swiglu_routing(x, Wg, Wu, n_experts, logits, scale, top_k, apply_weight, idx_out, weight_out, out0, Sg=None,
                              Su=None, shared_out=None, stream=None) -> None:
    """One token: the routed (+ shared) gate/up launch ranking the router logits itself (fk_routed_qmv_swiglu_routing)."""
    check(lib.fk_routed_qmv_swiglu_routing(_addr(x), _w(Wg), _w(Wu), n_experts, _addr(logits), _addr(scale), top_k,
                                           int(apply_weight), _addr(idx_out), _addr(weight_out), _addr(out0),
                                           _w(Sg) if Sg is not None else None, _w(Su) if Su is not None else None,
                                           _addr(shared_out), _addr(stream)))


lib.fk_routed_reduce_workspace_bytes.restype = C.c_size_t


lib.fk_routed_reduce_workspace_bytes_shared.restype = C.c_size_t


def routed_reduce_workspace_bytes(n_tokens, top_k, out_dim, shared_k=0, group=64) -> int:
    """shared_k: input width of a shared expert (several tokens then also need the multi-row matmul's workspace)."""
    return int(lib.fk_routed_reduce_workspace_bytes_shared(C.c_uint32(n_tokens), C.c_uint32(top_k), C.c_uint32(out_dim),
                                                           C.c_uint32(shared_k), C.c_uint32(group)))


def routed_qmv_reduce(h, n_h_rows, Wd, n_experts, row_idx, expert_idx, route_weight, shared_x, W_shared,
                      residual_extra, n_tokens, top_k, out, workspace, stream=None) -> None:
    check(lib.fk_routed_qmv_reduce(_addr(h), n_h_rows, _w(Wd), n_experts, _addr(row_idx), _addr(expert_idx),
                                   _addr(route_weight), _addr(shared_x), _w(W_shared) if W_shared is not None else None,
                                   _addr(residual_extra), n_tokens, top_k, _addr(out), _addr(workspace), _addr(stream)))


def routed_qmv_swiglu_ordered(x, n_x_rows, Wg, Wu, n_experts, row_idx, expert_idx, route_weight, n_routes, order, out0,
                              stream=None) -> None:
    """fk_routed_qmv_swiglu with the routes served one by one in `order` (fk_route_order): the same products, a dot product added up
    as the listed launch of few routes does it (a call whose routes are served together may differ in the last bit)."""
    check(lib.fk_routed_qmv_swiglu_ordered(_addr(x), n_x_rows, _w(Wg), _w(Wu), n_experts, _addr(row_idx), _addr(expert_idx),
                                           _addr(route_weight), n_routes, _addr(order), _addr(out0), _addr(stream)))


def routed_qmv_reduce_ordered(h, n_h_rows, Wd, n_experts, row_idx, expert_idx, route_weight, shared_x, W_shared,
                              residual_extra, n_tokens, top_k, order, out, workspace, stream=None) -> None:
    check(lib.fk_routed_qmv_reduce_ordered(_addr(h), n_h_rows, _w(Wd), n_experts, _addr(row_idx), _addr(expert_idx),
                                           _addr(route_weight), _addr(shared_x), _w(W_shared) if W_shared is not None else None,
                                           _addr(residual_extra), n_tokens, top_k, _addr(order), _addr(out), _addr(workspace),
                                           _addr(stream)))


def set_routed_fused_reduce(on: bool) -> None:
    lib.fk_set_routed_fused_reduce(C.c_int(int(on)))


def qgemm_workspace_bytes(m, n, k, group=64) -> int:
    out = C.c_size_t(0)
    check(lib.fk_qgemm_workspace_bytes(C.c_uint32(m), C.c_uint32(n), C.c_uint32(k), C.c_uint32(group), C.byref(out)))
    return int(out.value)


def qgemm(W, x, m, bias, residual, y, workspace, stream=None) -> None:
    check(lib.fk_qgemm(_w(W), _addr(x), m, _addr(bias), _addr(residual), _addr(y), _addr(workspace), _addr(stream)))


def qgemm_fanout(Ws, x, m, biases, ys, workspace, stream=None) -> None:
    """One to three matrices over the same activation rows (q / k / v of a prompt pass); workspace:
    qgemm_workspace_bytes(m, sum of n, k, group)."""
    n = len(Ws)
    w_arr = (C.POINTER(type(Ws[0].c)) * n)(*[C.pointer(W.c) for W in Ws])
    y_arr = (C.c_void_p * n)(*[_ptr(y).value for y in ys])
    b_arr = None if biases is None else (C.c_void_p * n)(*[_ptr(b).value for b in biases])
    check(lib.fk_qgemm_fanout(w_arr, C.c_uint32(n), _ptr(x), C.c_uint32(m), b_arr, y_arr, _ptr(workspace), _ptr(stream)))


def qgemm_swiglu(Wg, Wu, x, m, variant, out, workspace, stream=None) -> None:
    check(lib.fk_qgemm_swiglu(_w(Wg), _w(Wu), _addr(x), m, variant, _addr(out), _addr(workspace), _addr(stream)))


def final_rmsnorm_lm_head(x, norm_w, eps, W, logits, stream=None) -> None:
    check(lib.fk_final_rmsnorm_lm_head(_addr(x), _addr(norm_w), eps, _w(W), _addr(logits), _addr(stream)))


HEAD_ARGMAX_WORKSPACE_BYTES = 32776


def final_rmsnorm_lm_head_argmax(x, norm_w, eps, W, logits, next_token, history, hist_counter, hist_capacity, workspace,
                                 stream=None) -> None:
    """The LM head that also selects the greedy token (one launch); UnsupportedError unless gemv_form(...) == 1."""
    check(lib.fk_final_rmsnorm_lm_head_argmax(_addr(x), _addr(norm_w), eps, _w(W), _addr(logits), _addr(next_token),
                                              _addr(history), _addr(hist_counter), hist_capacity, _addr(workspace),
                                              _addr(stream)))


def rope_q_decode(q, q_norm, n_heads, head_dim, rope_dims, theta, eps=0.0, d_offset=None, offset=0, stream=None):
    check(lib.fk_rope_q_decode(_addr(q), _addr(q_norm), n_heads, head_dim, rope_dims, theta, eps, _addr(d_offset), offset,
                               _addr(stream)))


def rope_kv_cache_store_decode(k, v, k_norm, n_kv, k_dim, v_dim, rope_dims, theta, eps, d_offset, offset,
                               d_write_offset, write_offset, capacity, cache_k, cache_v, stream=None):
    check(lib.fk_rope_kv_cache_store_decode(_addr(k), _addr(v), _addr(k_norm), n_kv, k_dim, v_dim, rope_dims, theta, eps,
                                            _addr(d_offset), offset, _addr(d_write_offset), write_offset, capacity,
                                            _addr(cache_k), _addr(cache_v), _addr(stream)))


def kv_cache_store_split_decode(q, n_heads, q0_dim, q1_dim, k0, k0_stride, k1, k1_heads, v, v_stride, n_kv, k0_dim,
                                k1_dim, v_dim, rope_dims, traditional, theta, d_offset, offset, d_write_offset,
                                write_offset, capacity, cache_k, cache_v, stream=None):
    """Cache K row = [K0 | rope(K1)], V row; with a query also rope(Q1) in place (fk_kv_cache_store_split_decode)."""
    check(lib.fk_kv_cache_store_split_decode(_addr(q), n_heads, q0_dim, q1_dim, _addr(k0), k0_stride, _addr(k1), k1_heads,
                                             _addr(v), v_stride, n_kv, k0_dim, k1_dim, v_dim, rope_dims, int(traditional),
                                             theta, _addr(d_offset), offset, _addr(d_write_offset), write_offset, capacity,
                                             _addr(cache_k), _addr(cache_v), _addr(stream)))


def split_store_sdpa_decode(q, n_heads, q0_dim, q1_dim, k0, k0_stride, k1, k1_heads, v, v_stride, n_kv, v_dim, rope_dims,
                            traditional, theta, rope_tab, cache_k, cache_v, out, d_kv_len, kv_len, max_len, capacity, scale,
                            partials, counters, stream=None):
    """Split-key cache store + attention of a layer in one launch (fk_split_store_sdpa_decode)."""
    check(lib.fk_split_store_sdpa_decode(_addr(q), n_heads, q0_dim, q1_dim, _addr(k0), k0_stride, _addr(k1), k1_heads,
                                         _addr(v), v_stride, n_kv, v_dim, rope_dims, int(traditional), theta, _addr(rope_tab),
                                         _addr(cache_k), _addr(cache_v), _addr(out), _addr(d_kv_len), kv_len, max_len,
                                         capacity, scale, _addr(partials), _addr(counters), _addr(stream)))


def softmax_topk_route(logits, scale, scale_per_route, rows, row_n, top_k, idx, weight, stream=None):
    check(lib.fk_softmax_topk_route(_addr(logits), _addr(scale), int(scale_per_route), rows, row_n, top_k, _addr(idx),
                                    _addr(weight), _addr(stream)))


def moe_router(x, norm_w, eps, w, scale, hidden, experts, top_k, xn, logits, idx, weight, workspace, rows=1, stream=None):
    """RMSNorm + router projection (bf16 weights) + softmax top-k route in one launch (fk_moe_router);
    workspace: zeros(4 * rows * (experts + 1)), reusable by launches that do not overlap."""
    check(lib.fk_moe_router(_addr(x), _addr(norm_w), eps, _addr(w), _addr(scale), hidden, experts, top_k, _addr(xn),
                            _addr(logits), _addr(idx), _addr(weight), _addr(workspace), rows, _addr(stream)))


def kv_cache_store_split_rows(q, n_heads, q0_dim, q1_dim, k0, k0_stride, k0_row_stride, k1, k1_heads, k1_row_stride, v, v_stride,
                              v_row_stride, n_kv, k0_dim, k1_dim, v_dim, rope_dims, traditional, theta, rows, offset, capacity,
                              cache_k, cache_v, stream=None):
    check(lib.fk_kv_cache_store_split_rows(_addr(q), n_heads, q0_dim, q1_dim, _addr(k0), k0_stride, k0_row_stride, _addr(k1),
                                           k1_heads, k1_row_stride, _addr(v), v_stride, v_row_stride, n_kv, k0_dim, k1_dim,
                                           v_dim, rope_dims, int(traditional), theta, rows, offset, capacity, _addr(cache_k),
                                           _addr(cache_v), _addr(stream)))


def qkv_rope_store_decode(q, k, v, q_norm, k_norm, n_heads, n_kv, head_dim, rope_dims, theta, eps, d_offset,
                          offset, capacity, cache_k, cache_v, stream=None):
    check(lib.fk_qkv_rope_store_decode(_addr(q), _addr(k), _addr(v), _addr(q_norm), _addr(k_norm), n_heads, n_kv, head_dim,
                                       rope_dims, theta, eps, _addr(d_offset), offset, capacity, _addr(cache_k),
                                       _addr(cache_v), _addr(stream)))


def sdpa_workspace_bytes(n_heads, n_kv, qk_dim, v_dim, max_len):
    pb, cb = C.c_size_t(), C.c_size_t()
    check(lib.fk_sdpa_workspace_bytes(C.c_uint32(n_heads), C.c_uint32(n_kv), C.c_uint32(qk_dim), C.c_uint32(v_dim),
                                      C.c_uint32(max_len), C.byref(pb), C.byref(cb)))
    return int(pb.value), int(cb.value)


def sdpa_decode(q, cache_k, cache_v, out, d_kv_len, kv_len, max_len, n_heads, n_kv, qk_dim, v_dim, capacity,
                scale, partials, counters, stream=None):
    check(lib.fk_sdpa_decode(_addr(q), _addr(cache_k), _addr(cache_v), _addr(out), _addr(d_kv_len), kv_len, max_len, n_heads,
                             n_kv, qk_dim, v_dim, capacity, scale, _addr(partials), _addr(counters), _addr(stream)))


def sdpa_decode_static(q, cache_k, cache_v, out, d_kv_len, kv_len, max_len, n_heads, n_kv, qk_dim, v_dim, capacity,
                       scale, stream=None):
    """fk_sdpa_decode with the split-K workspace in the library's static device array: allocates nothing."""
    check(lib.fk_sdpa_decode_static(_addr(q), _addr(cache_k), _addr(cache_v), _addr(out), _addr(d_kv_len), kv_len, max_len,
                                    n_heads, n_kv, qk_dim, v_dim, capacity, scale, _addr(stream)))


class _KvQuantCache(C.Structure):
    _fields_ = [("packed", C.c_void_p), ("scales", C.c_void_p), ("biases", C.c_void_p)]


class QuantKvCache:
    """One K or V cache in the quantised layout, resident in HBM."""

    def __init__(self, n_kv: int, capacity: int, dim: int, bits: int, group: int = 64, zero: bool = True):
        self.n_kv, self.capacity, self.dim, self.bits, self.group = n_kv, capacity, dim, bits, group
        alloc = zeros if zero else DeviceBuffer
        self.packed = alloc(n_kv * capacity * dim * bits // 8)
        self.scales = alloc(n_kv * capacity * (dim // group) * 2)
        self.biases = alloc(n_kv * capacity * (dim // group) * 2)

    @property
    def c(self) -> _KvQuantCache:
        return _KvQuantCache(self.packed.ptr, self.scales.ptr, self.biases.ptr)

    @property
    def nbytes(self) -> int:
        return self.packed.nbytes + self.scales.nbytes + self.biases.nbytes


def kv_cache_dequant(cache: "QuantKvCache", rows: int, out, out_capacity: int, stream=None):
    """Rows [0, rows) of a quantised cache as bf16 [n_kv, out_capacity, dim]."""
    check(lib.fk_kv_cache_dequant(cache.c, cache.n_kv, cache.dim, cache.capacity, cache.bits, cache.group, rows, _addr(out),
                                  out_capacity, _addr(stream)))


def kv_cache_store_quant(k, v, k_norm, n_kv, head_dim, rope_dims, theta, eps, d_offset, offset, rows, K: QuantKvCache,
                         V: QuantKvCache, stream=None):
    check(lib.fk_kv_cache_store_quant(_addr(k), _addr(v), _addr(k_norm), n_kv, head_dim, rope_dims, theta, eps,
                                      _addr(d_offset), offset, rows, K.capacity, K.bits, K.group, K.c, V.c, _addr(stream)))


def sdpa_decode_quant(q, K: QuantKvCache, V: QuantKvCache, out, d_kv_len, kv_len, max_len, rows, n_heads, scale,
                      partials, counters, stream=None):
    check(lib.fk_sdpa_decode_quant(_addr(q), K.c, V.c, _addr(out), _addr(d_kv_len), kv_len, max_len, rows, n_heads, K.n_kv,
                                   K.dim, V.dim, K.capacity, K.bits, K.group, scale, _addr(partials), _addr(counters),
                                   _addr(stream)))


def rmsnorm_rows(x, w, eps, rows, hidden, y, stream=None):
    check(lib.fk_rmsnorm_rows(_addr(x), _addr(w), eps, rows, hidden, _addr(y), _addr(stream)))


def embed_lookup_rows(E, d_tokens, rows, out_scale, x, stream=None):
    check(lib.fk_embed_lookup_rows(_w(E), _addr(d_tokens), rows, out_scale, _addr(x), _addr(stream)))


def qkv_rope_store_rows(q, k, v, q_norm, k_norm, n_heads, n_kv, head_dim, rope_dims, theta, eps, rows, offset,
                        capacity, cache_k, cache_v, stream=None, rope_tab=None):
    check(lib.fk_qkv_rope_store_rows(_addr(q), _addr(k), _addr(v), _addr(q_norm), _addr(k_norm), n_heads, n_kv, head_dim,
                                     rope_dims, theta, eps, rows, offset, capacity, _addr(cache_k), _addr(cache_v),
                                     _addr(rope_tab), _addr(stream)))


def rope_table_rows(tab, rope_dims, theta, offset, rows, stream=None):
    """(cos, sin) of every rotary pair at positions offset .. offset + rows - 1, [rows][rope_dims/2][2] fp32."""
    check(lib.fk_rope_table_rows(_addr(tab), rope_dims, theta, offset, rows, _addr(stream)))


def sdpa_decode_rows(q, cache_k, cache_v, out, rows, kv_len, n_heads, n_kv, qk_dim, v_dim, capacity, scale, partials,
                     counters, stream=None):
    check(lib.fk_sdpa_decode_rows(_addr(q), _addr(cache_k), _addr(cache_v), _addr(out), rows, kv_len, n_heads, n_kv, qk_dim,
                                  v_dim, capacity, scale, _addr(partials), _addr(counters), _addr(stream)))


def sdpa_prefill(q, cache_k, cache_v, out, rows, kv_len, n_heads, n_kv, head_dim, capacity, scale, stream=None):
    """Causal attention of a group of rows on the matrix cores; kv_len counts the group's rows."""
    check(lib.fk_sdpa_prefill(_addr(q), _addr(cache_k), _addr(cache_v), _addr(out), rows, kv_len, n_heads, n_kv, head_dim,
                              capacity, scale, _addr(stream)))


class PromptLayer(C.Structure):
    """fk_prompt_layer."""
    _fields_ = ([(n, Weight) for n in ("q", "k", "v", "o", "gate", "up", "down")] +
                [(n, C.c_void_p) for n in ("input_norm", "post_norm", "q_norm", "k_norm", "q_bias", "k_bias", "v_bias", "cache_k", "cache_v")] +
                [("cache_kq", _KvQuantCache), ("cache_vq", _KvQuantCache)])


class PromptModel(C.Structure):
    """fk_prompt_model."""
    _fields_ = ([("embed", Weight), ("head", Weight), ("final_norm", C.c_void_p), ("layers", C.POINTER(PromptLayer))] +
                [(n, C.c_uint32) for n in ("n_layers", "hidden", "n_heads", "n_kv", "head_dim", "inter", "vocab", "capacity")] +
                [(n, C.c_float) for n in ("eps", "theta", "embed_scale")] + [("swiglu_variant", C.c_int)] +
                [(n, C.c_uint32) for n in ("kv_bits", "kv_group")] +
                [(n, C.c_void_p) for n in ("tokens", "x", "x2", "xn", "q", "k", "v", "att", "mid", "workspace", "rope_tab", "partials",
                                           "counters", "k_rows", "v_rows", "logits", "token", "argmax_workspace", "step_counter")])


def prompt_run(model: PromptModel, tokens, start: int, rows_per_pass: int, stream=None) -> int:
    """A prompt through the dense decoder (fk_prompt_run); returns the greedy next token."""
    t = np.ascontiguousarray(tokens, dtype=np.uint32)
    nxt = C.c_uint32()
    check(lib.fk_prompt_run(C.byref(model), t.ctypes.data_as(C.c_void_p), C.c_uint32(t.size), C.c_uint32(start),
                            C.c_uint32(rows_per_pass), C.byref(nxt), _ptr(stream)))
    return nxt.value


def gemm_library_available() -> bool:
    return bool(lib.fk_gemm_library_available())


def dequantize_bf16(W: DeviceWeight, stream=None) -> DeviceWeight:
    """The bf16 copy of a quantised matrix (fk_dequantize_bf16) as a bits-16 DeviceWeight."""
    D = DeviceWeight.__new__(DeviceWeight)
    D.n, D.k, D.bits, D.group, D.scales, D.biases = W.n, W.k, 16, 0, None, None
    D.w = DeviceBuffer(W.n * W.k * 2)
    check(lib.fk_dequantize_bf16(_w(W), _addr(D.w), _addr(stream)))
    return D


GEMM_LIBRARY_ROWS_DEFAULT = 0xFFFFFFFF  # the library's own choice (from 1024 rows, pairs as include/fusekit_hip.h says)


def set_gemm_library_rows(rows: int):
    """Row count from which qgemm / qgemm_swiglu take the dequantise + library-GEMM route (0: never)."""
    check(lib.fk_set_gemm_library_rows(rows))


def embed_lookup_decode(E, d_token, token, out_scale, x, stream=None):
    check(lib.fk_embed_lookup_decode(_w(E), _addr(d_token), token, out_scale, _addr(x), _addr(stream)))


ARGMAX_WORKSPACE_BYTES = 1288


def argmax_logits_decode(logits, n, next_token, history, hist_counter, hist_capacity, workspace, stream=None):
    check(lib.fk_argmax_logits_decode(_addr(logits), n, _addr(next_token), _addr(history), _addr(hist_counter), hist_capacity,
                                      _addr(workspace), _addr(stream)))


def step_init(step_counter, offset, kv_len, stream=None):
    check(lib.fk_step_init(_addr(step_counter), _addr(offset), _addr(kv_len), _addr(stream)))


def step_init_rope(step_counter, offset, kv_len, rope_tab, rope_dims, theta, stream=None):
    check(lib.fk_step_init_rope(_addr(step_counter), _addr(offset), _addr(kv_len), _addr(rope_tab), rope_dims, theta,
                                _addr(stream)))


def rope_store_sdpa_decode(q, k, v, q_norm, k_norm, cache_k, cache_v, out, d_kv_len, kv_len, max_len, n_heads, n_kv,
                           head_dim, rope_dims, theta, eps, capacity, scale, rope_tab, partials, counters, stream=None):
    check(lib.fk_rope_store_sdpa_decode(_addr(q), _addr(k), _addr(v), _addr(q_norm), _addr(k_norm), _addr(cache_k),
                                        _addr(cache_v), _addr(out), _addr(d_kv_len), kv_len, max_len, n_heads, n_kv, head_dim,
                                        rope_dims, theta, eps, capacity, scale, _addr(rope_tab), _addr(partials),
                                        _addr(counters), _addr(stream)))


def xcd_layer_supported(hidden, inter, n_heads, n_kv, head_dim, capacity, bits, group) -> bool:
    """Can a layer of this shape run as two XCD-resident launches (fk_xcd_layer_supported)?"""
    return lib.fk_xcd_layer_supported(C.c_uint32(hidden), C.c_uint32(inter), C.c_uint32(n_heads), C.c_uint32(n_kv),
                                      C.c_uint32(head_dim), C.c_uint32(capacity), C.c_uint32(bits), C.c_uint32(group)) == 0


def xcd_workspace_bytes(n_heads, head_dim):
    """(bytes of the control block, bytes of the attention partial rows)."""
    a, b = C.c_size_t(), C.c_size_t()
    check(lib.fk_xcd_workspace_bytes(C.c_uint32(n_heads), C.c_uint32(head_dim), C.byref(a), C.byref(b)))
    return a.value, b.value


lib.fk_xcd_sum_row_bytes.restype = C.c_size_t


def xcd_sum_row_bytes(hidden: int) -> int:
    return int(lib.fk_xcd_sum_row_bytes(C.c_uint32(hidden)))


def xcd_moe_supported(hidden, inter, shared_inter, experts, top_k, bits, group) -> bool:
    """Can the expert block of a layer of this shape run as one XCD-resident launch (fk_xcd_moe_supported)?"""
    return lib.fk_xcd_moe_supported(C.c_uint32(hidden), C.c_uint32(inter), C.c_uint32(shared_inter), C.c_uint32(experts),
                                    C.c_uint32(top_k), C.c_uint32(bits), C.c_uint32(group)) == FK_OK


def xcd_mla_supported(hidden, n_heads, rank, rope_dim, nope_dim, v_dim, capacity, bits, group) -> bool:
    """Can the attention half of a layer with low-rank keys run as one XCD-resident launch (fk_xcd_mla_supported)?"""
    u = C.c_uint32
    return lib.fk_xcd_mla_supported(u(hidden), u(n_heads), u(rank), u(rope_dim), u(nope_dim), u(v_dim), u(capacity), u(bits),
                                    u(group)) == FK_OK


def xcd_mla_workspace_bytes(n_heads, rank, rope_dim, v_dim):
    """(bytes of the `kva` slot, bytes of the attention partial rows) of fusekit_xcd_mla_block."""
    a, b = C.c_size_t(), C.c_size_t()
    check(lib.fk_xcd_mla_workspace_bytes(C.c_uint32(n_heads), C.c_uint32(rank), C.c_uint32(rope_dim), C.c_uint32(v_dim),
                                         C.byref(a), C.byref(b)))
    return a.value, b.value


lib.fk_xcd_moe_scratch_bytes.restype = C.c_size_t


def xcd_moe_scratch_bytes(inter: int) -> int:
    return int(lib.fk_xcd_moe_scratch_bytes(C.c_uint32(inter)))


def xcd_kslice_meta(src: "DeviceBuffer", n: int, groups: int, stream=None) -> "DeviceBuffer":
    """The per-XCD re-laid-out copy of a scale or bias array [n, groups] (fk_xcd_kslice_meta)."""
    dst = DeviceBuffer(n * groups * 2)
    check(lib.fk_xcd_kslice_meta(_addr(src), n, groups, _addr(dst), _addr(stream)))
    return dst


def xcd_sum_index(hidden: int):
    """Index of element e of a hidden-wide vector inside a sum row (numpy array of hidden indices)."""
    import numpy as np
    e = np.arange(hidden, dtype=np.int64)
    t = e >> 3
    return ((((t >> 6) * 4 + ((e & 7) >> 1)) * 64 + (t & 63)) << 1) | (e & 1)


def xcd_check(workspace, stream=None) -> None:
    check(lib.fk_xcd_check(_addr(workspace), _addr(stream)))


def copy(dst, src, nbytes, stream=None):
    check(lib.fk_copy(_ptr(dst), _ptr(src), C.c_size_t(nbytes), _ptr(stream)))


def route_order(expert_idx, n_routes: int, n_experts: int, order, stream=None) -> None:
    """order[position] = route, the routes sorted by expert index, stable (fk_route_order)."""
    check(lib.fk_route_order(_addr(expert_idx), n_routes, n_experts, _addr(order), _addr(stream)))


lib.fk_read_reduce_out_bytes.restype = C.c_size_t


def read_reduce_out_bytes() -> int:
    return int(lib.fk_read_reduce_out_bytes())


def read_reduce(src, nbytes, out, stream=None):
    """XOR of nbytes read with plain 16-byte loads, one word per workgroup into `out` (fk_read_reduce)."""
    check(lib.fk_read_reduce(_ptr(src), C.c_size_t(nbytes), _ptr(out), C.c_size_t(out.nbytes), _ptr(stream)))


def fill_u32(buf, value, count, stream=None):
    check(lib.fk_fill_u32(_ptr(buf), C.c_uint32(value), C.c_size_t(count), _ptr(stream)))


def zeros(nbytes: int) -> DeviceBuffer:
    b = DeviceBuffer(nbytes)
    b.upload(np.zeros(nbytes, dtype=np.uint8))
    return b


def set_gemv_policy(rows_per_tile: int = 0, grid_blocks: int = 0) -> None:
    check(lib.fk_set_gemv_policy(rows_per_tile, grid_blocks))


def gemv_form(n: int, k: int, bits: int, group: int = 64) -> int:
    """1 when a plain GEMV over an [n, k] matrix runs the row-group kernel form, 0 for the flat stream."""
    return int(lib.fk_gemv_form(C.c_uint32(n), C.c_uint32(k), C.c_uint32(bits), C.c_uint32(group)))


def set_qgemm_wide(enabled: bool) -> None:
    check(lib.fk_set_qgemm_wide(1 if enabled else 0))


def set_gemv_flat_only(flat_only: bool) -> None:
    check(lib.fk_set_gemv_flat_only(1 if flat_only else 0))


def sync(stream=None) -> None:
    check(lib.fk_stream_sync(_addr(stream)))


class Event:
    def __init__(self):
        p = C.c_void_p()
        check(lib.fk_event_create(C.byref(p)))
        self.ptr = p.value

    def record(self, stream=None) -> None:
        check(lib.fk_event_record(C.c_void_p(self.ptr), _ptr(stream)))

    def elapsed_ms_until(self, stop: "Event") -> float:
        ms = C.c_float()
        check(lib.fk_event_elapsed_ms(C.c_void_p(self.ptr), C.c_void_p(stop.ptr), C.byref(ms)))
        return float(ms.value)

    def __del__(self):
        try:
            if self.ptr:
                lib.fk_event_destroy(C.c_void_p(self.ptr))
        except Exception:
            pass


# Argument types of the operators, declared once: ctypes converts plain numbers and addresses in C, and a call does not build an
# object for each (rmsnorm + q / k / v, thirteen arguments: 6.4 us a call with the objects, 5.4 without; a launch
# alone takes 4.0).  p an address, W an fk_weight, Q a quantised cache, u / i / f a 32-bit number.
_SIGNATURES = {
    "fk_qgemv": "Wpppp", "fk_linear_residual": "Wppppp", "fk_rmsnorm_qkv": "ppfWWWppppppp",
    "fk_gateup_swiglu_rows": "pupfWWipp", "fk_rmsnorm_qkv_rows": "puupfWWWpupupup", "fk_gateup_swiglu": "ppfWWipp",
    "fk_routed_qmv_swiglu": "puWWupppupp", "fk_routed_qmv_swiglu_shared": "pWWuppupWWpp",
    "fk_routed_qmv_swiglu_routing": "pWWuppuipppWWpp", "fk_routed_qmv_reduce": "puWuppppWpuuppp",
    "fk_routed_qmv_swiglu_ordered": "puWWupppuppp", "fk_routed_qmv_reduce_ordered": "puWuppppWpuupppp", "fk_qgemm": "Wpuppppp",
    "fk_qgemm_swiglu": "WWpuippp", "fk_final_rmsnorm_lm_head": "ppfWpp", "fk_final_rmsnorm_lm_head_argmax": "ppfWppppupp",
    "fk_rope_q_decode": "ppuuuffpup", "fk_rope_kv_cache_store_decode": "pppuuuuffpupuuppp",
    "fk_kv_cache_store_split_decode": "puuupupupuuuuuuifpupuuppp", "fk_split_store_sdpa_decode": "puuupupupuuuuifpppppuuufppp",
    "fk_softmax_topk_route": "ppiuuuppp", "fk_moe_router": "ppfppuuupppppup",
    "fk_kv_cache_store_split_rows": "puuupuupuupuuuuuuuifuuuppp", "fk_qkv_rope_store_decode": "pppppuuuuffpuuppp",
    "fk_sdpa_decode": "pppppuuuuuuufppp", "fk_sdpa_decode_static": "pppppuuuuuuufp", "fk_kv_cache_dequant": "Quuuuuupup",
    "fk_kv_cache_store_quant": "pppuuuffpuuuuuQQp", "fk_sdpa_decode_quant": "pQQppuuuuuuuuuufppp", "fk_rmsnorm_rows": "ppfuupp",
    "fk_embed_lookup_rows": "Wpufpp", "fk_qkv_rope_store_rows": "pppppuuuuffuuupppp", "fk_rope_table_rows": "pufuup",
    "fk_sdpa_decode_rows": "ppppuuuuuuufppp", "fk_sdpa_prefill": "ppppuuuuuufp", "fk_dequantize_bf16": "Wpp",
    "fk_set_gemm_library_rows": "u", "fk_embed_lookup_decode": "Wpufpp", "fk_argmax_logits_decode": "pupppupp",
    "fk_step_init": "pppp", "fk_step_init_rope": "ppppufp", "fk_rope_store_sdpa_decode": "pppppppppuuuuuuffufpppp",
    "fk_xcd_kslice_meta": "puupp", "fk_xcd_check": "pp", "fk_route_order": "puupp", "fk_set_gemv_policy": "uu",
    "fk_set_qgemm_wide": "i", "fk_set_gemv_flat_only": "i", "fk_stream_sync": "p",
}

_TYPES = {"p": C.c_void_p, "W": C.POINTER(Weight), "Q": C.POINTER(_KvQuantCache), "u": C.c_uint32, "i": C.c_int, "f": C.c_float}
for _name, _signature in _SIGNATURES.items():
    getattr(lib, _name).argtypes = [_TYPES[_t] for _t in _signature]
