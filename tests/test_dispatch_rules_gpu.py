"""The rules by which a launch picks its kernel form or tile, at the sizes where they change over (against the oracle)."""
import numpy as np
import pytest

import oracle
from helpers import make_qweight, normal_bf16, rel_l2, to_device
from test_attention_gpu import _sdpa_case

pytestmark = pytest.mark.gpu


def test_gemv_tiling_is_looked_up_by_shape_and_policy(fk):
    """Shapes and tile policies in turn, each twice: what one call looked up is never another's."""
    cases = [(n, 64 * g, rows) for n, g, rows in ((896, 14, 0), (897, 14, 0), (896, 76, 0), (896, 14, 3), (64, 14, 0))]
    kept = [(W := make_qweight(7 + i, n, k, 4), to_device(fk, W), normal_bf16(i, k), fk.DeviceBuffer(2 * n), rows)
            for i, (n, k, rows) in enumerate(cases)]
    try:
        for _ in range(2):
            for W, dW, x, y, rows in kept:
                fk.set_gemv_policy(rows, 0)
                fk.qgemv(dW, fk.DeviceBuffer.from_numpy(x), None, y)
                assert rel_l2(y.to_numpy(np.uint16), oracle.linear_acc(W, x)) <= 5e-3
    finally:
        fk.set_gemv_policy(0, 0)


@pytest.mark.parametrize("heads,length", [((14, 2, 64), 4096), ((14, 2, 64), 4097), ((10, 2, 64), 130), ((16, 2, 128), 4200)])
def test_attention_tiles_of_groups_of_more_than_four_heads(fk, heads, length):
    n_heads, n_kv, dim = heads
    _sdpa_case(fk, n_heads, n_kv, dim, dim, length, length + 3, seed=length)


@pytest.mark.parametrize("bits,group", [(4, 64), (8, 64), (4, 128), (16, 64)])
@pytest.mark.parametrize("m,n,k", [(1, 17, 64), (15, 333, 896), (17, 4112, 128), (33, 4100, 384), (48, 16, 2048), (64, 40, 4864), (49, 8200, 128)])
def test_matmul_of_up_to_64_rows(fk, bits, group, m, n, k):
    """Row tiles, weight-row tiles, waves without a group, both block forms; bias and residual; against the oracle."""
    if k % group:
        pytest.skip("K is whole groups")
    W = make_qweight(11 + bits, n, k, bits, group=group)
    x, bias, res = normal_bf16(12, (m, k)), normal_bf16(13, n), normal_bf16(14, (m, n))
    y, ws = fk.DeviceBuffer(2 * m * n), fk.DeviceBuffer(fk.qgemm_workspace_bytes(m, n, k, 0 if bits == 16 else group))
    up = fk.DeviceBuffer.from_numpy
    fk.qgemm(to_device(fk, W), up(x), m, up(bias), up(res), y, ws)
    got = y.to_numpy(np.uint16, (m, n))
    for r in sorted({0, m // 2, m - 1}):
        want = oracle.linear_acc(W, x[r]) + oracle.bf16_to_f32(bias) + oracle.bf16_to_f32(res[r])
        assert rel_l2(got[r], want) <= 4e-3


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("m", [12, 37, 64])
def test_pair_and_fan_out_of_up_to_64_rows(fk, bits, m):
    k, inter, ns = 896, 1000, (896, 130, 128)
    x = normal_bf16(21, (m, k))
    up = fk.DeviceBuffer.from_numpy
    g, u = make_qweight(22, inter, k, bits), make_qweight(23, inter, k, bits)
    out, ws = fk.DeviceBuffer(2 * m * inter), fk.DeviceBuffer(2 * fk.qgemm_workspace_bytes(m, 2048, k, 0 if bits == 16 else 64))
    fk.qgemm_swiglu(to_device(fk, g), to_device(fk, u), up(x), m, 1, out, ws)
    Ws, biases = [make_qweight(24 + i, n, k, bits) for i, n in enumerate(ns)], [normal_bf16(30 + i, n) for i, n in enumerate(ns)]
    ys = [fk.DeviceBuffer(2 * m * n) for n in ns]
    fk.qgemm_fanout([to_device(fk, W) for W in Ws], up(x), m, [up(b) for b in biases], ys, ws)
    for r in (0, m - 1):
        want = oracle.gateup_swiglu(x[r], None, 0.0, g, u, 1)
        assert rel_l2(out.to_numpy(np.uint16, (m, inter))[r], oracle.bf16_to_f32(want)) <= 1e-2
        for W, b, y in zip(Ws, biases, ys):
            assert rel_l2(y.to_numpy(np.uint16, (m, W.n))[r], oracle.linear_acc(W, x[r]) + oracle.bf16_to_f32(b)) <= 4e-3


@pytest.mark.parametrize("rows,hidden", [(1, 8), (3, 2048), (5, 2056), (2, 4104), (2, 12288), (2, 16392), (2, 100)])
def test_norm_of_rows_in_16_byte_pieces(fk, rows, hidden):
    """One, two, four and eight pieces per thread, ragged last pieces, and the widths the strided form keeps."""
    x, w = normal_bf16(41, (rows, hidden)), normal_bf16(42, hidden, 0.1, 1.0)
    y = fk.DeviceBuffer(2 * rows * hidden)
    fk.rmsnorm_rows(fk.DeviceBuffer.from_numpy(x), fk.DeviceBuffer.from_numpy(w), 1e-6, rows, hidden, y)
    got = y.to_numpy(np.uint16, (rows, hidden))
    for r in range(rows):
        ref = oracle.rmsnorm(x[r], w, 1e-6)
        assert np.mean(got[r] != ref) <= 0.01 and rel_l2(got[r], oracle.bf16_to_f32(ref)) <= 1e-3


@pytest.mark.parametrize("kv_bits,bits,n", [(0, 4, 9), (0, 8, 40), (0, 16, 64), (0, 4, 65), (8, 4, 40), (8, 16, 20)])
def test_prompt_pass_is_the_single_token_pass(fk, kv_bits, bits, n):
    """A prompt in one pass and token by token: the same greedy token, close logits (the norms inside the projections, the
    forms up to 64 rows, the kept summation orders of a quantised cache)."""
    from fusekit_amd.decoder import DecoderConfig, DecoderRuntime, DecoderWeights
    cfg = DecoderConfig(n_layers=2, hidden=512, n_heads=14, n_kv=2, head_dim=64, inter=1024, vocab=800, capacity=128, bits=bits,
                        kv_bits=kv_bits, qkv_bias=True)
    W = DecoderWeights.random_init(cfg, seed=3)
    a, b = DecoderRuntime(cfg, W), DecoderRuntime(cfg, W)
    prompt = np.random.default_rng(n).integers(0, 800, n).tolist()
    b.prefill(prompt)
    for _ in range(2):
        a.prefill_rows(prompt)
        assert rel_l2(a.logits.to_numpy(np.uint16), oracle.bf16_to_f32(b.logits.to_numpy(np.uint16))) <= 2e-2
        assert a.step_counter.to_numpy(np.uint32)[0] == n


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k", [(65, 4, 768), (128, 132, 896), (129, 1000, 1024), (300, 2052, 2048), (257, 8200, 896), (640, 96, 4864)])
def test_matmul_from_65_rows(fk, bits, m, n, k):
    """Tiles of 128 and 256 activation rows, one to eight k splits, ragged rows and weight rows: one matrix with bias and
    residual, a gate / up pair, a fan-out of three."""
    x, bias, res = normal_bf16(41, (m, k)), normal_bf16(42, n), normal_bf16(43, (m, n))
    Ws = [make_qweight(44 + i, n, k, bits) for i in range(3)]
    dW, up = [to_device(fk, W) for W in Ws], fk.DeviceBuffer.from_numpy
    dx, ws = up(x), fk.DeviceBuffer(2 * fk.qgemm_workspace_bytes(m, 3 * n, k))
    ys = [fk.DeviceBuffer(2 * m * n) for _ in range(5)]
    fk.qgemm(dW[0], dx, m, up(bias), up(res), ys[0], ws)
    fk.qgemm_swiglu(dW[0], dW[1], dx, m, 1, ys[1], ws)
    fk.qgemm_fanout(dW, dx, m, [None, up(bias), None], ys[2:], ws)
    acc = [oracle.qgemm_bf16w(W, x, None, want_acc=True)[1].astype(np.float64) for W in Ws]
    b, r = oracle.bf16_to_f32(bias).astype(np.float64), oracle.bf16_to_f32(res).astype(np.float64)
    g, u = (oracle.bf16_to_f32(oracle.f32_to_bf16(a.astype(np.float32))).astype(np.float64) for a in acc[:2])
    for y, want in zip(ys, (acc[0] + b + r, g / (1 + np.exp(-g)) * u, acc[0], acc[1] + b, acc[2])):
        assert rel_l2(y.to_numpy(np.uint16, (m, n)), want) <= 4e-3


@pytest.mark.parametrize("heads,qk_norm", [((8, 2, 128), True), ((4, 2, 64), True), ((14, 2, 64), False), ((2, 2, 128), False)])
@pytest.mark.parametrize("kv_bits", [4, 8])
def test_quantised_cache_rows_appended_inside_the_attention(fk, heads, qk_norm, kv_bits):
    """One launch for rotation, quantisation, append and attention leaves the bits of the three launches it replaces: one,
    two and four heads a tile and eight, the first position, range boundaries, several ranges."""
    from fusekit_amd.decoder import DecoderConfig, DecoderRuntime, DecoderWeights
    n_heads, n_kv, dim = heads
    cfg = dict(n_layers=2, hidden=256, n_heads=n_heads, n_kv=n_kv, head_dim=dim, inter=512, vocab=500, capacity=2304, kv_bits=kv_bits,
               qk_norm=qk_norm)
    W = DecoderWeights.random_init(DecoderConfig(**cfg), seed=5)
    a, b = (DecoderRuntime(DecoderConfig(**cfg, fuse_attention=f), W) for f in (True, False))
    assert len(a.tasks) == len(b.tasks) - 2 * cfg["n_layers"]
    bufs = lambda rt: [x for c in rt.cache_k + rt.cache_v for x in (c.packed, c.scales, c.biases)]
    for pos in (0, 1, 31, 63, 64, 130, 700, 2303):
        for rt in (a, b):
            rt.d.decode_host_loop(rt.graph, rt.uniforms, pos, [7 + pos % 400])
        assert np.array_equal(a.logits.to_numpy(np.uint16), b.logits.to_numpy(np.uint16)), pos
        for x, y in zip(bufs(a), bufs(b)):
            assert np.array_equal(x.to_numpy(np.uint8), y.to_numpy(np.uint8)), pos


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m", [65, 300, 1024])
def test_swiglu_of_every_finite_gate(fk, bits, m):
    """All finite bf16 gates (and, in a row that doubles them, infinite ones) through the pair's one-launch form: the finite
    values against 64 bits, infinities and NaN as the form of up to 64 rows (expf and a divide) gives them."""
    n, k = 4096, 1024
    rng = np.random.default_rng(m)
    zeros = np.zeros((n, k // 64), np.uint16)
    # a weight is T(0 code + bias): a row that is one in group j and zero elsewhere selects gate n, j and its factor u
    gate = rng.permutation(np.arange(65536, dtype=np.uint16)).reshape(n, k // 64)
    gate[(gate & 0x7F80) == 0x7F80] = 0x42B5                      # (infinities and NaN: another 90.5)
    factor = oracle.f32_to_bf16(rng.normal(0, 1, (n, k // 64)).astype(np.float32))
    codes = np.zeros((n, k * bits // 32), np.uint32)
    g, u = (to_device(fk, oracle.QWeight(codes, zeros, b, n, k, bits)) for b in (gate, factor))
    x = np.zeros((m, k), np.float32)
    x[np.arange(m), 64 * (np.arange(m) % 16) + 5] = np.where(np.arange(m) == m - 1, 2.0, 1.0)
    x = oracle.f32_to_bf16(x)
    def run(rows):
        out, ws = fk.DeviceBuffer(2 * len(rows) * n), fk.DeviceBuffer(2 * fk.qgemm_workspace_bytes(len(rows), n, k))
        fk.qgemm_swiglu(g, u, fk.DeviceBuffer.from_numpy(x[rows]), len(rows), 1, out, ws)
        return oracle.bf16_to_f32(out.to_numpy(np.uint16, (len(rows), n))).astype(np.float64)
    got, sel = run(np.arange(m)), [r % 16 for r in range(m)]
    with np.errstate(all="ignore"):
        scale = np.where(np.arange(m) == m - 1, 2.0, 1.0)[:, None]
        gv, uv = (oracle.bf16_to_f32(oracle.f32_to_bf16(oracle.bf16_to_f32(b).T[sel] * np.float32(scale))).astype(np.float64) for b in (gate, factor))
        want = gv / (1 + np.exp(-gv)) * uv
        # half a unit of bf16, a few of fp32; below -88.73 e^-g overflows and the result may be -0 u, at most 88.8 2^-128 u away
        off = np.abs(got - want) > (2.0 ** -8 + 2.0 ** -20) * np.abs(want) + 3e-37 * np.abs(uv) + 1e-40
    plain = np.isfinite(gv) & (np.abs(want) < 3.3e38)
    assert plain.mean() > 0.99 and not (off & plain).any(), (gv[off & plain][:8], got[off & plain][:8])
    assert np.isfinite(got[plain]).all()
    few = np.r_[0:63, m - 1]
    ref = run(few)
    assert np.isposinf(gv[m - 1]).any() and np.isneginf(gv[m - 1]).any()
    assert np.array_equal(np.isnan(got[few]), np.isnan(ref)) and np.array_equal(np.isinf(got[few]), np.isinf(ref))


class _At:
    """A host array on the device at an address `off` bytes past a 256-byte boundary."""

    def __init__(self, fk, a, off):
        a = np.ascontiguousarray(a)
        self.nbytes, self.buf = a.nbytes, fk.DeviceBuffer(a.nbytes + 256)
        self.buf.upload(a.view(np.uint8).reshape(-1), off)
        self.ptr = self.buf.ptr + off


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("m", [1, 2, 9, 16, 37, 64])
def test_up_to_64_rows_at_any_address(fk, bits, m):
    """Activations, codes, scales and outputs on their element's alignment only: the bits of the aligned call."""
    k, n = 896, 200
    group = 0 if bits == 16 else 64
    Ws = [make_qweight(70 + i, n, k, bits) for i in range(3)]
    x, bias, res = normal_bf16(73, (m, k)), normal_bf16(74, n), normal_bf16(75, (m, n))
    ws = fk.DeviceBuffer(2 * fk.qgemm_workspace_bytes(m, 3 * n, k, group))
    def run(off, code_off):
        at = lambda a, o=off: _At(fk, a, o)
        dW = [to_device(fk, W) for W in Ws]
        for W, d in zip(Ws, dW):
            d.w = at(W.w, off if bits == 16 else code_off)
            if bits != 16:
                d.scales, d.biases = at(W.scales), at(W.biases)
        dx, db, dr = at(x), at(bias), at(res)
        ys = [at(np.zeros((m, n), np.uint16)) for _ in range(5)]
        fk.qgemm(dW[0], dx.ptr, m, db.ptr, dr.ptr, ys[0].ptr, ws)
        fk.qgemm_swiglu(dW[0], dW[1], dx.ptr, m, 1, ys[1].ptr, ws)
        fk.qgemm_fanout(dW, dx.ptr, m, [None, db.ptr, None], [y.ptr for y in ys[2:]], ws)
        fk.sync()
        return [y.buf.to_numpy(np.uint16, (m, n), off) for y in ys]
    want = run(0, 0)
    for got in (run(2, 4), run(8, 8)):
        assert all(np.array_equal(g, w) for g, w in zip(got, want))
    ref = oracle.linear_acc(Ws[0], x[m - 1]) + oracle.bf16_to_f32(bias) + oracle.bf16_to_f32(res[m - 1])
    assert rel_l2(want[0][m - 1], ref) <= 4e-3


def test_prompt_with_norm_weights_at_any_address(fk):
    from fusekit_amd.decoder import DecoderConfig, DecoderRuntime, DecoderWeights
    cfg = DecoderConfig(n_layers=2, hidden=512, n_heads=14, n_kv=2, head_dim=64, inter=1024, vocab=800, capacity=128, bits=4, qkv_bias=True)
    W = DecoderWeights.random_init(cfg, seed=3)
    rt = DecoderRuntime(cfg, W)
    prompt = np.random.default_rng(9).integers(0, 800, 9).tolist()
    rt.prefill_rows(prompt)
    want = oracle.bf16_to_f32(rt.logits.to_numpy(np.uint16))
    kept = dict(W.vecs)
    for name in kept:
        if "layernorm" in name:
            W.vecs[name] = _At(fk, kept[name].to_numpy(np.uint16), 2)
    other = DecoderRuntime(cfg, W)
    other.prefill_rows(prompt)
    assert rel_l2(other.logits.to_numpy(np.uint16), want) <= 2e-2   # (the norm in a launch of its own: sums in another order)


@pytest.mark.parametrize("bits", [4, 16])
def test_two_shapes_of_one_kernel_beyond_48_kilobytes_in_turn(fk, bits):
    """Each launch is allowed the LDS it needs, whichever shape was planned before it."""
    kept = [(W := make_qweight(90 + i, 40, k, bits), to_device(fk, W), normal_bf16(91 + i, k), fk.DeviceBuffer(80))
            for i, k in enumerate((40960, 25600, 32768))]
    for W, dW, x, y in kept + kept[:2] + kept[::-1]:
        fk.qgemv(dW, fk.DeviceBuffer.from_numpy(x), None, y)
        assert rel_l2(y.to_numpy(np.uint16), oracle.linear_acc(W, x)) <= 5e-3


def test_a_library_threshold_that_is_set_holds_for_pairs(fk):
    """Every count that a caller sets, 1024 among them, sends pairs from there on to the library route; the default never does."""
    m, hidden, inter = 1024, 896, 1216
    Wg, Wu = make_qweight(76, inter, hidden, 4), make_qweight(77, inter, hidden, 4)
    x, dg, du = fk.DeviceBuffer.from_numpy(normal_bf16(78, (m, hidden))), to_device(fk, Wg), to_device(fk, Wu)
    def run(rows):
        fk.set_gemm_library_rows(rows)
        out, ws = fk.DeviceBuffer(2 * m * inter), fk.DeviceBuffer(2 * fk.qgemm_workspace_bytes(m, inter, hidden, 64))
        fk.qgemm_swiglu(dg, du, x, m, 1, out, ws)
        return out.to_numpy(np.uint16)
    try:
        fused, library = run(0), run(1023)
        assert not np.array_equal(fused, library)   # (sums in another order: how the routes are told apart)
        assert np.array_equal(run(1024), library) and np.array_equal(run(1025), fused)
    finally:
        default = run(fk.GEMM_LIBRARY_ROWS_DEFAULT)
    assert np.array_equal(default, fused)


@pytest.mark.parametrize("bits,group", [(4, 64), (8, 128), (16, 0)])
@pytest.mark.parametrize("m", [1, 12, 33, 64])
def test_up_to_64_rows_by_the_routes_of_quantised_caches(fk, bits, group, m):
    """Split k and a second kernel (dense bf16: the library), one matrix, a pair and a fan-out: another kernel, the same values."""
    k, n = 2560, 320
    Ws = [make_qweight(70 + i, n, k, bits, group=group or 64) for i in range(3)]
    x, bias, res = normal_bf16(73, (m, k)), normal_bf16(74, n), normal_bf16(75, (m, n))
    dW, up = [to_device(fk, W) for W in Ws], fk.DeviceBuffer.from_numpy
    def run(wide):
        ws, ys = fk.DeviceBuffer(2 * fk.qgemm_workspace_bytes(m, 3 * n, k, group)), [fk.DeviceBuffer(2 * m * n) for _ in range(5)]
        fk.set_qgemm_wide(wide)
        try:
            fk.qgemm(dW[0], up(x), m, up(bias), up(res), ys[0], ws)
            fk.qgemm_swiglu(dW[0], dW[1], up(x), m, 1, ys[1], ws)
            fk.qgemm_fanout(dW, up(x), m, [None, up(bias), None], ys[2:], ws)
        finally:
            fk.set_qgemm_wide(True)
        return [y.to_numpy(np.uint16, (m, n)) for y in ys]
    one, other = run(True), run(False)
    # sums in another order are how the kernels are told apart (a bf16 result flips about once in a thousand)
    assert m == 1 or any(not np.array_equal(a, b) for a, b in zip(one, other))
    acc = [np.stack([oracle.linear_acc(W, r) for r in x]).astype(np.float64) for W in Ws]
    b, r = oracle.bf16_to_f32(bias).astype(np.float64), oracle.bf16_to_f32(res).astype(np.float64)
    g, u = (oracle.bf16_to_f32(oracle.f32_to_bf16(a.astype(np.float32))).astype(np.float64) for a in acc[:2])
    for a, o, want in zip(one, other, (acc[0] + b + r, g / (1 + np.exp(-g)) * u, acc[0], acc[1] + b, acc[2])):
        assert rel_l2(a, want) <= 4e-3 and rel_l2(o, want) <= 4e-3
