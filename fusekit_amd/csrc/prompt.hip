// A prompt through the dense decoder, several rows per pass: the launches of prefill variants (the reference dispatches them
// from Python, python/fusekit_runtime/__init__.py:4782-4900; variants src/commands/patch.rs:112-150) walked natively.
//
// A pass is some ten launches per layer.  Called one by one through the operator entry points from Python each costs 7..10 us
// of host time, more than a short prompt's kernels run for; from here a launch costs what the runtime takes (3.7 us), so that
// the GPU is what a pass waits for.  37 tokens of the 0.5B-class model, whole call: 1378 us from Python, 1055 from here
// with the norms inside the projections (two launches per layer fewer); of 512 tokens of the 4B-class model 7279 us with the
// norms in launches of their own, 7046 with them in the launches that add split sums up.
#include <math.h>

#include "fk_host.hpp"

namespace fk {
namespace {

// Whether a projection of N outputs takes the form of up to 64 rows AND the RMSNorm ahead of it: the form normalises on the
// way in (with the sums of squares that the launch which wrote the rows left), but every block does so for all rows, about
// 0.4 us per million values it normalises, where the norm as a launch of its own costs some 3.5 us.  37 rows of K = 896:
// 1152 outputs (2.4 million) 5.4 us against 4.1 + 4.1, a 4864 pair (10 million) 15.2 against 10.1 + 4.1; 50 rows of
// K = 2560, a 9728 pair (78 million) 54 against 30 + 5.
// (Rows and norm weights that are not 16-byte aligned take the norm's own launch.)
bool takes_norm(const fk_weight& W, uint32_t rows, uint32_t n_total, const uint16_t* x, const uint16_t* norm_w) {
    return qgemm_takes_rows(rows, W.bits, W.group, W.k) && (uint64_t)rows * W.k * ((n_total + 15u) / 16u) < 8000000ull &&
           (((uintptr_t)x | (uintptr_t)norm_w) & 15u) == 0;
}

fk_status run_rows(const RowsRequest& rq, hipStream_t s) {
    Launch l;
    FK_TRY(plan_qgemm_rows(rq, &l));
    return run_launch(l, s);
}

// Passes into a QUANTISED cache keep older kernels, whose sums are added in another order than those of the forms above: a key
// that differs in its last bit can turn the sign of its group's scale (MLX's rule takes it from the end of the range that is
// larger in magnitude) and shift the group's codes, so the same prompt would fill a cache with other bytes than before.  From 11
// rows: split-k sums up to 64 rows (dense bf16 weights: the library GEMM), beyond, the tiles of qgemm.hip and the library
// (kept_order of run_qgemm); at any row count the norm in a launch of its own, strided, and the older attention.  Passes of up to
// 10 rows take the one-launch matmul (what they took before is gone), so it is longer passes only that fill a cache with the
// bytes they always did.  The same prompt token by token differs in such bits either way.  What the newer kernels would give
// these passes has not been measured.
fk_status norm_rows(const fk_prompt_model& m, const uint16_t* x, const uint16_t* w, uint32_t rows, hipStream_t s) {
    Launch l;
    FK_TRY(plan_rmsnorm_rows(x, w, m.eps, rows, m.hidden, m.xn, &l, m.kv_bits != 0));
    return run_launch(l, s);
}
bool kept_order(const fk_prompt_model& m, const fk_weight& W, uint32_t rows) {
    return m.kv_bits != 0 && rows <= 64 && (W.bits == 16 ? gemm_library_available() : rows > 10);
}
fk_status matmul(const fk_prompt_model& m, const fk_weight& W, const uint16_t* x, uint32_t rows, const uint16_t* bias, const uint16_t* res,
                 uint16_t* y, hipStream_t s, RowsNorm* norm = nullptr) {
    if (!kept_order(m, W, rows)) return run_qgemm(&W, x, rows, bias, res, y, m.workspace, m.kv_bits != 0, s, norm);
    if (W.bits == 16) return run_qgemm_library(&W, nullptr, x, rows, bias, res, 0, y, m.workspace, s);
    Launch main, reduce;
    FK_TRY(plan_qgemm(&W, x, rows, bias, res, y, m.workspace, &main, &reduce, true));
    FK_TRY(run_launch(main, s));
    return run_launch(reduce, s);
}

// What the launch that wrote a projection's input rows left in m.xn, free between a projection's launch and the next norm.
enum Left { LEFT_NOTHING, LEFT_SQUARES /* the rows' sums of squares */, LEFT_NORMED /* the normalised rows */ };

// One matrix with the residual; next_norm: the weights of the norm that its rows enter next, or null.
fk_status residual_rows(const fk_prompt_model& m, const fk_weight& W, const uint16_t* x, uint32_t rows, const uint16_t* res, uint16_t* y,
                        const uint16_t* next_norm, Left* left, hipStream_t s) {
    const bool ssq = m.kv_bits == 0 && qgemm_takes_rows(rows, W.bits, W.group, W.k) && W.n % 64u == 0 && ((uintptr_t)m.xn & 15u) == 0;
    *left = ssq ? LEFT_SQUARES : LEFT_NOTHING;
    if (!ssq) {
        RowsNorm norm{next_norm, m.xn, m.eps};
        FK_TRY(matmul(m, W, x, rows, nullptr, res, y, s, next_norm && m.xn && m.kv_bits == 0 ? &norm : nullptr));
        if (norm.done) *left = LEFT_NORMED;
        return FK_OK;
    }
    RowsRequest rq;
    rq.W[0] = &W; rq.x = x; rq.M = rows; rq.res = res; rq.y[0] = y;
    rq.ssq_out = reinterpret_cast<float*>(m.xn);
    return run_rows(rq, s);
}

fk_status layer_pass(const fk_prompt_model& m, const fk_prompt_layer& l, const fk_prompt_layer* next, Left* left, uint32_t rows,
                     uint32_t pos, fk_stream s) {
    const uint32_t dim = m.head_dim, len = pos + rows;
    const float scale = (float)(1.0 / sqrt((double)dim));
    const uint16_t* bias[3] = {l.q_bias, l.k_bias, l.v_bias};
    RopeArgs rope;
    memset(&rope, 0, sizeof(rope));
    rope.q = m.q; rope.k = m.k; rope.v = m.v; rope.q_norm = l.q_norm; rope.k_norm = l.k_norm;
    rope.n_q = m.n_heads; rope.n_kv = m.n_kv; rope.head_dim = rope.k_dim = rope.v_dim = rope.rope_dims = dim; rope.rope_on = 1;
    rope.offset_imm = pos; rope.capacity = m.capacity; rope.cache_k = l.cache_k; rope.cache_v = l.cache_v;
    rope.eps = m.eps; rope.base_log2 = (float)log2((double)m.theta); rope.rows = rows; rope.rope_tab = m.rope_tab;
    FanSums sums{};   // (one split, or another kernel: finished rows)
    const bool takes_sums = m.kv_bits == 0 && rope_takes_sums(rope) && l.q.n == m.n_heads * dim && l.k.n == m.n_kv * dim && l.v.n == l.k.n;
    const bool tiled = dim == 64 || dim == 128;
    if (m.kv_bits == 0 && *left != LEFT_NORMED && l.k.bits == l.q.bits && l.v.bits == l.q.bits && l.k.group == l.q.group && l.v.group == l.q.group &&
        takes_norm(l.q, rows, l.q.n + l.k.n + l.v.n, m.x, l.input_norm)) {
        RowsRequest rq;
        rq.W[0] = &l.q; rq.W[1] = &l.k; rq.W[2] = &l.v; rq.n_mats = 3;
        rq.x = m.x; rq.M = rows; rq.norm_w = l.input_norm; rq.eps = m.eps;
        if (*left == LEFT_SQUARES) rq.ssq_in = reinterpret_cast<const float*>(m.xn);   // (not where the rows come from the embedding)
        rq.bias[0] = l.q_bias; rq.bias[1] = l.k_bias; rq.bias[2] = l.v_bias;
        rq.y[0] = m.q; rq.y[1] = m.k; rq.y[2] = m.v;
        FK_TRY(run_rows(rq, (hipStream_t)s));
    } else {
        if (*left != LEFT_NORMED) FK_TRY(norm_rows(m, m.x, l.input_norm, rows, (hipStream_t)s));
        const fk_weight* W[3] = {&l.q, &l.k, &l.v};
        uint16_t* y[3] = {m.q, m.k, m.v};
        if (kept_order(m, l.q, rows))
            for (int i = 0; i < 3; ++i) FK_TRY(matmul(m, *W[i], m.xn, rows, bias[i], nullptr, y[i], (hipStream_t)s));
        else
            FK_TRY(run_qgemm_fanout(W, 3, m.xn, rows, l.q_bias ? bias : nullptr, y, m.workspace, m.kv_bits != 0, (hipStream_t)s,
                                    takes_sums ? &sums : nullptr));
    }
    if (m.kv_bits) {
        FK_TRY(fk_qkv_rope_store_rows(m.q, nullptr, nullptr, l.q_norm, nullptr, m.n_heads, 0, dim, dim, m.theta, m.eps, rows, pos,
                                      m.capacity, nullptr, nullptr, m.rope_tab, s));
        FK_TRY(fk_kv_cache_store_quant(m.k, m.v, l.k_norm, m.n_kv, dim, dim, m.theta, m.eps, nullptr, pos, rows, m.capacity, m.kv_bits,
                                       m.kv_group, &l.cache_kq, &l.cache_vq, s));
        if (tiled) {   // the visible prefix as bf16, then the matrix-core attention
            FK_TRY(fk_kv_cache_dequant(&l.cache_kq, m.n_kv, dim, m.capacity, m.kv_bits, m.kv_group, len, m.k_rows, m.capacity, s));
            FK_TRY(fk_kv_cache_dequant(&l.cache_vq, m.n_kv, dim, m.capacity, m.kv_bits, m.kv_group, len, m.v_rows, m.capacity, s));
            FK_TRY(run_sdpa_prefill(m.q, m.k_rows, m.v_rows, m.att, rows, len, m.n_heads, m.n_kv, dim, m.capacity, scale, true, (hipStream_t)s));
        } else {
            FK_TRY(fk_sdpa_decode_quant(m.q, &l.cache_kq, &l.cache_vq, m.att, nullptr, pos + 1, len, rows, m.n_heads, m.n_kv, dim, dim,
                                        m.capacity, m.kv_bits, m.kv_group, scale, m.partials, m.counters, s));
        }
    } else {
        Launch store;
        FK_TRY(plan_rope_store(rope, &store, sums.p ? &sums : nullptr, l.q_bias ? bias : nullptr));
        FK_TRY(run_launch(store, (hipStream_t)s));
        if (tiled)
            FK_TRY(fk_sdpa_prefill(m.q, l.cache_k, l.cache_v, m.att, rows, len, m.n_heads, m.n_kv, dim, m.capacity, scale, s));
        else
            FK_TRY(fk_sdpa_decode_rows(m.q, l.cache_k, l.cache_v, m.att, rows, pos + 1, m.n_heads, m.n_kv, dim, dim, m.capacity, scale,
                                       m.partials, m.counters, s));
    }
    FK_TRY(residual_rows(m, l.o, m.att, rows, m.x, m.x2, l.post_norm, left, (hipStream_t)s));
    if (*left == LEFT_SQUARES && l.gate.bits == l.up.bits && l.gate.group == l.up.group && takes_norm(l.gate, rows, l.gate.n, m.x2, l.post_norm)) {
        RowsRequest rq;
        rq.W[0] = &l.gate; rq.W[1] = &l.up; rq.n_mats = 2; rq.pair = true;
        rq.x = m.x2; rq.M = rows; rq.norm_w = l.post_norm; rq.eps = m.eps; rq.variant = m.swiglu_variant;
        rq.ssq_in = reinterpret_cast<const float*>(m.xn);
        rq.y[0] = m.mid;
        FK_TRY(run_rows(rq, (hipStream_t)s));
    } else {
        if (*left != LEFT_NORMED) FK_TRY(norm_rows(m, m.x2, l.post_norm, rows, (hipStream_t)s));
        if (kept_order(m, l.gate, rows) && l.gate.bits == 16) {
            FK_TRY(run_qgemm_library(&l.gate, &l.up, m.xn, rows, nullptr, nullptr, m.swiglu_variant, m.mid, m.workspace, (hipStream_t)s));
        } else if (kept_order(m, l.gate, rows)) {
            Launch gate, up, reduce;
            FK_TRY(plan_qgemm_swiglu(&l.gate, &l.up, m.xn, rows, m.swiglu_variant, m.mid, m.workspace, &gate, &up, &reduce, true));
            FK_TRY(run_launch(gate, (hipStream_t)s));
            FK_TRY(run_launch(up, (hipStream_t)s));
            FK_TRY(run_launch(reduce, (hipStream_t)s));
        } else {
            FK_TRY(run_qgemm_swiglu(&l.gate, &l.up, m.xn, rows, m.swiglu_variant, m.mid, m.workspace, m.kv_bits != 0, (hipStream_t)s));
        }
    }
    return residual_rows(m, l.down, m.mid, rows, m.x2, m.x, next ? next->input_norm : nullptr, left, (hipStream_t)s);
}

}  // namespace
}  // namespace fk

using namespace fk;

extern "C" fk_status fk_prompt_run(const fk_prompt_model* model, const uint32_t* tokens, uint32_t count, uint32_t start,
                                   uint32_t rows_per_pass, uint32_t* next_token, fk_stream s) {
    if (!model || !tokens || !next_token || count == 0 || rows_per_pass == 0) return set_error(FK_ERR_INVALID, "fk_prompt_run: null argument, no tokens or no rows");
    const fk_prompt_model& m = *model;
    if (!m.layers || !m.tokens || !m.x || !m.logits || !m.token) return set_error(FK_ERR_INVALID, "fk_prompt_run: null buffer");
    if ((uint64_t)start + count > m.capacity) return set_error(FK_ERR_INVALID, "fk_prompt_run: prompt exceeds the KV-cache capacity");
    uint32_t rows = 0;
    for (uint32_t done = 0; done < count; done += rows) {
        rows = count - done < rows_per_pass ? count - done : rows_per_pass;
        const uint32_t pos = start + done;
        FK_HIP(hipMemcpyAsync(m.tokens, tokens + done, (size_t)rows * 4, hipMemcpyHostToDevice, (hipStream_t)s));
        FK_TRY(fk_embed_lookup_rows(&m.embed, m.tokens, rows, m.embed_scale, m.x, s));
        FK_TRY(fk_rope_table_rows(m.rope_tab, m.head_dim, m.theta, pos, rows, s));   // once per pass, for every layer and head
        Left left = LEFT_NOTHING;
        for (uint32_t i = 0; i < m.n_layers; ++i)
            FK_TRY(layer_pass(m, m.layers[i], i + 1u < m.n_layers ? &m.layers[i + 1u] : nullptr, &left, rows, pos, s));
    }
    // the last row's hidden state -> logits -> greedy token, and the decode loop's step counter
    FK_TRY(fk_final_rmsnorm_lm_head(m.x + (size_t)(rows - 1) * m.hidden, m.final_norm, m.eps, &m.head, m.logits, s));
    FK_TRY(fk_argmax_logits_decode(m.logits, m.vocab, m.token, nullptr, nullptr, 0, m.argmax_workspace, s));
    if (m.step_counter) FK_TRY(fk_fill_u32(m.step_counter, start + count, 1, s));
    FK_HIP(hipMemcpyAsync(next_token, m.token, 4, hipMemcpyDeviceToHost, (hipStream_t)s));
    FK_HIP(hipStreamSynchronize((hipStream_t)s));
    return FK_OK;
}
