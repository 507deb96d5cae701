// GQA scaled-dot-product attention for one new token over a KV cache
// (split-K "flash decoding"), gfx950, on vector instructions: quantised caches, and bf16
// caches where sdpa_mma.hip's form, which plan_sdpa_decode asks first, does not serve them
// (short contexts, widths other than 64, 128 and 192 / 128, rows that are not 16-byte aligned).
//
// Grid (splits, kv heads, head tiles).  A block owns one KV head, one range of
// `chunk_len` cache positions and up to GT query heads of that KV head's group,
// so every K and V element is read from HBM once and used for all of them.
//   phase A  scores: a key row is spread over LPK lanes (16 bytes = 8 dims per
//            lane, 1 KiB contiguous per wave load); each lane dots its 8 dims
//            with the matching q slice of each head (registers), a butterfly
//            over the LPK lanes finishes the dot; scores land in LDS.
//   softmax  per head by one wave: max, exp, sum (fp32, probabilities are never
//            rounded to bf16).
//   phase B  o += p * v with the same lane layout over V rows; lanes keep 8
//            output dims per head, reduced over key slots at the end.
// A range that covers the whole context writes the output directly; otherwise
// the block stores (m, l, o) and the last block to finish per (kv head, head
// tile) merges the partials in split order (so the result does not depend on
// arrival order) and resets the counter for the next launch.
#include "fk_host.hpp"

#include "fk_probe.hpp"
FK_PROBE_DEFINE(sdpa, 4096, 10)
#define FK_SDPA_STAMP(i) \
    FK_PROBE_STAMP(sdpa, 4096, 10, blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), threadIdx.x == 0, i)
#include "sdpa_kernel.hpp"

namespace fk {

namespace {
uint32_t pow2_ceil(uint32_t v) {
    uint32_t p = 1;
    while (p < v) p <<= 1;
    return p;
}
}  // namespace

// Positions per range: every lane owns exactly kSteps key rows, i.e.
// kSteps * (block threads / lanes per key row).  128 positions for head_dim 128
// (64 KiB of K+V per block); a 32k context then spreads over 256 ranges x kv heads.
uint32_t sdpa_chunk_len(uint32_t qk_dim, uint32_t v_dim, bool fused) {
    const uint32_t lpk = pow2_ceil(qk_dim / 8), lpv = pow2_ceil(v_dim / 8);
    const uint32_t wide = lpk > lpv ? lpk : lpv;
    return (fused ? kSdpaStepsFused : kSdpaSteps) * (kSdpaBlock / wide);
}

fk_status sdpa_workspace_bytes(uint32_t n_heads, uint32_t n_kv, uint32_t qk_dim, uint32_t v_dim, uint32_t max_len,
                               size_t* partial_bytes, size_t* counter_bytes) {
    const uint32_t chunk = sdpa_chunk_len(qk_dim, v_dim, false);
    const uint32_t n_splits = (max_len + chunk - 1) / chunk;
    *partial_bytes = (size_t)n_heads * n_splits * (v_dim + 2) * sizeof(float);
    *counter_bytes = (size_t)n_heads * sizeof(uint32_t);  // >= n_kv * head tiles
    (void)n_kv;
    return FK_OK;
}

namespace {

// The kernels by tile, cache and row form.  A bf16 cache has tiles of 1 and 2 heads (rows of up to 512 dims fit a wave, so that keys and
// values always share their lanes); those of 4 and 8 belong to quantised caches.  Two heads come over a bf16 cache beyond 4096 positions:
// of 64 and 128 dims those are rows that are not 16-byte aligned and calls without a workspace.
template <int GT, int Q>
const void* decode_func(int row) {
    if (row == 16) return reinterpret_cast<const void*>(&sdpa_decode_kernel<GT, Q, 16>);
    if (row == 8) return reinterpret_cast<const void*>(&sdpa_decode_kernel<GT, Q, 8>);
    return reinterpret_cast<const void*>(&sdpa_decode_kernel<GT, Q, 0>);
}
template <int GT, bool F, int Q>
const void* fused_func(int row) {
    if (row == 16) return reinterpret_cast<const void*>(&sdpa_rope_store_kernel<GT, F, Q, 16>);
    if (row == 8) return reinterpret_cast<const void*>(&sdpa_rope_store_kernel<GT, F, Q, 8>);
    return reinterpret_cast<const void*>(&sdpa_rope_store_kernel<GT, F, Q, 0>);
}
template <int Q>
const void* decode_func(int gt, int row) {
    if constexpr (Q != 0)
        if (gt >= 4) return gt == 4 ? decode_func<4, Q>(row) : decode_func<8, Q>(row);
    return gt == 1 ? decode_func<1, Q>(row) : decode_func<2, Q>(row);
}
template <bool F, int Q>
const void* fused_tile(int gt, int row) {
    if constexpr (Q != 0)
        if (gt >= 4) return gt == 4 ? fused_func<4, F, Q>(row) : fused_func<8, F, Q>(row);
    return gt == 1 ? fused_func<1, F, Q>(row) : fused_func<2, F, Q>(row);
}
template <int Q>
const void* fused_func(bool fast, int gt, int row) { return fast ? fused_tile<true, Q>(gt, row) : fused_tile<false, Q>(gt, row); }

}  // namespace

fk_status plan_sdpa_decode(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* out,
                           const uint32_t* kv_len_ptr, uint32_t kv_len_imm, uint32_t max_len, uint32_t n_heads,
                           uint32_t n_kv, uint32_t qk_dim, uint32_t v_dim, uint32_t capacity, float scale,
                           float* partials, uint32_t* counters, Launch* out_launch, uint32_t rows,
                           const KvQuant* quant, const SdpaFusion* fusion, bool vector_form) {
    const DeviceFacts* dev;
    FK_TRY(device_facts(&dev));
    if (!q || !k || !v || !out) return set_error(FK_ERR_INVALID, "sdpa: null tensor");
    if (n_kv == 0 || n_heads == 0 || n_heads % n_kv != 0)
        return set_error(FK_ERR_INVALID, "sdpa: n_heads must be a positive multiple of n_kv");
    if (qk_dim == 0 || v_dim == 0 || qk_dim % 8 || v_dim % 8 || qk_dim > 512 || v_dim > 512)
        return set_error(FK_ERR_UNSUPPORTED, "sdpa: head dims must be multiples of 8, at most 512");
    if (max_len == 0 || max_len > capacity) return set_error(FK_ERR_INVALID, "sdpa: kv length outside (0, capacity]");
    if (rows == 0 || rows > 1024) return set_error(FK_ERR_INVALID, "sdpa: 1..1024 active rows");
    const uint32_t kvq = quant ? quant->bits : 0u;
    if (kvq) {
        if (kvq != 4 && kvq != 8) return set_error(FK_ERR_UNSUPPORTED, "sdpa: quantised cache bits must be 4 or 8");
        if (!quant->k_scales || !quant->k_biases || !quant->v_scales || !quant->v_biases)
            return set_error(FK_ERR_INVALID, "sdpa: null cache scales / biases");
        const uint32_t g = quant->group;
        if ((g != 32 && g != 64 && g != 128) || qk_dim % g || v_dim % g)
            return set_error(FK_ERR_UNSUPPORTED, "sdpa: cache group size must be 32, 64 or 128 and divide the head dims");
    }
    if (fusion) {
        if (rows != 1 || (kvq && fusion->q0_dim)) return set_error(FK_ERR_UNSUPPORTED, "sdpa: the fused rope/store form takes one row, split heads a bf16 cache");
        if (!fusion->k_new || !fusion->v_new) return set_error(FK_ERR_INVALID, "sdpa: null new k / v row");
        if (fusion->rope_dims % 2 || fusion->rope_dims > qk_dim)
            return set_error(FK_ERR_INVALID, "sdpa: rope_dims must be even and within the head");
        if ((fusion->q_norm == nullptr) != (fusion->k_norm == nullptr))
            return set_error(FK_ERR_INVALID, "sdpa: q and k head norms come together");
        if (fusion->q0_dim) {
            if (fusion->q0_dim >= qk_dim || fusion->rope_dims > qk_dim - fusion->q0_dim || !fusion->k1_new || fusion->q_norm)
                return set_error(FK_ERR_INVALID, "sdpa: split heads need a second part that holds the rotated dims, a k1 row and no head norm");
            if (fusion->k0_stride < fusion->q0_dim || fusion->v_stride < v_dim || (fusion->k1_heads != 1 && fusion->k1_heads != n_kv))
                return set_error(FK_ERR_INVALID, "sdpa: split heads: strides below the row widths or a k1 head count other than 1 / n_kv");
            if ((fusion->v_stride * 2) % 16 || ((uintptr_t)fusion->v_new & 15u))
                return set_error(FK_ERR_INVALID, "sdpa: new value rows must be 16-byte aligned");
        }
    }
    if (!kv_len_ptr && rows > 1 && kv_len_imm + rows - 1 > max_len)
        return set_error(FK_ERR_INVALID, "sdpa: the last row's kv length exceeds max_len");
    if (!kv_len_ptr && (kv_len_imm == 0 || kv_len_imm > max_len))
        return set_error(FK_ERR_INVALID, "sdpa: kv_len outside (0, max_len]");
    if (!kvq && !vector_form && sdpa_takes_mma(q, k, v, out, n_heads, n_kv, qk_dim, v_dim, max_len, rows, partials, counters))
        return plan_sdpa_mma(q, k, v, out, kv_len_ptr, kv_len_imm, max_len, n_heads, n_kv, qk_dim, v_dim, capacity, scale, partials, counters,
                             rows, fusion, out_launch);
    const uint32_t chunk = sdpa_chunk_len(qk_dim, v_dim, false);
    const uint32_t n_chunks = (max_len + chunk - 1) / chunk;
    const uint32_t G = n_heads / n_kv;
    // Tiles of 1, 2 or 4 heads run the wave-local form, which needs a key row and its value row on
    // the same lanes (equal lanes per row); other shapes take the tile of 8, which goes through LDS.
    // Rows of different widths (192 / 128) both take the lane count of the wider one -- the spare
    // lanes of the narrower row idle -- as long as a row fits a wave; bf16 caches only.
    const uint32_t lpk0 = pow2_ceil(qk_dim / 8), lpv0 = pow2_ceil(v_dim / 8), lp_wide = lpk0 > lpv0 ? lpk0 : lpv0;
    const bool same_lanes = lpk0 == lpv0 || (!kvq && lp_wide <= (uint32_t)kWave);
    int gt = !same_lanes ? 8 : (G >= 8 ? 8 : (G >= 4 ? (G == 4 ? 4 : 8) : (G >= 2 ? (G == 2 ? 2 : 4) : 1)));
    // What of a bf16 cache comes here: 64 and 128 dims up to the matrix-core form's lines (192 positions; one row of 128 dims 704 .. 1792), unaligned
    // or without a workspace beyond them; other widths and one row of 192 / 128 at any length.  Figures of 64 and 128 dims beyond those lines
    // are what the lines of this form were drawn from, for the widths that keep it.
    // Groups of 2 .. 4 query heads per KV head: smaller tiles mean more blocks with fewer registers each, and the
    // repeated K / V reads of a KV head's tiles hit the L2.  Measured (32 q / 8 kv heads x 128, cold caches), tiles
    // of 1 / 2 / 4 heads: 512 positions 7.2 / 7.9 / 8.3 us, 4096 12.6 / 13.5 / 14.2, 8192 17.3 / 18.4 / 17.5, 32768 47.8 / 37.8 / 37.6.
    // (a quantised cache has other kernels and a merge that must stay as it is: its larger tile beyond 2048 positions)
    if (same_lanes && G >= 2 && G <= 4) gt = max_len <= (kvq ? 2048u : 4096u) ? 1 : (kvq ? gt : 2);
    // Larger groups (the tile of 8 goes through LDS, three block barriers per range).  14 q / 2 kv heads x 64, time of the
    // task alone with tiles of 8 / 4 / 2 / 1 heads: 544 positions 15.8 / 11.9 / 10.7 / 9.8 us, 4096 18.4 / 14.2 / 14.2 /
    // 13.4, 12032 30.6 / 19.1 / 17.7 / 18.6.  (Not over a quantised cache: the two forms differ in the last bit, and what
    // follows from that -- a key whose group takes the other sign of its scale -- stays in the cache.)
    if (same_lanes && G > 4 && !kvq) gt = max_len <= 4096 ? 1 : 2;
    // Long contexts: a block walks several consecutive ranges (online softmax, the next range's rows in flight), so that the
    // grid stays near one to two blocks per CU and the final merge, which draws every partial into one CU, stays short.
    // (several active rows multiply the tiles: each row then needs fewer ranges to fill the chip; 8 rows x 16 heads at
    // a capacity of 1024 ran 16 ranges per row and head -- 2048 blocks, most of them past the context -- in 14.4 us; with as
    // many blocks as CUs a block of those walks its ranges alone on its CU, so from four rows on there are two a CU: a layer of
    // the 16-head model, us, one / two / four a CU: 4 rows behind 480 positions 114 / 113 / 118, 8 rows behind 1500 156 / 143 / 145, 16
    // rows 229 / 202 / 204, 16 behind 480 189 / 182 / 185; 2 rows 102 / 103 / 103.  A quantised cache keeps its ranges: their
    // merge is the last bit of a row)
    const uint32_t tiles = n_kv * ((G + gt - 1) / gt) * rows;
    uint32_t want = (n_chunks > 128 || (rows >= 4 && !kvq) ? 2u : 1u) * (uint32_t)dev->cus / tiles;
    // Up to 4096 positions, in groups: two blocks a CU where one would walk four ranges or more, up to the 16 that a merge has
    // from one trip to memory.  Tiles of one head, one a CU (for 2049 positions and more as it was, tiles of two) / this: 32 q / 8 kv x 128,
    // 2048 positions 10.5 / 10.2 us, 3300 12.9 / 12.1, 4096 13.5 / 12.7; 28 / 4, 4096 14.3 / 12.3; 64 / 8, 1000 10.1 / 9.6, 4096
    // 22.0 / 16.2.  Where one a CU walks fewer it is the slower: 32 / 8, 1000 positions 8.4 / 8.8; and with a KV head per query
    // head, whose reads share nothing: 32 / 32, 2048 positions 12.7 / 13.6.
    if (rows == 1 && same_lanes && !kvq && G >= 2 && max_len <= 4096 && want < 16u && n_chunks > 3u * want) {
        const uint32_t two = 2u * (uint32_t)dev->cus / tiles;
        want = two < 16u ? two : 16u;
    }
    // Up to three ranges of a bf16 cache: one block walks them.  A range more in the same block costs 1.04 us, the partials of two
    // blocks, their count and their merge 2.5: 14 q / 2 kv heads x 64, split / walked, 256 positions 6.0 / 4.1 us, 384 6.1 / 4.7; eight rows of
    // 384 7.3 / 5.1; 32 / 8 x 128, 128 positions 5.9 / 4.0, 192 6.2 / 4.7; 4 / 1 heads of 192 / 128 dims, 96 positions 6.4 / 5.7; 16 / 16 of 96
    // dims 6.6 / 5.9; 8 / 1 of 512 dims, 48 positions 9.1 / 6.2.  (18 shapes of 32 .. 512 dims, 1 .. 128 KV heads, 1 / 2 / 4 / 8 rows, two and three
    // ranges: walked takes 0.57 .. 0.91 of the time, the same where the rows fill the chip either way.  Over a quantised cache the two
    // differ in the last bit.)
    if (!kvq && n_chunks <= 3u) want = 1;
    // No workspace: one block walks the context, for callers whose heads and rows fill the chip that way (at one block a CU, tiles of
    // two heads from 2049 positions on); where they do not a null workspace is taken for an oversight.
    if (n_chunks > 1u && (!partials || !counters)) {
        const uint32_t pair = same_lanes && !kvq && G >= 2 && G <= 4 && max_len > 2048 ? 2u : (uint32_t)gt;
        if ((n_chunks > 128 ? 2u : 1u) * (uint32_t)dev->cus / (n_kv * ((G + pair - 1) / pair) * rows) > 1u)
            return set_error(FK_ERR_INVALID, "sdpa: workspace required when the context spans several ranges");
        want = 1;
    }
    if (want < 1) want = 1;
    if (want > 256) want = 256;
    const uint32_t cpb = (n_chunks + want - 1) / want;
    const uint32_t n_splits = (n_chunks + cpb - 1) / cpb;

    SdpaArgs a;
    memset(&a, 0, sizeof(a));
    a.q = q; a.k = k; a.v = v; a.out = out;
    a.kv_len_ptr = kv_len_ptr;
    a.kv_len_imm = kv_len_imm;
    a.n_heads = n_heads; a.n_kv = n_kv; a.qk_dim = qk_dim; a.v_dim = v_dim; a.capacity = capacity;
    a.chunk_len = chunk;
    a.n_splits = n_splits;
    a.chunks_per_block = cpb;
    a.rows = rows;
    if (kvq) {
        a.k_scales = quant->k_scales; a.k_biases = quant->k_biases;
        a.v_scales = quant->v_scales; a.v_biases = quant->v_biases;
        a.kv_group = quant->group;
    }
    if (fusion) {
        a.k_new = fusion->k_new; a.v_new = fusion->v_new;
        a.q_norm = fusion->q_norm; a.k_norm = fusion->k_norm;
        a.cache_k_w = const_cast<uint16_t*>(k);
        a.cache_v_w = const_cast<uint16_t*>(v);
        a.rope_dims = fusion->rope_dims;
        a.eps = fusion->eps; a.base_log2 = fusion->base_log2;
        a.rope_tab = fusion->rope_tab;
        a.k1_new = fusion->k1_new;
        a.q0_dim = fusion->q0_dim; a.k0_stride = fusion->k0_stride; a.k1_heads = fusion->k1_heads;
        a.traditional = fusion->traditional;
        a.v_stride = fusion->q0_dim ? fusion->v_stride : v_dim;
    }
    a.lpk = gt <= 4 ? lp_wide : lpk0;
    a.lpv = gt <= 4 ? lp_wide : lpv0;
    a.scale = scale;
    a.partials = partials;
    a.counters = counters;

    // heads of 128 (64) dims on 16 (8) lanes a row: each lane finishes its own scores, scales and biases together (sdpa_block, ROW;
    // the general form / this, 64 dims: 16 q / 4 kv heads, 11308 positions of an int4 cache 19.2 / 16.9 us; 56 / 8, the tile of 8
    // with the scales alone, 30.1 / 28.2)
    const bool alike = qk_dim == v_dim && (!kvq || quant->group == 64);
    const bool words = !kvq || (((uintptr_t)quant->k_scales | (uintptr_t)quant->k_biases | (uintptr_t)quant->v_scales | (uintptr_t)quant->v_biases) & 3u) == 0;
    const int row = alike && qk_dim == 128 && words ? 16 : (alike && qk_dim == 64 ? 8 : 0);
    const void* func = nullptr;
    if (fusion) {
        // whole-width rotation of at most 128 dims with a table: the form whose loads run ahead
        // (heads of fewer than 128 dims add their squares in another order there: a quantised cache keeps the one it has)
        const bool fast = fusion->rope_tab && fusion->rope_dims == qk_dim && qk_dim <= 128 && !(kvq && fusion->q_norm && qk_dim != 128);
        func = kvq == 4 ? fused_func<4>(fast, gt, row) : (kvq == 8 ? fused_func<8>(fast, gt, row) : fused_func<0>(fast, gt, row));
    } else {
        func = kvq == 4 ? decode_func<4>(gt, row) : (kvq == 8 ? decode_func<8>(gt, row) : decode_func<0>(gt, row));
    }
    out_launch->func = func;
    out_launch->grid = dim3(n_splits, n_kv, ((G + gt - 1) / gt) * rows);
    out_launch->block = dim3(kSdpaBlock, 1, 1);
    out_launch->shmem = (uint32_t)(sdpa_lds_floats(gt, chunk, qk_dim, v_dim, fusion != nullptr, kvq != 0) * sizeof(float));
    out_launch->set_args(a);
    return FK_OK;
}

}  // namespace fk
