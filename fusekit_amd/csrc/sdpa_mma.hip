// Decode attention over a bf16 cache on the matrix cores: the queries that read the same K / V rows -- the heads of a KV head's
// group, of one token or of several -- are the columns of v_mfma_f32_16x16x32_bf16.
//
//     S^T[key, query] = K[key, :] . Q[query, :]        A = K rows, B = Q rows
//     O^T[d, query] += V^T[d, key] . P^T[key, query]   A = V^T, B = P^T = the score registers as they lie
//
// Probabilities are fp32 and stay so: p = hi + mid + lo, three bf16 values that add up to it exactly, are columns (tiles of 4 queries:
// 12 of the 16) or matrix instructions of their own (8 queries: two, 16: three); products are exact, sums fp32 as before.  A lane owns one
// query and four keys of each 16; its softmax reference moves only when a step's maximum outgrows it by 2^8, and a probability carries
// the factor 2^-8 all the way (sums, too: it cancels), so that none is above 1 and values up to bf16's largest are summed as they
// would be behind the true maximum.
//
// A wave owns its steps of 32 keys: K and V rows go from memory into its own part of LDS (global_load_lds, 16-byte pieces XOR-swizzled by
// the row, so that the fragment reads meet all banks); the next step's keys are requested as soon as this one's are in registers, its
// values behind the second product.  No barrier and no wait for another wave stands in a wave's loop; V^T is read with ds_read_b64_tr_b16.
// The waves meet once, after their last step; blocks that share a context leave (m, l, o) partials in 16-byte pieces, and the one that
// arrives last merges them in range order, all of a head requested together.
//
// The form on vector instructions (sdpa_kernel.hpp: quantised caches, other widths, short contexts) spends about 110 of them on a lane's 8
// dims of a key for 4 heads; here the products cost none and a step's softmax about 100 for 32 keys of a whole tile, so that what remains is
// the bytes, the start and, where blocks share a context, the 2.2 us of partials, count and merge.  That form -> this, us, launch to launch
// in a graph, caches from memory: 32 / 8 heads x 128 at 1024 positions 8.9 -> 7.8, 4096 13.3 -> 9.9, 12000 21.3 -> 14.6, 32768 37 ->
// 28.1 (134 MB: 4.8 TB/s of the 5.8 that a plain read reaches); 14 / 2 x 64 at 544 6.9 -> 5.5, 4096 10.0 -> 6.9, 12000 13.0 -> 8.4; 64 rows of
// 32 / 8 x 128 at 500 33 -> 9.6; 16 heads of 192 / 128, 8 rows at 480 12.6 -> 10.8, 96 rows at 1500 141 -> 19.4.
#include "dma_device.hpp"
#include "fk_host.hpp"
#include "rope_device.hpp"

namespace fk {

typedef __bf16 mma_bf16x8_t __attribute__((ext_vector_type(8)));
typedef short mma_s16x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t mma_u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t mma_u32x2_t __attribute__((ext_vector_type(2)));

struct SdpaMmaArgs {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    uint16_t* out;
    const uint32_t* kv_len_ptr;  // device scalar, or null -> kv_len_imm
    uint32_t kv_len_imm;
    uint32_t n_heads, group, capacity;
    uint32_t span, n_splits;     // positions of a block, blocks that share a context
    uint32_t rows;               // active token rows: row r attends to kv_len + r positions
    float scale;
    float* partials;             // o [rows * n_heads][n_splits][v_dim], then (m, l) [rows * n_heads][n_splits]
    uint32_t* counters;          // [n_kv * tiles], zero before the first launch
    // with the rotation and the append (one row): the raw projection outputs of the token at position kv_len - 1
    const uint16_t* k_new;
    const uint16_t* v_new;
    const uint16_t* q_norm;
    const uint16_t* k_norm;
    uint16_t* cache_k_w;
    uint16_t* cache_v_w;
    uint32_t rope_dims;
    float eps, base_log2;
    const float* rope_tab;
};
// MMA_STAGED: the token's rows, norms and table are copied value by value (any address; heads of two parts, as SdpaArgs has them), so
// that such a launch takes the form that the pair it stands for takes.  Against the form on vector instructions, us, that / this: 14 / 2 heads x 64,
// 256 positions 5.2 / 5.6, 544 7.1 / 6.6, 4096 9.7 / 7.6; 32 / 8 x 128, 256 6.1 / 6.3, 1024 8.2 / 8.7, 4096 12.2 / 10.4.
// (A block of its own: 32 bytes more in every launch's took 0.15 us where ranges are merged, 14 / 2 heads x 64, 4096 positions 6.82 / 6.97.)
struct SdpaMmaStagedArgs : SdpaMmaArgs {
    const uint16_t* k1_new;
    uint32_t q0_dim, k0_stride, v_stride, k1_heads, traditional;
};

constexpr uint32_t kMmaStep = 32;   // keys of a wave's step
constexpr uint32_t kMmaMaxSplits = 64;
constexpr float kLagLog2 = 8.0f, kLag = 1.0f / 256.0f;   // how far a step's maximum may lie above the softmax reference

// LDS of a block: what the first barrier hands over, then the waves' stages (the meeting reuses them).
constexpr uint32_t mma_input_bytes(uint32_t qk, uint32_t qt, bool fused) {
    // fused: q heads, k, v, two norms, the table, each in 16-byte pieces; rounded up to whole requests
    const uint32_t raw = fused ? ((qt + 4u) * qk * 2u + qk * 4u + 1023u) / 1024u * 1024u : (qt * qk * 2u + 1023u) / 1024u * 1024u;
    return raw + (fused ? ((qt + 1u) * (qk * 2u + 16u) + 1023u) / 1024u * 1024u : 0u);
}
constexpr uint32_t mma_stage_bytes(uint32_t qk, uint32_t vd) { return kMmaStep * (qk + vd) * 2u; }
constexpr uint32_t mma_lds_bytes(uint32_t qk, uint32_t vd, uint32_t qt, uint32_t nw, bool fused) {
    const uint32_t stages = nw * mma_stage_bytes(qk, vd), meet = nw * qt * (vd + 4u) * 4u + 2u * nw * qt * 4u + 64u;
    return mma_input_bytes(qk, qt, fused) + (stages > meet ? stages : meet);
}

__device__ __forceinline__ float mma_rows_sum(float v) {   // over the wave's four 16-lane rows, lane by lane
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
template <int CTRL>   // (lanes without a source get zero, and no register to clear first as dpp_move has: 0.1 us of a block of 128 dims)
__device__ __forceinline__ float mma_dpp(float v) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true)); }
// what another block of this launch wrote, or is to read, moves past every cache that the two do not share (sc1)
constexpr int kShared = 16;

// QT queries of a KV head a block, NW waves.  FORM: what the launch does ahead of the attention.
enum MmaForm { MMA_PLAIN, MMA_FUSED, MMA_STAGED };   // nothing; rotation and append; the same with its inputs copied value by value
template <int QK, int VD, int QT, int NW, MmaForm FORM>
__global__ __launch_bounds__(NW * 64, 1) void sdpa_mma_kernel(const std::conditional_t<FORM == MMA_STAGED, SdpaMmaStagedArgs, SdpaMmaArgs> a) {
    constexpr bool FUSED = FORM != MMA_PLAIN, STAGED = FORM == MMA_STAGED;
    constexpr uint32_t KROW = QK * 2u, VROW = VD * 2u, KP = QK / 8u, VP = VD / 8u;      // bytes and 16-byte pieces of a row
    constexpr uint32_t KT = kMmaStep * KROW, STAGE = mma_stage_bytes(QK, VD);
    constexpr int KREQ = (int)(KT / 1024u), VREQ = (int)(kMmaStep * VROW / 1024u), REQ = KREQ + VREQ;   // requests of a step
    constexpr int KS = QK / 32, DT = VD / 16;
    constexpr int PARTS = QT == 4 ? 1 : (QT == 8 ? 2 : 3);                              // matrix instructions for the probabilities' parts
    constexpr uint32_t IN = mma_input_bytes(QK, QT, FUSED), ROUND = NW * kMmaStep;
    static_assert(!FUSED || QK == VD, "");
    extern __shared__ uint4 mma_lds[];
    unsigned char* const lds = reinterpret_cast<unsigned char*>(mma_lds);
    kernarg_warm<(int)sizeof(a)>();

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15u, g = lane >> 4;
    const uint32_t split = blockIdx.x, kvh = blockIdx.y, tile = blockIdx.z, blk0 = split * a.span;
    const uint32_t G = a.group, e0 = tile * QT, left = a.rows * G - e0, nq = left < (uint32_t)QT ? left : (uint32_t)QT;
    const uint32_t mine = n % QT < nq ? n % QT : nq - 1u;   // this lane's query (columns past the last repeat it and store nothing)
    const uint32_t row_lo = e0 / G, row_hi = (e0 + nq - 1u) / G;

    auto k_swizzle = [](uint32_t row) { return KP == 16u ? row & 15u : (row >> 1) & 7u; };
    auto v_swizzle = [](uint32_t row) { return VP == 16u ? (row & 7u) << 1 : ((row >> 1) & 3u) << 1; };
    auto k_at = [&](uint32_t row, uint32_t piece) { return row * KROW + ((KP == 24u ? (piece & ~7u) | ((piece ^ k_swizzle(row)) & 7u) : piece ^ k_swizzle(row)) * 16u); };

    uint32_t kv_raw = a.kv_len_imm;
    if (a.kv_len_ptr) kv_raw = *(const __attribute__((address_space(4))) uint32_t*)(uintptr_t)a.kv_len_ptr;
    __builtin_amdgcn_sched_barrier(0);

    // ---- what the first barrier hands over: one request a wave (plain: the query rows; else see the order below) ----
    // FUSED: q heads | k | v | q norm | k norm | table
    constexpr uint32_t AT_K = QT * KP, AT_V = AT_K + KP, AT_QN = AT_V + VP, AT_KN = AT_QN + KP, AT_TAB = AT_KN + KP, PIECES = AT_TAB + QK / 4u;
    constexpr uint32_t RAW = FUSED ? (PIECES * 16u + 1023u) / 1024u : (QT * KROW + 1023u) / 1024u;   // requests
    if constexpr (STAGED) {
        const uint32_t d0 = a.q0_dim ? a.q0_dim : (uint32_t)QK;
        const uint16_t* k0 = a.k_new + (size_t)kvh * a.k0_stride;
        const uint16_t* k1 = a.q0_dim ? a.k1_new + (size_t)(a.k1_heads == 1u ? 0u : kvh) * (QK - d0) : k0;
        static_assert(PIECES <= NW * 64u, "a piece a thread");
        if (const uint32_t p = tid; p < PIECES) {
            // eight values: from `src`, from the cut-th on from `src2`, none from the last-th on
            const uint16_t *src = a.q + (size_t)(kvh * G + e0 + (p / KP < nq ? p / KP : 0u)) * QK + (p % KP) * 8u, *src2 = k0;
            uint32_t cut = 8u, last = 8u;
            if (p >= AT_K && p < AT_V) {
                const uint32_t e = (p - AT_K) * 8u;
                cut = d0 > e ? (d0 - e < 8u ? d0 - e : 8u) : 0u;
                src = k0 + e;
                src2 = k1 + ((ptrdiff_t)e - (ptrdiff_t)d0);
            }
            if (p >= AT_V && p < AT_QN) src = a.v_new + (size_t)kvh * a.v_stride + (p - AT_V) * 8u;
            if (p >= AT_QN && p < AT_KN) src = a.q_norm + (p - AT_QN) * 8u;
            if (p >= AT_KN && p < AT_TAB) src = a.k_norm + (p - AT_KN) * 8u;
            if (p >= AT_QN && p < AT_TAB && !a.q_norm) last = 0u;
            if (p >= AT_TAB) {
                const uint32_t at = (p - AT_TAB) * 8u, n = a.rope_tab ? a.rope_dims * 2u : 0u;   // (halves of floats)
                src = reinterpret_cast<const uint16_t*>(a.rope_tab) + at;
                last = n > at ? (n - at < 8u ? n - at : 8u) : 0u;
            }
            uint32_t x[8];   // (where nothing stands behind a value, q's first is read)
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) x[j] = *(j < last ? (j < cut ? src : src2) + j : a.q);
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) x[j] = j < last ? x[j] : 0u;
            *reinterpret_cast<uint4*>(lds + p * 16u) = make_uint4(x[0] | x[1] << 16, x[2] | x[3] << 16, x[4] | x[5] << 16, x[6] | x[7] << 16);
        }
    }
    for (uint32_t i = wave; i < (STAGED ? 0u : RAW); i += NW) {
        const uint32_t p = i * 64u + lane;
        const unsigned char* src;
        if constexpr (FUSED) {
            const uint32_t h = p / KP < nq ? p / KP : 0u;
            src = reinterpret_cast<const unsigned char*>(a.q + (size_t)(kvh * G + e0 + h) * QK) + (p % KP) * 16u;
            if (p >= AT_K && p < AT_V) src = reinterpret_cast<const unsigned char*>(a.k_new + (size_t)kvh * QK) + (p - AT_K) * 16u;
            if (p >= AT_V && p < AT_QN) src = reinterpret_cast<const unsigned char*>(a.v_new + (size_t)kvh * VD) + (p - AT_V) * 16u;
            if (a.q_norm && p >= AT_QN && p < AT_KN) src = reinterpret_cast<const unsigned char*>(a.q_norm) + (p - AT_QN) * 16u;
            if (a.q_norm && p >= AT_KN && p < AT_TAB) src = reinterpret_cast<const unsigned char*>(a.k_norm) + (p - AT_KN) * 16u;
            if (a.rope_tab && p >= AT_TAB && p - AT_TAB < a.rope_dims / 4u) src = reinterpret_cast<const unsigned char*>(a.rope_tab) + (p - AT_TAB) * 16u;
        } else {
            const uint32_t c = p / KP < nq ? p / KP : 0u, e = e0 + c, r = e / G;
            src = reinterpret_cast<const unsigned char*>(a.q + ((size_t)r * a.n_heads + kvh * G + (e - r * G)) * QK) + (p % KP) * 16u;
        }
        dma16(i * 1024u, src);
    }

    // ---- K and V of a step into this wave's stage ----
    const unsigned char* kbase = reinterpret_cast<const unsigned char*>(a.k + (size_t)kvh * a.capacity * QK);
    const unsigned char* vbase = reinterpret_cast<const unsigned char*>(a.v + (size_t)kvh * a.capacity * VD);
    const uint32_t my_stage = IN + wave * STAGE;
    uint32_t koff[KREQ], voff[VREQ];
#pragma unroll
    for (int i = 0; i < KREQ; ++i) {
        const uint32_t flat = (uint32_t)i * 64u + lane, row = flat / KP;
        koff[i] = row * KROW + (k_at(row, flat % KP) - row * KROW);   // (the piece that lies at this place: the swizzle is its own inverse)
    }
#pragma unroll
    for (int i = 0; i < VREQ; ++i) {
        const uint32_t flat = (uint32_t)i * 64u + lane, row = flat / VP;
        voff[i] = row * VROW + ((flat % VP) ^ v_swizzle(row)) * 16u;
    }
    // (rows past the allocation repeat its last row: they are masked)
    auto issue_k = [&](uint32_t kv0) {
        const uint32_t at = kv0 < a.capacity ? kv0 : a.capacity - 1u, more = a.capacity - 1u - at;
        const unsigned char* base = kbase + (size_t)at * KROW;
        if (__builtin_expect(more >= kMmaStep - 1u, 1)) {
#pragma unroll
            for (int i = 0; i < KREQ; ++i) dma16(my_stage + (uint32_t)i * 1024u, koff[i], base);
        } else {
#pragma unroll
            for (int i = 0; i < KREQ; ++i) {
                const uint32_t row = ((uint32_t)i * 64u + lane) / KP, over = row > more ? row - more : 0u;
                dma16(my_stage + (uint32_t)i * 1024u, koff[i] - over * KROW, base);
            }
        }
    };
    auto issue_v = [&](uint32_t kv0) {
        const uint32_t at = kv0 < a.capacity ? kv0 : a.capacity - 1u, more = a.capacity - 1u - at;
        const unsigned char* base = vbase + (size_t)at * VROW;
        if (__builtin_expect(more >= kMmaStep - 1u, 1)) {
#pragma unroll
            for (int i = 0; i < VREQ; ++i) dma16(my_stage + KT + (uint32_t)i * 1024u, voff[i], base);
        } else {
#pragma unroll
            for (int i = 0; i < VREQ; ++i) {
                const uint32_t row = ((uint32_t)i * 64u + lane) / VP, over = row > more ? row - more : 0u;
                dma16(my_stage + KT + (uint32_t)i * 1024u, voff[i] - over * VROW, base);
            }
        }
    };
    const uint32_t first = blk0 + wave * kMmaStep;
    // a device scalar is not trusted: a length beyond what the launch was sized for would leave ranges without a block
    const uint32_t covered = a.n_splits * a.span < a.capacity ? a.n_splits * a.span : a.capacity;
    // The first range's keys are requested ahead of a length on the device (its values are not: a short context would wait for what it does not
    // need), of rows of 128 dims and more the first two waves' only, and the length in front of everything.  All waves' keys, then the
    // length / this, us: 32 / 8 heads x 128, contexts of 50 in plans of 256 4.9 / 4.5, of 1024 4.5 / 4.4, of 4096 4.9 / 4.5, 150 in 256 5.4 / 5.0; 8 rows,
    // 30 in 1024 6.1 / 5.8; 16 heads of 192 / 128, 8 rows, 30 in 256 7.1 / 6.3; whole plans the same.  (64 dims: 14 / 2 heads, 50 in 1024
    // 3.9 / 3.8, but three rounds in one block, 544, 5.7 / 5.8.)
    const bool ahead = split == 0 && first < covered && (QK == 64 || !a.kv_len_ptr || wave < 2u);
    if (ahead) issue_k(first);
    const uint32_t kv0_len = kv_raw > covered ? covered : kv_raw;   // (before a row is added: a tile's rows stay in order whatever was read)
    auto limit_of = [&](uint32_t row) {
        const uint32_t l = kv0_len + row;
        return l < 1u ? 1u : (l > covered ? covered : l);
    };
    const uint32_t lim_hi = limit_of(row_hi), lim_lo = limit_of(row_lo), q_limit = limit_of((e0 + mine) / G);
    const uint32_t n_active = (lim_hi + a.span - 1u) / a.span, pos = lim_hi - 1u;
    if (split >= n_active) {   // the whole block; nothing may be on its way into LDS that another block gets
        wait_loads<0>();
        return;
    }
    const uint32_t end = lim_hi - blk0 < a.span ? lim_hi : blk0 + a.span;
    const uint32_t n_steps = end > first ? (end - first + ROUND - 1u) / ROUND : 0u;
    if (n_steps != 0) {
        if (!ahead) issue_k(first);
        issue_v(first);
    }
    if (n_steps != 0) {
        wait_loads<REQ>();
    } else if (ahead) {
        wait_loads<KREQ>();
    } else {
        wait_loads<0>();
    }
    __syncthreads();

    // ---- queries ----
    uint16_t* const qn = reinterpret_cast<uint16_t*>(lds + RAW * 1024u);   // FUSED: [QT + 1][QK + 8], rotated heads, then the new key
    constexpr uint32_t QN = QK + 8u;
    const uint16_t* const raw = reinterpret_cast<const uint16_t*>(lds);
    const bool owner = FUSED && pos >= blk0 && pos < blk0 + a.span;
    if constexpr (FUSED) {
        const float* tab = a.rope_tab ? reinterpret_cast<const float*>(lds + AT_TAB * 16u) : nullptr;
        const bool fast = a.rope_tab && a.rope_dims == (uint32_t)QK, norm = a.q_norm != nullptr;
        for (uint32_t h = wave; h < nq + (owner ? 1u : 0u); h += NW) {
            const bool key = h == nq;
            const uint16_t* src = raw + (key ? AT_K * 8u : h * QK);
            uint16_t* dst = qn + (key ? (uint32_t)QT : h) * QN;
            const uint16_t* nw = raw + (key ? AT_KN : AT_QN) * 8u;
            if constexpr (STAGED) {
                if (a.q0_dim) {
                    split_head_transform(src, src + a.q0_dim, dst, a.q0_dim, QK - a.q0_dim, a.rope_dims, a.traditional != 0, pos, a.base_log2, lane, tab);
                    continue;
                }
            }
            if (fast) {
                const HeadPair p = head_pair_fetch(src, nw, tab, QK / 2u, lane);
                head_pair_apply(p, dst, norm, QK / 2u, a.eps, lane, true);
            } else {
                head_transform(src, dst, norm ? nw : nullptr, QK, a.rope_dims, pos, a.base_log2, a.eps, true, lane, tab);
            }
        }
        __syncthreads();
        if (owner && tile == 0 && tid < KP) {
            const size_t row = (size_t)kvh * a.capacity + pos;
            *reinterpret_cast<uint4*>(a.cache_k_w + row * QK + tid * 8u) = *reinterpret_cast<const uint4*>(qn + QT * QN + tid * 8u);
            *reinterpret_cast<uint4*>(a.cache_v_w + row * VD + tid * 8u) = *reinterpret_cast<const uint4*>(raw + AT_V * 8u + tid * 8u);
        }
    }
    mma_bf16x8_t qf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const mma_bf16x8_t*>((FUSED ? qn + mine * QN : raw + mine * QK) + s * 32 + g * 8u);

    f32x4_t acc[PARTS][DT];
#pragma unroll
    for (int p = 0; p < PARTS; ++p)
#pragma unroll
        for (int i = 0; i < DT; ++i) acc[p][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    const float scale2 = a.scale * 1.44269504088896341f;
    const uint32_t part = n / QT;   // QT 4, 8: which part of the probabilities this column multiplies

    for (uint32_t j = 0; j < n_steps; ++j) {
        const uint32_t kv0 = first + j * ROUND;
        unsigned char* const ks = lds + my_stage;
        unsigned char* const vs = ks + KT;
        const bool more = j + 1u < n_steps;
        wait_loads<VREQ>();
        const bool has_new = FUSED && pos >= kv0 && pos < kv0 + kMmaStep;
        if constexpr (FUSED) {
            if (has_new) {   // the new key, not yet cached
                const uint32_t r = pos - kv0;
                if (lane < KP) *reinterpret_cast<uint4*>(ks + k_at(r, lane)) = *reinterpret_cast<const uint4*>(qn + QT * QN + lane * 8u);
                wave_lds_order();
            }
        }
        mma_bf16x8_t kf[2][KS];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int s = 0; s < KS; ++s) kf[t][s] = *reinterpret_cast<const mma_bf16x8_t*>(ks + k_at((uint32_t)t * 16u + n, (uint32_t)s * 4u + g));
        // Beyond 64 dims a score is formed in two chains: in one, each instruction's rounding is that of the whole sum so far.  And a
        // probability's exponent is scaled and referred with one rounding.  Outputs rounded to the wrong side, of a million, queries of four
        // times unit variance: the form on vector instructions / one chain and two roundings / this: 32 / 8 heads x 128, 1000 positions
        // 429 / 490 / 334, 4096 493 / 645 / 394; 56 / 8, 1500 480 / 524 / 379; 14 / 2 x 64, 2000 391 / 446 / 349.
        float raw_s[8], x[8];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            constexpr int HALF = KS >= 4 ? KS / 2 : KS;
            f32x4_t s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < HALF; ++s) s4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][s], qf[s], s4, 0, 0, 0);
            if constexpr (HALF < KS) {
                f32x4_t s5 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = HALF; s < KS; ++s) s5 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][s], qf[s], s5, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) s4[i] += s5[i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                raw_s[t * 4 + i] = s4[i];
                x[t * 4 + i] = s4[i] * scale2;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue_k(kv0 + ROUND);   // the keys are in registers: their place takes the next step's
        if (kv0 + kMmaStep > lim_lo) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (kv0 + (uint32_t)(i / 4) * 16u + 4u * g + (uint32_t)(i % 4) >= q_limit) x[i] = -INFINITY;
        }
        float mx = x[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) mx = fmaxf(mx, x[i]);
        if (__builtin_amdgcn_ballot_w64(mx > m_run + kLagLog2) != 0) {   // rare after the first steps
            mx = rows_max(mx);
            const bool grow = mx > m_run + kLagLog2;
            const float alpha = grow ? __builtin_amdgcn_exp2f(m_run - mx) : 1.0f;
            m_run = grow ? mx : m_run;
            l_run *= alpha;
#pragma unroll
            for (int p = 0; p < PARTS; ++p)
#pragma unroll
                for (int i = 0; i < DT; ++i) acc[p][i] *= alpha;
        }
        const float m_ref = m_run == -INFINITY ? 0.f : m_run;   // no live key yet: every term is 2^-inf = 0
        float ex[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) ex[i] = fmaf(raw_s[i], scale2, -m_ref);
        if (kv0 + kMmaStep > lim_lo) {
#pragma unroll
            for (int i = 0; i < 8; ++i) ex[i] = x[i] == -INFINITY ? -INFINITY : ex[i];
        }
        mma_u32x4_t pb[PARTS];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float p0 = __builtin_amdgcn_exp2f(ex[2 * i]) * kLag, p1 = __builtin_amdgcn_exp2f(ex[2 * i + 1]) * kLag;
            l_run += p0 + p1;
            const uint32_t hi = pack_bf16(p0, p1);
            if constexpr (QT == 4) {
                const uint32_t take1 = part >= 1u ? ~0u : 0u, take2 = part >= 2u ? ~0u : 0u;
                p0 -= __uint_as_float((hi << 16) & take1);
                p1 -= __uint_as_float(hi & take1 & 0xffff0000u);
                const uint32_t mid = pack_bf16(p0, p1);
                p0 -= __uint_as_float((mid << 16) & take2);
                p1 -= __uint_as_float(mid & take2 & 0xffff0000u);
                pb[0][i] = pack_bf16(p0, p1);   // (the fourth part's columns are not read)
            } else {
                p0 -= bf16_lo(hi);
                p1 -= bf16_hi(hi);
                const uint32_t mid = pack_bf16(p0, p1);
                p0 -= bf16_lo(mid);
                p1 -= bf16_hi(mid);
                const uint32_t lo = pack_bf16(p0, p1);
                if constexpr (QT == 8) {
                    pb[0][i] = part ? mid : hi;
                    pb[1][i] = lo;              // (its upper columns are not read)
                } else {
                    pb[0][i] = hi;
                    pb[1][i] = mid;
                    pb[2][i] = lo;
                }
            }
        }
        if (more) wait_loads<KREQ>();
        else wait_loads<0>();
        bool repeat = false;
        if (kv0 + kMmaStep > lim_lo || has_new) {
            if (kv0 + kMmaStep > lim_hi) {   // rows behind the context may hold anything: zero
                for (uint32_t i = (lim_hi - kv0) * VP + lane; i < kMmaStep * VP; i += 64u) *reinterpret_cast<uint4*>(vs + i * 16u) = make_uint4(0, 0, 0, 0);
            }
            if constexpr (FUSED) {
                if (has_new && lane < VP) {
                    const uint32_t r = pos - kv0;
                    *reinterpret_cast<uint4*>(vs + r * VROW + ((lane ^ v_swizzle(r)) * 16u)) = *reinterpret_cast<const uint4*>(raw + (AT_V + lane) * 8u);
                }
            }
            wave_lds_order();
            if constexpr (!FUSED) {
                // rows that only some of the queries see: an infinity or a NaN there must not reach the others through a zero
                if (lim_lo < lim_hi) {
                    bool odd = false;
                    for (uint32_t i = (lim_lo > kv0 ? lim_lo - kv0 : 0u) * VP + lane; i < kMmaStep * VP; i += 64u) {
                        const uint4 w = *reinterpret_cast<const uint4*>(vs + i * 16u);
                        for (uint32_t c : {w.x, w.y, w.z, w.w}) odd |= (c & 0x7f80u) == 0x7f80u || (c & 0x7f800000u) == 0x7f800000u;
                    }
                    repeat = __builtin_amdgcn_ballot_w64(odd) != 0;
                }
            }
        }
        auto values = [&](int i) {
            mma_s16x4_t v4[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t row = (uint32_t)h * 16u + 4u * g + (n >> 2), piece = (uint32_t)(2 * i) + ((n & 3u) >> 1);
                unsigned char* at = vs + row * VROW + ((piece ^ v_swizzle(row)) * 16u) + (n & 1u) * 8u;
                typedef __attribute__((address_space(3))) mma_s16x4_t* lds_ptr;
                v4[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(mma_s16x4_t*)at);
            }
            return __builtin_bit_cast(mma_bf16x8_t, __builtin_shufflevector(v4[0], v4[1], 0, 1, 2, 3, 4, 5, 6, 7));
        };
        if (!repeat) {
            mma_bf16x8_t vf[DT];
#pragma unroll
            for (int i = 0; i < DT; ++i) vf[i] = values(i);
#pragma unroll
            for (int p = 0; p < PARTS; ++p)
#pragma unroll
                for (int i = 0; i < DT; ++i)
                    acc[p][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[i], __builtin_bit_cast(mma_bf16x8_t, pb[p]), acc[p][i], 0, 0, 0);
        } else {   // row by row, the last first: what the next one does not see is zeroed
            for (uint32_t r = row_hi + 1u; r-- > row_lo;) {
                const uint32_t lim = limit_of(r), from = lim > kv0 ? lim - kv0 : 0u;
                for (uint32_t i = from * VP + lane; i < kMmaStep * VP; i += 64u) *reinterpret_cast<uint4*>(vs + i * 16u) = make_uint4(0, 0, 0, 0);
                wave_lds_order();
                const bool take_it = (e0 + mine) / G == r;
#pragma unroll
                for (int i = 0; i < DT; ++i) {
                    const mma_bf16x8_t v8 = values(i);
#pragma unroll
                    for (int p = 0; p < PARTS; ++p) {
                        const f32x4_t o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v8, __builtin_bit_cast(mma_bf16x8_t, pb[p]), acc[p][i], 0, 0, 0);
#pragma unroll
                        for (int c = 0; c < 4; ++c) acc[p][i][c] = take_it ? o[c] : acc[p][i][c];
                    }
                }
                wave_lds_order();
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue_v(kv0 + ROUND);
    }
    wait_loads<0>();   // (a first step that no key of the context lies in)

    // ---- the waves meet ----
    const float l_all = mma_rows_sum(l_run);
    __syncthreads();
    constexpr uint32_t OS = VD + 4u;
    float* const red = reinterpret_cast<float*>(lds + IN);              // [wave][query][OS]
    float* const wm = red + NW * QT * OS;                               // [wave][query] references, sums
    float* const wl = wm + NW * QT;
    uint32_t* const flag = reinterpret_cast<uint32_t*>(wl + NW * QT);
    if (g == 0 && n < (uint32_t)QT) {
        wm[wave * QT + n] = m_run;
        wl[wave * QT + n] = l_all;
    }
    // An infinite value's products with zero parts are no numbers: where a sum of the first parts is infinite it stands alone.  Looked for once, over
    // the tile, and the sums formed by all lanes ahead of one test of the column; value by value / this, us: 32 / 8 heads x 128, 1024 positions
    // 8.07 / 7.93, 50 of 1024 5.51 / 5.29, 256 6.01 / 5.97; 14 / 2 x 64, 544 5.11 / 5.02, 12000 8.04 / 7.94.
    float o[DT][4], far = 0.f;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float hi = acc[0][i][r];
            float rest;
            if constexpr (QT == 4) rest = mma_dpp<0x104>(hi) + mma_dpp<0x108>(hi);            // the columns 4 and 8 on
            else if constexpr (QT == 8) rest = mma_dpp<0x108>(hi) + acc[1][i][r];
            else rest = acc[1][i][r] + acc[2][i][r];
            o[i][r] = hi + rest;
            far = fmaxf(far, __builtin_fabsf(hi));
        }
    if (__builtin_amdgcn_ballot_w64(far == INFINITY) != 0) {
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[i][r] = __builtin_fabsf(acc[0][i][r]) < INFINITY ? o[i][r] : acc[0][i][r];
    }
    if (n < (uint32_t)QT) {
#pragma unroll
        for (int i = 0; i < DT; ++i)
            *reinterpret_cast<float4*>(red + (wave * QT + n) * OS + (uint32_t)i * 16u + 4u * g) = make_float4(o[i][0], o[i][1], o[i][2], o[i][3]);
    }
    __syncthreads();
    const bool direct = n_active == 1u;
    const uint32_t heads = a.rows * a.n_heads;
    const __amdgpu_buffer_rsrc_t parts = __builtin_amdgcn_make_buffer_rsrc(a.partials, 0, (int)(heads * a.n_splits * (VD + 2u) * 4u), 0x27000);
    for (uint32_t i = tid; i < nq * (VD / 4u); i += NW * 64u) {
        const uint32_t qi = i / (VD / 4u), d = (i % (VD / 4u)) * 4u, e = e0 + qi, r = e / G;
        float M = wm[qi];
#pragma unroll
        for (int w = 1; w < NW; ++w) M = fmaxf(M, wm[w * QT + qi]);
        const float ref = M == -INFINITY ? 0.f : M;
        float l = 0.f;
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float f = __builtin_amdgcn_exp2f(wm[w * QT + qi] - ref);
            const float4 p = *reinterpret_cast<const float4*>(red + (w * QT + qi) * OS + d);
            l = fmaf(wl[w * QT + qi], f, l);
            o = make_float4(fmaf(p.x, f, o.x), fmaf(p.y, f, o.y), fmaf(p.z, f, o.z), fmaf(p.w, f, o.w));
        }
        const uint32_t head = r * a.n_heads + kvh * G + (e - r * G);
        if (direct) {
            *reinterpret_cast<uint2*>(a.out + (size_t)head * VD + d) = make_uint2(pack_bf16(o.x / l, o.y / l), pack_bf16(o.z / l, o.w / l));
        } else {
            const uint32_t at = head * a.n_splits + split;
            const mma_u32x4_t w = {__float_as_uint(o.x), __float_as_uint(o.y), __float_as_uint(o.z), __float_as_uint(o.w)};
            __builtin_amdgcn_raw_buffer_store_b128(w, parts, (int)((at * VD + d) * 4u), 0, kShared);
            if (d == 0) {
                const mma_u32x2_t ml = {__float_as_uint(M), __float_as_uint(l)};
                __builtin_amdgcn_raw_buffer_store_b64(ml, parts, (int)((heads * a.n_splits * VD + at * 2u) * 4u), 0, kShared);
            }
        }
    }
    if (direct) return;

    // ---- the block that arrives last merges: one wave a query, every partial of a head requested together ----
    wait_memory_ops_done();
    __syncthreads();
    if (tid == 0) {
        const uint32_t prev = atomicAdd(&a.counters[kvh * gridDim.z + tile], 1u);
        *flag = prev == n_active - 1u ? 1u : 0u;
    }
    __syncthreads();
    if (*flag == 0u) return;
    if (tid == 0) __hip_atomic_store(&a.counters[kvh * gridDim.z + tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    constexpr uint32_t LP = VD / 4u, SPR = 64u / LP;   // lanes of a partial, partials of a request
    const uint32_t ranges = __builtin_amdgcn_readfirstlane(n_active);
    for (uint32_t qi = wave; qi < nq; qi += NW) {
        const uint32_t e = e0 + qi, r = e / G, head = r * a.n_heads + kvh * G + (e - r * G), at = head * a.n_splits;
        const mma_u32x2_t ml = __builtin_bit_cast(mma_u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(
            parts, (int)((heads * a.n_splits * VD + (at + (lane < ranges ? lane : 0u)) * 2u) * 4u), 0, kShared));
        auto merge = [&](auto count) {
            constexpr uint32_t N = decltype(count)::value / SPR;
            mma_u32x4_t po[N];
#pragma unroll
            for (uint32_t i = 0; i < N; ++i) {
                const uint32_t s = i * SPR + lane / LP;
                po[i] = __builtin_bit_cast(mma_u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                    parts, (int)(((at + (s < ranges ? s : 0u)) * VD + (lane % LP) * 4u) * 4u), 0, kShared));
            }
            __builtin_amdgcn_sched_barrier(0);
            const float m = lane < ranges ? __uint_as_float(ml[0]) : -INFINITY, M = wave_max(m);
            const float w_mine = __builtin_amdgcn_exp2f(m - (M == -INFINITY ? 0.f : M));
            const float L = wave_sum(lane < ranges ? __uint_as_float(ml[1]) * w_mine : 0.f);
            float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (uint32_t i = 0; i < N; ++i) {
                const uint32_t s = i * SPR + lane / LP;
                const float w = __int_as_float(__builtin_amdgcn_ds_bpermute((int)(s * 4u), __float_as_int(w_mine)));
#pragma unroll
                for (int c = 0; c < 4; ++c) o[c] = s < ranges ? fmaf(__uint_as_float(po[i][c]), w, o[c]) : o[c];
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {   // the partials that a request brought side by side
                const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[c]), __float_as_uint(o[c]), false, false);
                o[c] = __uint_as_float(h[0]) + __uint_as_float(h[1]);
                if constexpr (SPR == 4) {
                    const auto f = __builtin_amdgcn_permlane16_swap(__float_as_uint(o[c]), __float_as_uint(o[c]), false, false);
                    o[c] = __uint_as_float(f[0]) + __uint_as_float(f[1]);
                }
            }
            if (lane < LP)
                *reinterpret_cast<uint2*>(a.out + (size_t)head * VD + lane * 4u) = make_uint2(pack_bf16(o[0] / L, o[1] / L), pack_bf16(o[2] / L, o[3] / L));
        };
        if (ranges <= 16u) merge(std::integral_constant<uint32_t, 16>{});
        else if (ranges <= 32u) merge(std::integral_constant<uint32_t, 32>{});
        else merge(std::integral_constant<uint32_t, kMmaMaxSplits>{});
    }
}

namespace {

template <int QK, int VD, int QT, int NW, MmaForm FORM = MMA_PLAIN>
fk_status fill(Launch* l) {
    l->func = reinterpret_cast<const void*>(&sdpa_mma_kernel<QK, VD, QT, NW, FORM>);
    l->block = dim3(NW * 64, 1, 1);
    l->shmem = mma_lds_bytes(QK, VD, QT, NW, FORM != MMA_PLAIN);
    return raise_dynamic_lds(l->func, l->shmem);
}
template <int DIM, int QT, int NW>
fk_status fill(Launch* l, MmaForm form) {
    return form == MMA_PLAIN ? fill<DIM, DIM, QT, NW>(l) : (form == MMA_FUSED ? fill<DIM, DIM, QT, NW, MMA_FUSED>(l) : fill<DIM, DIM, QT, NW, MMA_STAGED>(l));
}

}  // namespace

bool sdpa_takes_mma(const uint16_t* q, const uint16_t* k, const uint16_t* v, const uint16_t* out, uint32_t n_heads, uint32_t n_kv,
                    uint32_t qk_dim, uint32_t v_dim, uint32_t max_len, uint32_t rows, const float* partials, const uint32_t* counters) {
    if (!((qk_dim == v_dim && (qk_dim == 64 || qk_dim == 128)) || (qk_dim == 192 && v_dim == 128 && rows > 1))) return false;
    if (!partials || !counters) return false;
    // (by what a launch with the rotation and the append shares with the launch pair that it equals bit for bit, and nothing else)
    if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out | (uintptr_t)partials) & 15u) return false;
    // The lines are in the length that the launch is planned for, which the host knows; in a graph that is the capacity, and shorter contexts come
    // along.  Those of one range of the vector form (64 positions of 128 dims, 128 of 64) are the slower for it, longer ones the faster, us, that
    // / this: plans of 256, 32 / 8 heads x 128, 50 positions 3.2 / 4.5, 100 5.8 / 4.7, 150 6.1 / 5.0, 256 6.3 / 5.3; of 1024, 50 3.2 / 4.4, 100 4.1 / 4.5,
    // 600 7.6 / 6.9, 1024 8.4 / 7.3; of 4096, 50 3.8 / 4.5, 1000 10.0 / 7.8; 14 / 2 x 64, of 1024, 50 3.2 / 3.9, 300 6.1 / 5.8, 1024 6.9 / 6.3; of 12000, 200
    // 4.8 / 4.1; 8 rows of 32 / 8 x 128, of 1024, 30 4.2 / 5.8, 300 8.0 / 7.9, 1000 15.1 / 10.0.  A cache that fills meets the first for 64 (128)
    // tokens of its hundreds and more.
    // Short contexts of few rows: the form on vector instructions has less to set up (us, that / this: 32 / 8 heads x 128, 64 positions 4.0 / 4.7, 128
    // 4.9 / 4.9, 256 6.8 / 6.6, 8 rows at 100 4.3 / 6.6, 64 rows at 100 14.7 / 8.1; 14 / 2 x 64, 128 positions 4.1 / 4.1, 256 5.1 / 4.5; 16 heads of
    // 192 / 128, 8 rows at 30 5.4 / 6.1, 2 rows at 100 7.6 / 6.2).
    if (max_len <= (qk_dim == 192 ? 64u : 192u) && (uint64_t)n_heads * rows <= 512u) return false;
    // One row of 128 dims beyond the one round of a block: the partials, their count and their merge come with either form, and the vector form's
    // blocks, four times as many, have the shorter way until a block of it walks two or three ranges (caches from memory, that / this: 32 / 8
    // heads, 300 positions 5.5 / 6.5, 700 6.9 / 7.0, 900 7.4 / 7.2; 16 / 4, 600 6.4 / 6.5, 700 6.6 / 6.5; 8 / 2, 900 6.0 / 6.4, 1500 7.0 / 6.4; a head a
    // KV head, 8, 1100 7.0 / 7.2, 1500 7.8 / 7.5; groups of more than four, whose tiles of 8 this form fills in part: 14 / 2, 1500 7.4 / 7.9, 2100 9.0 / 8.7;
    // 32 / 4, 1500 8.5 / 9.0, 2100 9.5 / 9.1; 56 / 8, 1100 8.9 / 9.0, 1500 9.6 / 9.1).
    const uint32_t group = n_heads / n_kv;
    const uint32_t line = group > 4u ? (n_heads <= 32u ? 1792u : 1088u) : (group == 1u ? 1280u : (n_heads <= 8u ? 1024u : 704u));
    if (qk_dim == 128 && rows == 1 && max_len > 256u && max_len <= line) return false;
    // (partials are addressed with 32 bits)
    return (uint64_t)rows * n_heads * kMmaMaxSplits * (v_dim + 2u) * 4u < 0x7fffffffull;
}

fk_status plan_sdpa_mma(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* out, const uint32_t* kv_len_ptr, uint32_t kv_len_imm,
                        uint32_t max_len, uint32_t n_heads, uint32_t n_kv, uint32_t qk_dim, uint32_t v_dim, uint32_t capacity, float scale,
                        float* partials, uint32_t* counters, uint32_t rows, const SdpaFusion* fusion, Launch* l) {
    const DeviceFacts* dev;
    FK_TRY(device_facts(&dev));
    SdpaMmaStagedArgs a;
    memset(&a, 0, sizeof(a));
    a.q = q; a.k = k; a.v = v; a.out = out;
    a.kv_len_ptr = kv_len_ptr; a.kv_len_imm = kv_len_imm;
    a.n_heads = n_heads; a.group = n_heads / n_kv; a.capacity = capacity;
    a.rows = rows; a.scale = scale; a.partials = partials; a.counters = counters;
    MmaForm form = MMA_PLAIN;
    if (fusion) {
        a.k_new = fusion->k_new; a.v_new = fusion->v_new; a.q_norm = fusion->q_norm; a.k_norm = fusion->k_norm;
        a.cache_k_w = const_cast<uint16_t*>(k); a.cache_v_w = const_cast<uint16_t*>(v);
        a.rope_dims = fusion->rope_dims; a.eps = fusion->eps; a.base_log2 = fusion->base_log2; a.rope_tab = fusion->rope_tab;
        a.k1_new = fusion->k1_new; a.q0_dim = fusion->q0_dim; a.k1_heads = fusion->k1_heads; a.traditional = fusion->traditional;
        a.k0_stride = fusion->q0_dim ? fusion->k0_stride : qk_dim;
        a.v_stride = fusion->q0_dim ? fusion->v_stride : v_dim;
        // requests of sixteen bytes take whole heads, a table of whole pieces and aligned addresses
        const uintptr_t at = (uintptr_t)a.k_new | (uintptr_t)a.v_new | (uintptr_t)a.q_norm | (uintptr_t)a.k_norm | (uintptr_t)a.rope_tab;
        form = (at & 15u) || a.q0_dim || (a.rope_tab && a.rope_dims % 4u) ? MMA_STAGED : MMA_FUSED;
    }
    // Tiles of 4 queries put the three parts of the probabilities into one matrix instruction's columns, of 8 into two instructions, of 16
    // into three.  More than 8 queries: tiles of 8 while there is a CU for each (of 16 / 8, us: 32 / 8 heads x 128, 3 rows at 500 positions 10.2 /
    // 7.0, 64 rows 13.7 / 8.4, 128 rows -- 512 tiles -- 12.4 / 15.1; 16 heads of 192 / 128, 32 rows at 480 positions 10.9 / 8.8).
    const uint32_t queries = rows * a.group;
    const uint32_t qt = queries <= 4u ? 4u : (queries <= 8u || rows == 1u || (uint64_t)n_kv * ((queries + 7u) / 8u) <= (uint64_t)dev->cus ? 8u : 16u);
    // Waves, and the rounds of theirs that one block walks rather than leave partials.  A block draws 90 bytes a ns where its rows lie in the
    // L2, half of that where they come from memory; partials, their count and their merge take 2.2 us.  Cold caches, us: 64 dims (256
    // positions a round), one block / several, 544 positions 5.5 / 6.2, 1024 6.5 / 6.5 (16 / 8 heads 6.4 / 6.4, 8.1 / 6.5).  One row of 128 dims: at
    // 256 positions one round of 8 waves 6.6, two of 4 7.4; beyond, 32 KB a wave in fewer CUs is the slower, until the rounds are many:
    // 8 / 4 waves, 512 8.5 / 7.4, 1024 8.6 / 7.8, 2048 8.9 / 8.5, 4096 9.9 / 10.1, 12000 14.6 / 14.9; tiles of 8 are the slower with 4 at every
    // length (warm, 14 / 2 heads, 480 8.2 / 9.7, 2500 8.5 / 10.7).  Several rows share what is drawn: 8 of them
    // at 500 positions, 8 waves in one block 8.6, 4 in four 9.2.  (Two steps of a wave in flight at half the waves: 64 dims 544 5.8, 12000 8.5.)
    uint32_t nw = 8, alone = rows > 1 ? 2u : 1u;
    if (qk_dim == 64) {
        alone = 3;
        FK_TRY(qt == 4 ? (fill<64, 4, 8>(l, form)) : (qt == 8 ? fill<64, 8, 8>(l, form) : fill<64, 64, 16, 8>(l)));
    } else if (qk_dim == 128) {
        if (qt == 16) {
            nw = 4;
            alone = 4;
            FK_TRY((fill<128, 128, 16, 4>(l)));
        } else if (rows == 1 && qt == 4u && max_len > 256u && max_len <= 3072u) {
            nw = 4;
            FK_TRY((fill<128, 4, 4>(l, form)));
        } else {
            FK_TRY(qt == 4 ? (fill<128, 4, 8>(l, form)) : (fill<128, 8, 8>(l, form)));
        }
    } else if (qt <= 8) {
        nw = 7;   // (160 KB)
        alone = 3;
        FK_TRY(qt == 4 ? (fill<192, 128, 4, 7>(l)) : (fill<192, 128, 8, 7>(l)));
    } else {
        nw = 4;
        alone = 4;
        FK_TRY((fill<192, 128, 16, 4>(l)));
    }
    // Beyond that a block a CU, but no shorter than two rounds where there would be more than the 16 partials that a merge has soonest.
    const uint32_t tiles = (queries + qt - 1u) / qt, round = nw * kMmaStep, rounds = (max_len + round - 1u) / round;
    uint32_t want = (uint32_t)dev->cus / (n_kv * tiles), many = (rounds + 1u) / 2u;
    many = many < 16u ? 16u : (many > kMmaMaxSplits ? kMmaMaxSplits : many);
    want = want > many ? many : want;
    if (want < 1u || rounds <= alone) want = 1;
    const uint32_t per = (rounds + want - 1u) / want;
    a.span = per * round;
    a.n_splits = (max_len + a.span - 1u) / a.span;
    l->grid = dim3(a.n_splits, n_kv, tiles);
    if (form == MMA_STAGED) l->set_args(a);
    else l->set_args(static_cast<const SdpaMmaArgs&>(a));
    return FK_OK;
}

}  // namespace fk
