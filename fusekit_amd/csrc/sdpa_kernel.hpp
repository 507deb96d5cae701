// Device side of the split-K attention decode: SdpaArgs, the per-work-item
// function sdpa_block and the stand-alone kernel.  See sdpa.hip for the scheme.
#pragma once
#include <stddef.h>

#include <type_traits>

#include "fk_device.hpp"
#include "kv_quant_device.hpp"
#include "rope_device.hpp"

// Hook for timing probes: a build may define FK_SDPA_STAMP(i) to record a clock at
// phase boundary i; the library build leaves it empty.
#ifndef FK_SDPA_STAMP
#define FK_SDPA_STAMP(i)
#endif

namespace fk {

constexpr int kSdpaBlock = 256;
constexpr int kSdpaWaves = kSdpaBlock / kWave;
constexpr int kSdpaSteps = 4;       // K rows (and at most as many V rows) each lane owns per range
constexpr int kSdpaStepsFused = 4;  // inside the whole-token kernel: half the registers, twice the ranges

struct SdpaArgs {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    uint16_t* out;
    const uint32_t* kv_len_ptr;  // device scalar, or null -> kv_len_imm
    uint32_t kv_len_imm;
    uint32_t n_heads, n_kv, qk_dim, v_dim, capacity;
    uint32_t chunk_len, n_splits;
    uint32_t chunks_per_block;  // consecutive ranges one block walks (online softmax across them)
    uint32_t rows;              // active token rows (stand-alone kernel): row r attends to kv_len + r positions
    // Quantised cache (stand-alone kernel, KVQ = 4 or 8): k / v point at packed uint32
    // [n_kv, capacity, dim * bits / 32]; scales / biases are bf16 [n_kv, capacity, dim / kv_group].
    const uint16_t* k_scales;
    const uint16_t* k_biases;
    const uint16_t* v_scales;
    const uint16_t* v_biases;
    uint32_t kv_group;
    uint32_t lpk, lpv;  // lanes per key row / value row (powers of two)
    float scale;
    float* partials;     // [n_heads][n_splits][v_dim + 2]
    uint32_t* counters;  // [n_kv * head tiles], zero before the first launch
    // Fused mode (the whole-token kernel): q, k_new, v_new are the raw projection
    // outputs of this token at position kv_len - 1.  Every block transforms its q
    // heads itself (head norm + RoPE); the block whose range holds the new position
    // transforms k_new, uses it and v_new in place of the cache row and writes both
    // into the cache.
    const uint16_t* k_new;
    const uint16_t* v_new;
    const uint16_t* q_norm;
    const uint16_t* k_norm;
    uint16_t* cache_k_w;
    uint16_t* cache_v_w;
    uint32_t rope_dims;
    float eps, base_log2;
    const float* rope_tab;  // (cos, sin) per pair at this token's position, or null
    // Heads given as two parts (low-rank keys): q0_dim != 0 means q = [Q0 | Q1] with the first rope_dims of
    // Q1 rotated, the new key row = [k_new row (k0_stride apart) | k1_new (one shared head or one per KV
    // head)] with the same rotation on its second part, v_new rows v_stride apart (both may point into one
    // packed projection output); no head norm in this form.
    const uint16_t* k1_new;
    uint32_t q0_dim, k0_stride, v_stride, k1_heads, traditional;
};

// m[GT] at 0, l[GT] at 8 (GT <= 8), the last-block flag at 16, the per-range rescale factors at 24;
// wave-local form: per-wave maxima [wave][8] at 32 and per-wave sums [wave][8] at 64.
constexpr uint32_t kSdpaStatFloats = 96;

// The new row of a quantised cache in the block that appends it, floats behind the transformed heads: the rows in fp32, their
// packed words, scale | bias << 16 per group, their codes as bytes.
__host__ __device__ inline uint32_t sdpa_quant_row_floats(uint32_t qk_dim, uint32_t v_dim) { return 2u * (qk_dim + v_dim); }

// LDS floats one block needs.
__host__ __device__ inline uint32_t sdpa_lds_floats(uint32_t gt, uint32_t chunk, uint32_t qk_dim, uint32_t v_dim,
                                                     bool fused, bool quant = false) {
    uint32_t lpv = 1;
    while (lpv < v_dim / 8) lpv <<= 1;
    const uint32_t slots = kSdpaBlock / lpv;  // key rows handled side by side in the value phase
    return gt * chunk + slots * gt * v_dim + kSdpaStatFloats + (fused ? (gt + 1) * qk_dim / 2 + 8 : 0) +
           (fused && quant ? sdpa_quant_row_floats(qk_dim, v_dim) : 0);
}

// f(0), ... f(N - 1) with constant arguments.
template <int N, typename F, int I = 0>
__device__ __forceinline__ void each_index(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        each_index<N, F, I + 1>(static_cast<F&&>(f));
    }
}
// Lane J of the caller's 16-lane row (row_newbcast).
template <int J>
__device__ __forceinline__ uint32_t row_lane(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + J, 0xF, 0xF, false); }
// Lane J of the caller's half of a 16-lane row.
template <int J>
__device__ __forceinline__ uint32_t half_row_lane(uint32_t v) {
    const int low = __builtin_amdgcn_update_dpp(0, (int)v, 0x150 + J, 0xF, 0x3, false);
    return (uint32_t)__builtin_amdgcn_update_dpp(low, (int)v, 0x158 + J, 0xF, 0xC, false);
}

// One (range, kv head, head tile) work item.  Uniform per block; `kv_len` already read.
// MODE 0: q is already rotated and the new K/V rows are in the cache.  MODE 1: a phase of the
// whole-token kernel (kv_len known on entry, coherent stores); MODE 2: a kernel of its own.  In
// modes 1 and 2 the block applies head norm + RoPE to its q heads itself, and the block whose
// range holds the new position does the same for the new k row, uses it and v_new in place of
// the cache row and appends both to the cache.
// FASTHEAD (mode 2): heads rotated over their whole width of at most 128 dims with a rotary table;
// the transforms' loads are issued ahead of the cache rows and used after them.
// NOMERGE: the caller merges the ranges' results itself: every active block writes its (m, l, o) partial with
// ordinary stores -- also when one range covers the context -- and returns; no arrival counter is touched.
// ROW: 16, heads of 128 dims for keys and values, a row on 16 lanes; 8, heads of 64 dims on 8 (a quantised cache: groups of 64,
// with 128 dims scale and bias arrays 4-byte aligned); else 0.  See the wave-local form below.
template <int GT, int MODE, typename ARGS, int KVQ = 0, bool FASTHEAD = false, bool NOMERGE = false, int ROW = 0>
__device__ __forceinline__ void sdpa_block(const ARGS& a, uint32_t kv_raw, uint32_t split, uint32_t kvh,
                                           uint32_t gz, uint32_t gz_count, float* lds, uint32_t kv_add = 0) {
    // kv_raw + kv_add positions are visible (kv_add: the row's index among several active rows).  The sum is formed
    // inside settle(), behind the points where the length is first allowed to be looked at: formed by the caller, it
    // is a use of the loaded length at the very top of the kernel.
    uint32_t kv_len = 0;
    constexpr bool FUSED = MODE == 1;   // inside the whole-token kernel
    constexpr bool XFORM = MODE != 0;   // q / new-row transforms happen here
    // Tiles of up to 4 heads outside the whole-token kernel: every wave runs the online softmax
    // over its own 16 keys of a range in registers (scores never leave the lanes that computed
    // them, a key row and its value row share their lanes: the planner guarantees lpk == lpv), so
    // the ranges of a block need no barrier; the waves meet once, after the last range.
    constexpr bool WAVES = MODE != 1 && GT <= 4;
    constexpr int kSteps = FUSED ? kSdpaStepsFused : kSdpaSteps;
    static_assert(ROW == 0 || (MODE != 1 && kSteps == 4), "");
    static_assert(!(FUSED && KVQ != 0), "the whole-token kernel reads a bf16 cache");
    const uint32_t span = a.chunk_len * a.chunks_per_block;  // cache positions per block
    const uint32_t blk0 = split * span;
    const uint32_t G = a.n_heads / a.n_kv;
    const uint32_t h0 = kvh * G + gz * GT;
    const uint32_t gcount = (G - gz * GT) < (uint32_t)GT ? (G - gz * GT) : (uint32_t)GT;
    // Stand-alone kernel: kv_len is still on its way from memory (a scalar load the
    // caller issued); nothing below touches it until the first K/V rows have been
    // requested, so that round trip overlaps the cache reads.
    uint32_t n_active = 0, blk_keys = 0, n_chunks = 0;
    uint32_t pos = 0;  // fused: position of the new token
    auto settle = [&]() {
        // a device scalar is not trusted: a length beyond what the launch was sized for would leave ranges
        // without a block (the last-arrival count would never complete), zero would divide by an empty sum
        const uint32_t covered = a.n_splits * span < a.capacity ? a.n_splits * span : a.capacity;
        const uint32_t given = kv_raw + kv_add;
        kv_len = given < 1u ? 1u : (given > covered ? covered : given);
        pos = XFORM ? kv_len - 1 : 0u;
        n_active = (kv_len + span - 1) / span;
        if (split < n_active) {
            blk_keys = (kv_len - blk0) < span ? (kv_len - blk0) : span;
            n_chunks = (blk_keys + a.chunk_len - 1) / a.chunk_len;
        }
    };
    if constexpr (FUSED) {
        settle();
        if (split >= n_active) return;  // uniform: whole block leaves before any barrier
    }
    const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    FK_SDPA_STAMP(0);

    float* s = lds;                               // [GT][chunk_len]
    float* red = s + GT * a.chunk_len;            // [value slots][GT][v_dim]
    float* stat = red + (kSdpaBlock / a.lpv) * GT * a.v_dim;  // m[GT], l[GT], misc
    uint16_t* qn = reinterpret_cast<uint16_t*>(stat + kSdpaStatFloats);  // fused: [GT][qk_dim] + k row
    uint16_t* kn = qn + GT * a.qk_dim;
    // quantised cache: the new K and V rows (k, then v): fp32, packed words, scale | bias << 16 of a group, codes
    float* nrow = reinterpret_cast<float*>(kn + a.qk_dim);
    uint32_t* nword = reinterpret_cast<uint32_t*>(nrow + a.qk_dim + a.v_dim);
    uint32_t* nmeta = nword + (a.qk_dim + a.v_dim) / 4u;
    uint8_t* ncode = reinterpret_cast<uint8_t*>(nmeta + (a.qk_dim + a.v_dim) / 32u);
    bool blk_owner = false;

    // Head norm + RoPE of this block's q heads (one wave per head), and of the new k row
    // in the block that owns its position; results in LDS as bf16.  Then one block per kv
    // head appends the new rows to the cache.
    auto head_dst = [&](uint32_t h) { return h < gcount ? qn + h * a.qk_dim : kn; };
    auto transform_heads = [&](uint32_t h_first) {
        blk_owner = pos >= blk0 && pos < blk0 + blk_keys;
        if constexpr (KVQ != 0) {
            if (blk_owner && wave < 2u) {   // wave 0 the key, wave 1 the value; the first head tile's block writes them to the cache
                const bool is_v = wave != 0u;
                const uint32_t dim = is_v ? a.v_dim : a.qk_dim, at = is_v ? a.qk_dim : 0u, bits = (uint32_t)KVQ, groups = dim / a.kv_group;
                float* row = nrow + at;
                uint32_t *word = nword + at / 4u, *meta = nmeta + at / 32u;
                uint8_t* code = ncode + at;
                if (is_v)
                    for (uint32_t d = lane; d < dim; d += kWave) row[d] = bf16_bits_to_f32(a.v_new[(size_t)kvh * dim + d]);
                else
                    kv_key_row(a.k_new + (size_t)kvh * dim, a.k_norm, row, dim, a.rope_dims, pos, a.base_log2, a.eps, lane, a.rope_tab);
                const size_t crow = (size_t)kvh * a.capacity + (pos % a.capacity);
                uint32_t* packed = reinterpret_cast<uint32_t*>(const_cast<uint16_t*>(is_v ? a.v : a.k)) + crow * (dim * bits / 32u);
                uint16_t* scales = const_cast<uint16_t*>(is_v ? a.v_scales : a.k_scales) + crow * groups;
                uint16_t* biases = const_cast<uint16_t*>(is_v ? a.v_biases : a.k_biases) + crow * groups;
                wave_lds_order();
                kv_quantize_row(row, code, dim, a.kv_group, bits, lane, [&](uint32_t g, uint32_t sc, uint32_t bi) {
                    meta[g] = sc | (bi << 16);
                    if (gz == 0) {
                        scales[g] = (uint16_t)sc;
                        biases[g] = (uint16_t)bi;
                    }
                });
                wave_lds_order();
                kv_pack_row(code, dim, bits, lane, [&](uint32_t wi, uint32_t w) {
                    word[wi] = w;
                    if (gz == 0) packed[wi] = w;
                });
            }
        }
        for (uint32_t h = h_first + wave; h < gcount + (blk_owner && KVQ == 0 ? 1u : 0u); h += kSdpaWaves) {
            if (a.q0_dim) {
                const uint32_t d1 = a.qk_dim - a.q0_dim;
                if (h < gcount) {
                    const uint16_t* qh = a.q + (size_t)(h0 + h) * a.qk_dim;
                    split_head_transform(qh, qh + a.q0_dim, head_dst(h), a.q0_dim, d1, a.rope_dims, a.traditional != 0, pos,
                                         a.base_log2, lane, a.rope_tab);
                } else {
                    split_head_transform(a.k_new + (size_t)kvh * a.k0_stride, a.k1_new + (size_t)(a.k1_heads == 1 ? 0 : kvh) * d1,
                                         kn, a.q0_dim, d1, a.rope_dims, a.traditional != 0, pos, a.base_log2, lane, a.rope_tab);
                }
            } else if (h < gcount) {
                head_transform(a.q + (size_t)(h0 + h) * a.qk_dim, head_dst(h), a.q_norm, a.qk_dim, a.rope_dims,
                               pos, a.base_log2, a.eps, true, lane, a.rope_tab);
            } else {
                head_transform(a.k_new + (size_t)kvh * a.qk_dim, kn, a.k_norm, a.qk_dim, a.rope_dims, pos, a.base_log2,
                               a.eps, true, lane, a.rope_tab);
            }
        }
        __syncthreads();
        if (KVQ == 0 && blk_owner && gz == 0) {
            const size_t row = (size_t)kvh * a.capacity + (pos % a.capacity);
            for (uint32_t d = tid; d < a.qk_dim; d += kSdpaBlock) a.cache_k_w[row * a.qk_dim + d] = kn[d];
            for (uint32_t d = tid; d < a.v_dim; d += kSdpaBlock)
                a.cache_v_w[row * a.v_dim + d] = a.v_new[(size_t)kvh * (MODE == 2 ? a.v_stride : a.v_dim) + d];
        }
    };
    // Whole-token kernel: done before the K/V loads are issued: the trigonometry needs
    // ~60 registers that the 64 registers of in-flight rows would otherwise have to share.
    if constexpr (MODE == 1) transform_heads(0);

    const uint32_t lpk = ROW ? (uint32_t)ROW : a.lpk, cpk = ROW ? (uint32_t)ROW : a.qk_dim >> 3;
    const uint32_t lpv = ROW ? (uint32_t)ROW : a.lpv, cpv = ROW ? (uint32_t)ROW : a.v_dim >> 3;
    const uint32_t ck = tid & (lpk - 1), kslot = tid / lpk, kslots = kSdpaBlock / lpk;
    const uint32_t cv = tid & (lpv - 1), vslot = tid / lpv, vslots = kSdpaBlock / lpv;
    const bool kcol_ok = ck < cpk, vcol_ok = cv < cpv;

    // Running softmax state per head (m, l) in LDS; the value accumulators stay in
    // registers across ranges: a lane owns the same 8 output dims in every range.
    if (tid < (uint32_t)GT) {
        stat[tid] = -INFINITY;
        stat[8 + tid] = 0.f;
    }
    float m_own = -INFINITY;     // ROW: running maximum of the head whose score the lane finishes
    float m_run[GT], l_run[GT];  // wave-local form: running maximum (uniform) and this lane row's share of the sum
#pragma unroll
    for (int h = 0; h < GT; ++h) {
        m_run[h] = -INFINITY;
        l_run[h] = 0.f;
    }
    float acc[GT][8];
    float accb[GT];  // quantised V: sum_j p_j * bias_j of this lane's group, added to its 8 dims at the end
#pragma unroll
    for (int h = 0; h < GT; ++h) {
        accb[h] = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[h][i] = 0.f;
    }

    // This lane's 8 dims of each query head; fetched before the K/V rows so that the
    // scores can start as soon as the first keys arrive (loads return in order).
    // The request is straight-line (a lane past the head width or a head past the tile reads a valid address and
    // is zeroed afterwards): with the load under a condition the compiler waits for it where the paths join, i.e.
    // before the K/V rows are requested -- a whole trip to memory at the start of every block.  settle_q zeroes the
    // unused lanes and derives what the quantised forms need; it runs behind the first K/V request.
    uint4 qf[GT];
    float sq[GT];  // quantised K: sum of this lane's 8 query dims (the affine bias term b * sum q)
    auto load_q = [&]() {
#pragma unroll
        for (int h = 0; h < GT; ++h) {
            const uint32_t hc = (uint32_t)h < gcount ? (uint32_t)h : 0u, cc = kcol_ok ? ck : 0u;
            if constexpr (XFORM)
                qf[h] = *reinterpret_cast<const uint4*>(qn + hc * a.qk_dim + 8 * cc);
            else
                qf[h] = *reinterpret_cast<const uint4*>(a.q + (size_t)(h0 + hc) * a.qk_dim + 8 * cc);
        }
    };
    auto settle_q = [&]() {
#pragma unroll
        for (int h = 0; h < GT; ++h) {
            pin_u128(qf[h]);  // looked at only from here on
            if (!(kcol_ok && (uint32_t)h < gcount)) qf[h] = make_uint4(0, 0, 0, 0);
            if constexpr (KVQ != 0) {
                const uint4 v = qf[h];
                sq[h] = ((bf16_lo(v.x) + bf16_hi(v.x)) + (bf16_lo(v.y) + bf16_hi(v.y))) +
                        ((bf16_lo(v.z) + bf16_hi(v.z)) + (bf16_lo(v.w) + bf16_hi(v.w)));
                if constexpr (KVQ == 4)  // nibble pairing of q4_word_dot: (x0,x2) (x4,x6) (x1,x3) (x5,x7)
                    qf[h] = make_uint4((v.x & 0xffffu) | (v.y << 16), (v.z & 0xffffu) | (v.w << 16),
                                       (v.x >> 16) | (v.y & 0xffff0000u), (v.z >> 16) | (v.w & 0xffff0000u));
            }
        }
    };
    if constexpr (MODE != 2) load_q();
    if constexpr (MODE == 1) settle_q();  // whole-token kernel: q comes from LDS, its rows are requested per range

    // All K and V loads of a range are issued up front (the range is sized so that
    // each lane owns kSteps rows of each), so one HBM round trip covers both phases.
    // Stand-alone: every row that exists in the cache allocation is requested, whether
    // or not it is below kv_len (rows past kv_len are masked where they are used).
    uint4 kc[kSteps], vc[kSteps];
    // Stand-alone: the next range, in flight while this one is consumed; of a quantised cache, whose ranges are a quarter to a
    // half of the bytes, the one behind it too (12016 positions of an 8-bit cache, three ranges a block, cold: the last range
    // starts 8.8 us into the launch instead of 13.6; a bf16 cache is bound by the bytes and was 5 % slower with it).
    constexpr bool DEEP = MODE != 1 && WAVES && KVQ != 0;
    uint4 kn_[kSteps], vn_[kSteps], kf_[DEEP ? kSteps : 1], vf_[DEEP ? kSteps : 1];
    // Quantised, ROW: scales and biases of a range with one request a wave (128 dims: lane 4 u + i of a row's 16 holds both groups'
    // entries of key row u in array i: scales and biases of the keys, of the values) or two (64 dims: lane 2 u + i of a row's 8
    // the scale and the bias of key row u of the keys, of the values) -- two bytes a lane from each array and row they were 16
    // of its 24, and a CU issues one in 16 .. 20 cycles.
    constexpr bool META = ROW != 0 && KVQ != 0;
    struct Meta {
        uint32_t a, b;   // (64 dims: the scale and the bias, put together where they are used: not a wait at the request)
    };
    Meta mc = {0u, 0u}, mn_ = {0u, 0u}, mf_ = {0u, 0u};
    // (global accesses: chosen among the arguments' pointers as they are, the arguments move to memory and the access is a flat one)
    typedef const __attribute__((address_space(1))) uint32_t* gmeta32;
    typedef const __attribute__((address_space(1))) uint16_t* gmeta16;
    uintptr_t mbase = 0, mbase2 = 0;
    if constexpr (META) {
        const uintptr_t ks = (uintptr_t)a.k_scales, kb = (uintptr_t)a.k_biases, vs = (uintptr_t)a.v_scales, vb = (uintptr_t)a.v_biases;
        if constexpr (ROW == 16) {
            const uintptr_t kk = (lane & 1u) ? kb : ks, vv = (lane & 1u) ? vb : vs;
            mbase = (lane & 2u) ? vv : kk;
        } else {
            mbase = (lane & 1u) ? vs : ks;
            mbase2 = (lane & 1u) ? vb : kb;
        }
    }
    auto request_rows = [&](uint4(&kd)[kSteps], uint4(&vd)[kSteps], Meta& md, uint32_t key0, uint32_t nkeys, bool owner,
                            uint32_t jpos) {
        const uint16_t* kbase = a.k + ((size_t)kvh * a.capacity + key0) * a.qk_dim + 8 * ck;
        const uint16_t* vbase = a.v + ((size_t)kvh * a.capacity + key0) * a.v_dim + 8 * cv;
        if constexpr (KVQ != 0) {
            // 8 dims per lane as in the bf16 layout: one packed word (int4) or two (int8) in
            // .x / .y, the group's scale and bias bits in .z; rows clamped as below.
            constexpr uint32_t WPL = KVQ == 4 ? 1u : 2u;
            const uint32_t kw = a.qk_dim * KVQ / 32u, vw = a.v_dim * KVQ / 32u;
            const uint32_t kg = a.qk_dim / a.kv_group, vg = a.v_dim / a.kv_group;
            const uint32_t kcol = kcol_ok ? ck : 0u, vcol = vcol_ok ? cv : 0u;
            const uint32_t* kp = reinterpret_cast<const uint32_t*>(a.k) + (size_t)kvh * a.capacity * kw + kcol * WPL;
            const uint32_t* vp = reinterpret_cast<const uint32_t*>(a.v) + (size_t)kvh * a.capacity * vw + vcol * WPL;
            const size_t kmeta = (size_t)kvh * a.capacity * kg + (8u * kcol) / a.kv_group;
            const size_t vmeta = (size_t)kvh * a.capacity * vg + (8u * vcol) / a.kv_group;
            const uint32_t last = a.capacity - 1;
            if constexpr (META) {
                const uint32_t r0 = key0 + kslot + (ROW == 16 ? (lane >> 2) & 3u : (lane >> 1) & 3u) * kslots, r = r0 < last ? r0 : last;
                const size_t at = (size_t)kvh * a.capacity + r;
                if constexpr (ROW == 16) {
                    md.a = ((gmeta32)mbase)[at];
                } else {
                    md.a = ((gmeta16)mbase)[at];
                    md.b = ((gmeta16)mbase2)[at];
                }
            }
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                const uint32_t r0 = key0 + kslot + u * kslots, r = r0 < last ? r0 : last;
                kd[u].x = kp[(size_t)r * kw];
                kd[u].y = WPL == 2 ? kp[(size_t)r * kw + 1] : 0u;
                kd[u].z = META ? 0u : (uint32_t)a.k_scales[kmeta + (size_t)r * kg] | ((uint32_t)a.k_biases[kmeta + (size_t)r * kg] << 16);
                kd[u].w = 0u;
            }
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                const uint32_t r0 = key0 + vslot + u * vslots, r = r0 < last ? r0 : last;
                vd[u].x = vp[(size_t)r * vw];
                vd[u].y = WPL == 2 ? vp[(size_t)r * vw + 1] : 0u;
                vd[u].z = META ? 0u : (uint32_t)a.v_scales[vmeta + (size_t)r * vg] | ((uint32_t)a.v_biases[vmeta + (size_t)r * vg] << 16);
                vd[u].w = 0u;
            }
            return;
        }
        if constexpr (MODE != 1) {
            // Straight-line, clamped (row to the last row of the allocation, a lane beyond
            // the head width to column 0): no branch separates the loads, so the compiler
            // can wait for exactly the rows it needs while later requests stay in flight.
            const uint16_t* khead = a.k + (size_t)kvh * a.capacity * a.qk_dim + (kcol_ok ? 8 * ck : 0u);
            const uint16_t* vhead = a.v + (size_t)kvh * a.capacity * a.v_dim + (vcol_ok ? 8 * cv : 0u);
            const uint32_t last = a.capacity - 1;
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                const uint32_t r = key0 + kslot + u * kslots;
                kd[u] = *reinterpret_cast<const uint4*>(khead + (size_t)(r < last ? r : last) * a.qk_dim);
            }
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                const uint32_t r = key0 + vslot + u * vslots;
                vd[u] = *reinterpret_cast<const uint4*>(vhead + (size_t)(r < last ? r : last) * a.v_dim);
            }
            return;
        }
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            const uint32_t j = kslot + u * kslots;
            kd[u] = make_uint4(0, 0, 0, 0);
            if (kcol_ok && j < nkeys && !(owner && j == jpos))
                kd[u] = *reinterpret_cast<const uint4*>(kbase + (size_t)j * a.qk_dim);
        }
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            const uint32_t j = vslot + u * vslots;
            vd[u] = make_uint4(0, 0, 0, 0);
            if (vcol_ok && j < nkeys) {
                const uint16_t* src = vbase + (size_t)j * a.v_dim;
                if (owner && j == jpos) {  // the new row, not yet cached
                    vd[u] = *reinterpret_cast<const uint4*>(a.v_new + (size_t)kvh * a.v_dim + 8 * cv);
                } else {
                    vd[u] = *reinterpret_cast<const uint4*>(src);
                }
            }
        }
    };
    uint4 vnew = make_uint4(0, 0, 0, 0);  // mode 2: this lane's 8 dims of the new V row
    if constexpr (MODE != 1) {
        // Mode 2, fast heads: every wave requests the inputs of two heads (its own index and
        // that plus the wave count; index gcount is the new k row) before the cache rows, so
        // they arrive first and the transforms run while the rows are still in flight.
        HeadPair ha, hb;
        const uint32_t half = a.qk_dim >> 1, hi_a = wave, hi_b = wave + kSdpaWaves;
        if constexpr (MODE == 2 && FASTHEAD) {
            auto src = [&](uint32_t h) {
                return h < gcount ? a.q + (size_t)(h0 + h) * a.qk_dim : a.k_new + (size_t)kvh * a.qk_dim;
            };
            ha = head_pair_fetch(src(hi_a), hi_a < gcount ? a.q_norm : a.k_norm, a.rope_tab, half, lane);
            hb = head_pair_fetch(src(hi_b), hi_b < gcount ? a.q_norm : a.k_norm, a.rope_tab, half, lane);
        }
        // The first range always exists and is requested before kv_len has arrived.  Later
        // ranges wait for it (it was the kernel's first request and is long back by now):
        // a fixed grid sized for the whole cache would otherwise read every range's rows
        // each launch, megabytes of traffic for a context of a few hundred tokens.
        // (kv_len is made opaque at both places where it is first looked at: settle() runs on both paths, and
        // the compiler otherwise computes its common part once, AHEAD of the branch -- the first range's request
        // then waits for the length after all)
        if (split != 0) {
            asm volatile("" : "+v"(kv_raw));
            settle();
            if (split >= n_active) return;
        }
        request_rows(kc, vc, mc, blk0, 0, false, 0);
        if constexpr (MODE == 0) settle_q();
        if constexpr (MODE == 2 && KVQ == 0)
            vnew = *reinterpret_cast<const uint4*>(a.v_new + (size_t)kvh * a.v_stride + (vcol_ok ? 8 * cv : 0u));
        asm volatile("" : "+v"(kv_raw));
        settle();
        if (split >= n_active) return;  // uniform: whole block leaves before any barrier
        if constexpr (MODE == 2) {
            if constexpr (FASTHEAD) {
                const bool own = KVQ == 0 && pos >= blk0 && pos < blk0 + blk_keys;
                head_pair_apply(ha, head_dst(hi_a), a.q_norm != nullptr, half, a.eps, lane,
                                hi_a < gcount || (hi_a == gcount && own));
                head_pair_apply(hb, head_dst(hi_b), a.q_norm != nullptr, half, a.eps, lane,
                                hi_b < gcount || (hi_b == gcount && own));
                transform_heads(2 * kSdpaWaves);  // a ninth head (tile of 8 plus the k row), barrier, cache append
            } else {
                // the transforms' own loads queue behind the cache rows requested above; q comes
                // back from LDS rotated
                transform_heads(0);
            }
            load_q();
            settle_q();
        }
    }

    if constexpr (DEEP)
        if (n_chunks > 1) request_rows(kn_, vn_, mn_, blk0 + a.chunk_len, 0, false, 0);
    for (uint32_t c = 0; c < n_chunks; ++c) {
    const uint32_t key0 = blk0 + c * a.chunk_len;
    const uint32_t nkeys = (kv_len - key0) < a.chunk_len ? (kv_len - key0) : a.chunk_len;
    const bool owner = XFORM && pos >= key0 && pos < key0 + nkeys;
    const uint32_t jpos = pos - key0;
    if constexpr (FUSED) {
        request_rows(kc, vc, mc, key0, nkeys, owner, jpos);
    } else if constexpr (DEEP) {
        if (c + 2 < n_chunks) request_rows(kf_, vf_, mf_, key0 + 2 * a.chunk_len, 0, false, 0);
    } else {
        if (c + 1 < n_chunks) request_rows(kn_, vn_, mn_, key0 + a.chunk_len, 0, false, 0);
    }

    FK_SDPA_STAMP(1);
    uint32_t kz[kSteps], vz[kSteps];   // quantised: scale | bias << 16 of this lane's group of each row
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
        kz[u] = kc[u].z;
        vz[u] = vc[u].z;
    }
    if constexpr (META) {
        const uint32_t half = ck >= 8u ? 0x07060302u : 0x05040100u;   // this lane's group
        const uint32_t both = ROW == 16 ? mc.a : mc.a | (mc.b << 16);
        each_index<kSteps>([&](auto u) __attribute__((always_inline)) {
            constexpr int U = decltype(u)::value;
            if constexpr (ROW == 16) {
                kz[U] = __builtin_amdgcn_perm(row_lane<4 * U + 1>(both), row_lane<4 * U>(both), half);
                vz[U] = __builtin_amdgcn_perm(row_lane<4 * U + 3>(both), row_lane<4 * U + 2>(both), half);
            } else {
                kz[U] = half_row_lane<2 * U>(both);
                vz[U] = half_row_lane<2 * U + 1>(both);
            }
        });
    }
    if constexpr (XFORM) {
        if constexpr (KVQ != 0) {
            if (owner) {
                constexpr uint32_t WPL = KVQ == 4 ? 1u : 2u;
                const uint32_t kcol = kcol_ok ? ck : 0u, vcol = vcol_ok ? cv : 0u;
                const uint32_t *kw = nword + kcol * WPL, *vw = nword + a.qk_dim / 4u + vcol * WPL;
#pragma unroll
                for (int u = 0; u < kSteps; ++u) {
                    if (kslot + u * kslots == jpos) {
                        kc[u].x = kw[0];
                        kc[u].y = kw[WPL - 1u];
                        kz[u] = nmeta[8u * kcol / a.kv_group];
                    }
                    if (vslot + u * vslots == jpos) {
                        vc[u].x = vw[0];
                        vc[u].y = vw[WPL - 1u];
                        vz[u] = nmeta[a.qk_dim / 32u + 8u * vcol / a.kv_group];
                    }
                }
            }
        } else if (owner && kcol_ok) {
#pragma unroll
            for (int u = 0; u < kSteps; ++u)
                if (kslot + u * kslots == jpos) kc[u] = *reinterpret_cast<const uint4*>(kn + 8 * ck);
        }
    }
    // q . k of key row u and head h, complete in every lane of the row
    auto score = [&](int u, int h) {
        float d = 0.f;
        if constexpr (KVQ == 4) {
            d = q4_word_dot(kc[u].x, qf[h], 0.f);
            d = fmaf(bf16_lo(kz[u]), d, bf16_hi(kz[u]) * sq[h]);  // s * sum(q * code) + b * sum(q)
        } else if constexpr (KVQ == 8) {
            const uint32_t w0 = kc[u].x, w1 = kc[u].y;
            d = dot2_bf16(pack_bf16((float)(w0 & 0xffu), (float)((w0 >> 8) & 0xffu)), qf[h].x, d);
            d = dot2_bf16(pack_bf16((float)((w0 >> 16) & 0xffu), (float)(w0 >> 24)), qf[h].y, d);
            d = dot2_bf16(pack_bf16((float)(w1 & 0xffu), (float)((w1 >> 8) & 0xffu)), qf[h].z, d);
            d = dot2_bf16(pack_bf16((float)((w1 >> 16) & 0xffu), (float)(w1 >> 24)), qf[h].w, d);
            d = fmaf(bf16_lo(kz[u]), d, bf16_hi(kz[u]) * sq[h]);
        } else {
            d = dot2_bf16(kc[u].x, qf[h].x, d);
            d = dot2_bf16(kc[u].y, qf[h].y, d);
            d = dot2_bf16(kc[u].z, qf[h].z, d);
            d = dot2_bf16(kc[u].w, qf[h].w, d);
        }
        return d;  // this lane's 8 dims only: scores_of() finishes the dot over the row's lanes
    };
    // All scores of the range: the per-lane dots first, then ONE uniform choice of the row width
    // around the cross-lane sums (a width test inside every sum costs six scalar branches each).
    auto scores_of = [&](float(&d)[kSteps][GT]) {
#pragma unroll
        for (int u = 0; u < kSteps; ++u)
#pragma unroll
            for (int h = 0; h < GT; ++h) d[u][h] = score(u, h);
        auto reduce = [&](auto width) {
#pragma unroll
            for (int u = 0; u < kSteps; ++u)
#pragma unroll
                for (int h = 0; h < GT; ++h) d[u][h] = group_sum(d[u][h], decltype(width)::value);
        };
        if (lpk == 16) reduce(std::integral_constant<int, 16>{});
        else if (lpk == 8) reduce(std::integral_constant<int, 8>{});
        else if (lpk == 32) reduce(std::integral_constant<int, 32>{});
        else if (lpk == 64) reduce(std::integral_constant<int, 64>{});
        else if (lpk == 4) reduce(std::integral_constant<int, 4>{});
        else if (lpk == 2) reduce(std::integral_constant<int, 2>{});
    };
    // This lane's 8 dims of value row u as floats (quantised: the codes; `vs`, `vb` the group's
    // scale and bias).  Rows past kv_len were requested speculatively: their bits may be
    // anything, so they are zeroed.
    auto value = [&](int u, uint32_t j, float(&f)[8], float& vs, float& vb) {
        const bool ok = j < nkeys && vcol_ok;
        if constexpr (KVQ != 0) {
            vs = ok ? bf16_lo(vz[u]) : 0.f;
            vb = ok ? bf16_hi(vz[u]) : 0.f;
            if constexpr (KVQ == 4) {
                const uint32_t even = vc[u].x & 0x0F0F0F0Fu, odd = (vc[u].x >> 4) & 0x0F0F0F0Fu;
                f[0] = (float)(even & 0xffu); f[2] = (float)((even >> 8) & 0xffu);
                f[4] = (float)((even >> 16) & 0xffu); f[6] = (float)(even >> 24);
                f[1] = (float)(odd & 0xffu); f[3] = (float)((odd >> 8) & 0xffu);
                f[5] = (float)((odd >> 16) & 0xffu); f[7] = (float)(odd >> 24);
            } else {
                const uint32_t w0 = vc[u].x, w1 = vc[u].y;
                f[0] = (float)(w0 & 0xffu); f[1] = (float)((w0 >> 8) & 0xffu);
                f[2] = (float)((w0 >> 16) & 0xffu); f[3] = (float)(w0 >> 24);
                f[4] = (float)(w1 & 0xffu); f[5] = (float)((w1 >> 8) & 0xffu);
                f[6] = (float)((w1 >> 16) & 0xffu); f[7] = (float)(w1 >> 24);
            }
        } else {
            vs = 1.f;
            vb = 0.f;
            uint4 vv = (FUSED || ok) ? vc[u] : make_uint4(0, 0, 0, 0);
            if constexpr (MODE == 2) {
                if (owner && j == jpos && vcol_ok) vv = vnew;  // the new row, not yet cached
            }
            f[0] = bf16_lo(vv.x); f[1] = bf16_hi(vv.x); f[2] = bf16_lo(vv.y); f[3] = bf16_hi(vv.y);
            f[4] = bf16_lo(vv.z); f[5] = bf16_hi(vv.z); f[6] = bf16_lo(vv.w); f[7] = bf16_hi(vv.w);
        }
    };

    if constexpr (WAVES) {
        // ---------------- wave-local: scores, online softmax and value sums in registers ----------------
        // Scores and running maxima are kept in base-2 units (scale * log2(e) folded into one
        // multiply), so a probability is one v_exp_f32.
        const float scale2 = a.scale * 1.44269504088896341f;
        float pr[kSteps][GT];
        if constexpr (ROW != 0) {
            // A row's lanes each finish ONE of its 4 GT scores (64 dims and four heads: two; fewer scores than lanes: several the
            // same one): at every step of the butterfly a lane keeps the half of the sums that its own score is in and hands over
            // the other -- the same additions -- then scales it and raises it to a probability alone, where every lane did so for
            // all of them (16 exponentials of a quarter rate for one at four heads), and hands it round.  Score v = u GT + h is
            // that of the lanes with bits (b0 ^ b2, b1 ^ b2, b2 ^ b3, b3) of v, which the row's half mirror and mirror pair as
            // they need be (8 lanes: (b0 ^ b2, b1 ^ b2, b2)).
            // 32 q / 8 kv heads x 128, every lane all scores / this: 32768 positions of a bf16 cache 40.5 / 36.8 us; with the
            // scales' single request a token of the 4B-class model behind 12000 positions of an 8-bit cache 1938 / 1807 us.
            constexpr int LR = ROW == 16 ? 4 : 3;                                                      // log2 of the lanes,
            constexpr int LH = GT == 4 ? 2 : (GT == 2 ? 1 : 0), LV = LH + 2 < LR ? LH + 2 : LR;        // the heads, the scores by lane
            constexpr int R = (kSteps * GT) >> LV;                                                     // scores a lane finishes
            const bool sel[4] = {((lane ^ (lane >> 2)) & 1u) != 0, (((lane >> 1) ^ (lane >> 2)) & 1u) != 0,
                                 ROW == 16 ? (((lane >> 2) ^ (lane >> 3)) & 1u) != 0 : (lane & 4u) != 0, (lane & 8u) != 0};
            float x[kSteps * GT];
#pragma unroll
            for (int u = 0; u < kSteps; ++u)
#pragma unroll
                for (int h = 0; h < GT; ++h) x[u * GT + h] = score(u, h);
            each_index<LR>([&](auto step) __attribute__((always_inline)) {
                constexpr int S = decltype(step)::value, CTRL = S == 0 ? 0xB1 : (S == 1 ? 0x4E : (S == 2 ? 0x141 : 0x140));
                if constexpr (S < LV) {
#pragma unroll
                    for (int i = 0; i < ((kSteps * GT) >> (S + 1)); ++i) {   // (in place: the step leaves half as many sums)
                        const float keep = sel[S] ? x[2 * i + 1] : x[2 * i], give = sel[S] ? x[2 * i] : x[2 * i + 1];
                        x[i] = keep + dpp_move<CTRL>(give);
                    }
                } else {
                    x[0] = dpp_add<CTRL>(x[0]);
                }
            });
            uint32_t own = 0;   // this lane's score, the first
#pragma unroll
            for (int k = 0; k < LV; ++k) own |= sel[k] ? 1u << k : 0u;
            float mine[R], mx = -INFINITY;   // mx of the lane's head: over the row's four keys, then the wave's rows
#pragma unroll
            for (int i = 0; i < R; ++i) {
                mine[i] = kslot + ((own + ((uint32_t)i << LV)) >> LH) * kslots < nkeys ? x[i] * scale2 : -INFINITY;
                mx = fmaxf(mx, mine[i]);
            }
            each_index<4>([&](auto step) __attribute__((always_inline)) {
                constexpr int S = decltype(step)::value, CTRL = S == 0 ? 0xB1 : (S == 1 ? 0x4E : (S == 2 ? 0x141 : 0x140));
                if constexpr ((S >= LH && S < LV) || S >= LR) mx = dpp_max<CTRL>(mx);   // (8 lanes: the neighbouring row's too)
            });
            mx = rows_max(mx);
            const float m_new = fmaxf(m_own, mx), m_ref = m_new == -INFINITY ? 0.f : m_new;   // no live key yet: every term is 2^-inf = 0
            const float alpha_own = __builtin_amdgcn_exp2f(m_own - m_ref);
            float p_own[R];
#pragma unroll
            for (int i = 0; i < R; ++i) p_own[i] = __builtin_amdgcn_exp2f(mine[i] - m_ref);
            m_own = m_new;
            each_index<kSteps * GT>([&](auto v) __attribute__((always_inline)) {
                constexpr int V = decltype(v)::value, W = V & ((1 << LV) - 1);
                constexpr int B3 = ROW == 16 ? (W >> 3) & 1 : 0, B2 = ((W >> 2) & 1) ^ B3, B1 = ((W >> 1) & 1) ^ B2, B0 = (W & 1) ^ B2;
                constexpr int FROM = 8 * B3 + 4 * B2 + 2 * B1 + B0;
                const uint32_t p = (uint32_t)__float_as_int(p_own[V >> LV]);
                pr[V / GT][V % GT] = __int_as_float((int)(ROW == 16 ? row_lane<FROM>(p) : half_row_lane<FROM & 7>(p)));
            });
#pragma unroll
            for (int h = 0; h < GT; ++h) {
                const int bits = __builtin_amdgcn_readlane(__float_as_int(alpha_own), h);   // (lane h: score h)
                const float alpha = __int_as_float(bits);
                float psum = 0.f;
#pragma unroll
                for (int u = 0; u < kSteps; ++u) psum += pr[u][h];
                l_run[h] = fmaf(l_run[h], alpha, psum);
                if (bits != 0x3F800000) {  // the maximum rose (rare after the first ranges)
                    accb[h] *= alpha;
#pragma unroll
                    for (int i = 0; i < 8; ++i) acc[h][i] *= alpha;
                }
            }
        } else {
        scores_of(pr);
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            const bool live = kslot + u * kslots < nkeys;
#pragma unroll
            for (int h = 0; h < GT; ++h) pr[u][h] = live ? pr[u][h] * scale2 : -INFINITY;
        }
        float mx[GT];
#pragma unroll
        for (int h = 0; h < GT; ++h) {
            mx[h] = pr[0][h];
#pragma unroll
            for (int u = 1; u < kSteps; ++u) mx[h] = fmaxf(mx[h], pr[u][h]);
        }
        if (lpk < 16) {  // two or more key rows share a 16-lane row: finish the maximum inside it
#pragma unroll
            for (int h = 0; h < GT; ++h) {
                mx[h] = dpp_max<0xB1>(mx[h]);
                mx[h] = dpp_max<0x4E>(mx[h]);
                mx[h] = dpp_max<0x141>(mx[h]);
                mx[h] = dpp_max<0x140>(mx[h]);
            }
        }
#pragma unroll
        for (int h = 0; h < GT; ++h) {
            // every 16-lane row is uniform now: the wave's maximum is that of lanes 0, 16, 32, 48
            const float r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mx[h]), 0));
            const float r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mx[h]), 16));
            const float r2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mx[h]), 32));
            const float r3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mx[h]), 48));
            const float m_new = fmaxf(fmaxf(m_run[h], fmaxf(r0, r1)), fmaxf(r2, r3));
            const float m_ref = m_new == -INFINITY ? 0.f : m_new;  // no live key yet: every term below is 2^-inf = 0
            const float alpha = __builtin_amdgcn_exp2f(m_run[h] - m_ref);
            float psum = 0.f;
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                pr[u][h] = __builtin_amdgcn_exp2f(pr[u][h] - m_ref);
                psum += pr[u][h];
            }
            l_run[h] = fmaf(l_run[h], alpha, psum);
            m_run[h] = m_new;
            if (alpha != 1.f) {  // the maximum rose (rare after the first ranges)
                accb[h] *= alpha;
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[h][i] *= alpha;
            }
        }
        }
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            float f[8], vs, vb;
            value(u, vslot + u * vslots, f, vs, vb);
#pragma unroll
            for (int h = 0; h < GT; ++h) {
                const float p = pr[u][h];
                const float ps = KVQ != 0 ? p * vs : p;
                if constexpr (KVQ != 0) accb[h] = fmaf(p, vb, accb[h]);
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[h][i] = fmaf(ps, f[i], acc[h][i]);
            }
        }
    } else {
    // ---------------- phase A: scores ----------------
    {
        float d[kSteps][GT];
        scores_of(d);
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            const uint32_t j = kslot + u * kslots;
#pragma unroll
            for (int h = 0; h < GT; ++h)
                if (ck == 0 && j < nkeys) s[h * a.chunk_len + j] = d[u][h] * a.scale;
        }
    }
    FK_SDPA_STAMP(2);
    __syncthreads();
    FK_SDPA_STAMP(3);

    // ---------------- softmax over this range, one wave per head ----------------
    // Online form: the running maximum may rise, in which case what was summed so
    // far is rescaled by alpha = exp(m_old - m_new) (0 for the first range).
    for (uint32_t h = wave; h < gcount; h += kSdpaWaves) {
        float* sh = s + h * a.chunk_len;
        const float m_old = stat[h], l_old = stat[8 + h];
        float m = m_old;
        for (uint32_t j = lane; j < nkeys; j += kWave) m = fmaxf(m, sh[j]);
        m = wave_max(m);
        float l = 0.f;
        for (uint32_t j = lane; j < nkeys; j += kWave) {
            const float p = expf(sh[j] - m);
            sh[j] = p;
            l += p;
        }
        l = wave_sum(l);
        if (lane == 0) {
            const float alpha = c ? expf(m_old - m) : 0.f;
            stat[h] = m;
            stat[8 + h] = c ? fmaf(l_old, alpha, l) : l;
            stat[24 + h] = alpha;
        }
    }
    __syncthreads();

    FK_SDPA_STAMP(4);
    // ---------------- phase B: o = sum_j p_j v_j ----------------
    if (c) {
#pragma unroll
        for (int h = 0; h < GT; ++h) {
            const float alpha = stat[24 + h];
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[h][i] *= alpha;
            accb[h] *= alpha;
        }
    }
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
        const uint32_t j = vslot + u * vslots;
        const uint32_t jj = j < nkeys ? j : 0u;
        const float live = j < nkeys ? 1.f : 0.f;
        float f[8], vs, vb;
        value(u, j, f, vs, vb);
#pragma unroll
        for (int h = 0; h < GT; ++h) {
            const float p = s[h * a.chunk_len + jj] * live;
            const float ps = KVQ != 0 ? p * vs : p;
            if constexpr (KVQ != 0) accb[h] = fmaf(p, vb, accb[h]);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[h][i] = fmaf(ps, f[i], acc[h][i]);
        }
    }
    }
    if (c + 1 < n_chunks) {
        if constexpr (!WAVES) __syncthreads();  // the scores are overwritten by the next range
        if constexpr (MODE != 1) {
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                kc[u] = kn_[u];
                vc[u] = vn_[u];
                if constexpr (DEEP) {
                    kn_[u] = kf_[u];
                    vn_[u] = vf_[u];
                }
            }
            mc = mn_;
            mn_ = mf_;
        }
    }
    }  // ranges of this block
    FK_SDPA_STAMP(5);

    if constexpr (WAVES) {
        // The waves meet: maxima and sums through LDS, every wave rescales its value sums to the block's
        // maximum (exp(-inf) = 0 for a wave that saw no live key).
        float* wm = stat + 32;
        float* wl = stat + 64;
        const float inv_lanes = 1.0f / (float)lpk;  // a row's sum is held by each of its lpk lanes (power of two: exact)
#pragma unroll
        for (int h = 0; h < GT; ++h) {
            const float lw = wave_sum(l_run[h]) * inv_lanes;
            if constexpr (ROW != 0) m_run[h] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m_own), h));
            if (lane == 0) {
                wm[wave * 8 + h] = m_run[h];
                wl[wave * 8 + h] = lw;
            }
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < GT; ++h) {
            float M = wm[h];
#pragma unroll
            for (int w = 1; w < kSdpaWaves; ++w) M = fmaxf(M, wm[w * 8 + h]);
            const float f = __builtin_amdgcn_exp2f(m_run[h] - M);
            accb[h] *= f;
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[h][i] *= f;
        }
    }
    // Every lane parks its sums in LDS, [value slot][head][dim]; the output loop below
    // adds the slots in index order (no cross-lane shuffles, fixed order).
    if constexpr (KVQ != 0) {
#pragma unroll
        for (int h = 0; h < GT; ++h)
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[h][i] += accb[h];
    }
    if (vcol_ok) {
#pragma unroll
        for (int h = 0; h < GT; ++h) {
            float4* dst = reinterpret_cast<float4*>(red + ((size_t)vslot * GT + h) * a.v_dim + 8 * cv);
            dst[0] = make_float4(acc[h][0], acc[h][1], acc[h][2], acc[h][3]);
            dst[1] = make_float4(acc[h][4], acc[h][5], acc[h][6], acc[h][7]);
        }
    }
    __syncthreads();

    FK_SDPA_STAMP(6);
    const uint32_t n_out = gcount * a.v_dim;
    const bool direct = !NOMERGE && (n_active == 1);
    // Maximum (natural units) and sum of a head over the block.  Wave-local form: of the waves' own, by whichever thread
    // needs them (a few LDS reads that arrive with the value sums', instead of a round through LDS and a barrier).
    auto head_stats = [&](uint32_t h, float& m, float& l) {
        if constexpr (WAVES) {
#pragma clang fp contract(off)
            const float *wm = stat + 32, *wl = stat + 64;
            float mw[kSdpaWaves], lw[kSdpaWaves];
#pragma unroll
            for (int w = 0; w < kSdpaWaves; ++w) {
                mw[w] = wm[w * 8 + h];
                lw[w] = wl[w * 8 + h];
            }
            float M = mw[0];
#pragma unroll
            for (int w = 1; w < kSdpaWaves; ++w) M = fmaxf(M, mw[w]);
            l = lw[0] * __builtin_amdgcn_exp2f(mw[0] - M);
#pragma unroll
            for (int w = 1; w < kSdpaWaves; ++w) l += lw[w] * __builtin_amdgcn_exp2f(mw[w] - M);  // a product's rounding, then a sum's
            m = M * 0.693147180559945309f;
        } else {
            m = stat[h];
            l = stat[8 + h];
        }
    };
    for (uint32_t e = tid; e < n_out; e += kSdpaBlock) {
        const uint32_t h = e / a.v_dim, d = e - h * a.v_dim;
        float o = 0.f;
        // sixteen slots are read at once (every bf16 / quantised head of up to 128 dims has 16 or 32): read one by one, each
        // waits out the LDS (heads of 128: 0.8 us of the launch)
        uint32_t sl = 0;
        for (; sl + 16 <= vslots; sl += 16) {
            float v[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = red[((sl + i) * GT + h) * a.v_dim + d];
#pragma unroll
            for (int i = 0; i < 16; ++i) o += v[i];
        }
        for (; sl < vslots; ++sl) o += red[(sl * GT + h) * a.v_dim + d];
        float m, l;
        if (direct) {
            head_stats(h, m, l);
            st_u16<FUSED>(a.out + (size_t)(h0 + h) * a.v_dim + d, f32_to_bf16_bits(o / l));
        } else {
            float* p = a.partials + ((size_t)(h0 + h) * a.n_splits + split) * (a.v_dim + 2);
            st_f32<!NOMERGE>(p + 2 + d, o);
            if (d == 0) {
                head_stats(h, m, l);
                st_f32<!NOMERGE>(p, m);
                st_f32<!NOMERGE>(p + 1, l);
            }
        }
    }
    FK_SDPA_STAMP(7);
    if (direct || NOMERGE) return;

    // ---------------- last block merges the partials ----------------
    // Partials and the arrival counter move through agent-scope (write-through /
    // cache-bypassing) accesses, so no device-wide fence is needed: every wave waits
    // until its own stores have landed, the block barrier collects the waves, then one
    // thread counts the block in.
    wait_memory_ops_done();
    __syncthreads();
    uint32_t* flag = reinterpret_cast<uint32_t*>(stat + 16);
    if (tid == 0) {
        const uint32_t prev = atomicAdd(&a.counters[kvh * gz_count + gz], 1u);
        *flag = (prev == n_active - 1) ? 1u : 0u;
    }
    __syncthreads();
    FK_SDPA_STAMP(8);
    if (*flag == 0u) return;
    if (tid == 0)  // ready for the next launch (or the next layer of this one)
        __hip_atomic_store(&a.counters[kvh * gz_count + gz], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    // One wave per head, no block barriers.  The ranges are folded 16 at a time into a running (M, L, o) with the usual
    // rescaling, in range order, so the result does not depend on arrival order.  For every 16 ranges a lane issues 17
    // eight-byte loads: (m, l) of range base + (lane % 16), whose weight e^(m - M) that lane alone forms and hands to the
    // others through scalar registers, and its own two output dims of each of the 16 ranges.  The loads pass every cache
    // (some 1.2 us a trip), so all of up to 64 ranges are requested before the first is folded.
    constexpr uint32_t kBatch = 16;
    const uint32_t ranges = __builtin_amdgcn_readfirstlane(n_active);   // (the length came through a vector register)
    const uint32_t row = a.v_dim + 2;
    // (the head is the same for the whole wave, which the compiler has to be told: the rows' addresses then are scalars)
    for (uint32_t h = __builtin_amdgcn_readfirstlane(wave); h < gcount; h += kSdpaWaves) {
        const float* ph = a.partials + (size_t)(h0 + h) * a.n_splits * row;
        if constexpr ((KVQ != 0 ? ROW != 0 : ROW == 16) && MODE != 1) {
            // Heads of 128 (64) dims: sixteen (eight) bytes a lane, two ranges a load -- half the loads, of which a CU issues one in 16 .. 20
            // cycles --, which the half-waves then exchange: lanes l and l + 32 hold dims 4 l, 4 l + 1 and 4 l + 2, 4 l + 3 (both 2 l, 2 l + 1) of
            // every range.  The same additions in the same order.  8-bit caches, us, one range a load / two: 32 q / 8 kv heads x 128, 480
            // positions 11.5 / 10.5, 12000 24.5 / 23.2; 14 / 2 x 128, 480 17.5 / 14.3, 32000 67 / 49.
            constexpr uint32_t VD = ROW * 8u, LINE = (VD + 2u) * 4u, WL = ROW == 16 ? 4u : 2u;   // dims, bytes of a partial, words of a lane
            const __amdgpu_buffer_rsrc_t parts = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(ph), 0, (int)(a.n_splits * LINE), 0x27000);
            typedef uint32_t words2 __attribute__((ext_vector_type(2)));
            typedef uint32_t words __attribute__((ext_vector_type(WL)));
            constexpr int kPast = 1 << 4;   // sc1: past every cache that blocks do not share
            const uint32_t own = 8u + (lane & 31u) * (4u * WL);
            float M = -INFINITY, L = 0.f, o0 = 0.f, o1 = 0.f;
            auto fetch = [&](uint32_t base, words2& ml, words(&po)[kBatch / 2]) {
                const uint32_t first = base < ranges ? base : 0u, mine = base + (lane & (kBatch - 1));
                ml = __builtin_bit_cast(words2, __builtin_amdgcn_raw_buffer_load_b64(parts, (int)((mine < ranges ? mine : first) * LINE), 0, kPast));
#pragma unroll
                for (uint32_t i = 0; i < kBatch / 2; ++i) {
                    const uint32_t r = base + 2u * i + (lane >> 5);
                    const int at = (int)((r < ranges ? r : first) * LINE + own);
                    if constexpr (ROW == 16)
                        po[i] = __builtin_bit_cast(words, __builtin_amdgcn_raw_buffer_load_b128(parts, at, 0, kPast));
                    else
                        po[i] = __builtin_bit_cast(words, __builtin_amdgcn_raw_buffer_load_b64(parts, at, 0, kPast));
                }
            };
            auto fold = [&](uint32_t base, const words2& ml, const words(&po)[kBatch / 2]) {
                const float m_mine = __uint_as_float(ml[0]);
                float mx = dpp_max<0xB1>(m_mine);
                mx = dpp_max<0x4E>(mx);
                mx = dpp_max<0x141>(mx);
                mx = dpp_max<0x140>(mx);
                const float mn = fmaxf(M, mx);
                const float w_mine = base + (lane & (kBatch - 1)) < ranges ? expf(m_mine - mn) : 0.f;
                const float alpha = base ? expf(M - mn) : 0.f;
                L *= alpha;
                o0 *= alpha;
                o1 *= alpha;
#pragma unroll
                for (uint32_t i = 0; i < kBatch; i += 2) {
                    const auto x0 = __builtin_amdgcn_permlane32_swap(po[i / 2][0], po[i / 2][WL - 2u], false, false);
                    const auto x1 = __builtin_amdgcn_permlane32_swap(po[i / 2][1], po[i / 2][WL - 1u], false, false);
#pragma unroll
                    for (uint32_t e = 0; e < 2; ++e) {
                        const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w_mine), i + e));
                        const float pl = __int_as_float(__builtin_amdgcn_readlane((int)ml[1], i + e));
                        L = fmaf(pl, w, L);
                        o0 = fmaf(__uint_as_float(x0[e]), w, o0);
                        o1 = fmaf(__uint_as_float(x1[e]), w, o1);
                    }
                }
                M = mn;
            };
            auto merge = [&](auto n_const, uint32_t base) {
                constexpr uint32_t N = decltype(n_const)::value;
                words2 ml[N];
                words po[N][kBatch / 2];
#pragma unroll
                for (uint32_t b = 0; b < N; ++b) fetch(base + b * kBatch, ml[b], po[b]);
#pragma unroll
                for (uint32_t b = 0; b < N; ++b)
                    if (base + b * kBatch < ranges) fold(base + b * kBatch, ml[b], po[b]);
            };
            if (ranges <= kBatch) {
                merge(std::integral_constant<uint32_t, 1>{}, 0u);
            } else if (ranges <= 2 * kBatch) {
                merge(std::integral_constant<uint32_t, 2>{}, 0u);
            } else {
                for (uint32_t base = 0; base < ranges; base += 4 * kBatch) merge(std::integral_constant<uint32_t, 4>{}, base);
            }
            const float inv_l = 1.0f / L;
            if (ROW == 16 || lane < 32u) {
                uint16_t* dst = a.out + (size_t)(h0 + h) * VD + (ROW == 16 ? 4u * (lane & 31u) + 2u * (lane >> 5) : 2u * lane);
                st_u16<FUSED>(dst, f32_to_bf16_bits(o0 * inv_l));
                st_u16<FUSED>(dst + 1, f32_to_bf16_bits(o1 * inv_l));
            }
            continue;
        }
        for (uint32_t d2 = lane; d2 < ((a.v_dim >> 1) + kWave - 1) / kWave * kWave; d2 += kWave) {
            const bool live = d2 < (a.v_dim >> 1);
            const uint32_t at = 2u + 2u * (live ? d2 : 0u);
            float M = -INFINITY, L = 0.f, o0 = 0.f, o1 = 0.f;
            // two floats at ph + (uniform) + (per lane), as a GLOBAL access with a scalar base and a 32-bit lane offset: the generic
            // form keeps a 64-bit address in registers for every load in flight
            auto ld_partial = [&](uint32_t uniform, uint32_t per_lane) {
                typedef const __attribute__((address_space(1))) char* gptr;
                typedef const __attribute__((address_space(1))) unsigned long long* gptr8;
                const gptr base = (gptr)(uintptr_t)(ph + uniform);
                const unsigned long long v = __hip_atomic_load((gptr8)(base + 4u * per_lane), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
            };
            auto fetch = [&](uint32_t base, float2& ml, float2(&po)[kBatch]) {
                const uint32_t first = base < ranges ? base : 0u, mine = base + (lane & (kBatch - 1));
                ml = ld_partial(0u, (mine < ranges ? mine : first) * row);
#pragma unroll
                for (uint32_t i = 0; i < kBatch; ++i)
                    po[i] = ld_partial((base + i < ranges ? base + i : first) * row, at);
            };
            auto fold = [&](uint32_t base, const float2& ml, const float2(&po)[kBatch]) {
                // (a lane past the last range holds the batch's first: the maximum is that of the live ones)
                float mx = dpp_max<0xB1>(ml.x);
                mx = dpp_max<0x4E>(mx);
                mx = dpp_max<0x141>(mx);
                mx = dpp_max<0x140>(mx);
                const float mn = fmaxf(M, mx);
                const float w_mine = base + (lane & (kBatch - 1)) < ranges ? expf(ml.x - mn) : 0.f;
                const float alpha = base ? expf(M - mn) : 0.f;
                L *= alpha;
                o0 *= alpha;
                o1 *= alpha;
#pragma unroll
                for (uint32_t i = 0; i < kBatch; ++i) {
                    const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w_mine), i));
                    const float pl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ml.y), i));
                    L = fmaf(pl, w, L);
                    o0 = fmaf(po[i].x, w, o0);
                    o1 = fmaf(po[i].y, w, o1);
                }
                M = mn;
            };
            // N batches requested together, then folded; batches past the last range are requested (clamped: a branch between
            // the loads would make the first fold wait for all of them) and not folded.
            auto merge = [&](auto n_const, uint32_t base) {
                constexpr uint32_t N = decltype(n_const)::value;
                float2 ml[N], po[N][kBatch];
#pragma unroll
                for (uint32_t b = 0; b < N; ++b) fetch(base + b * kBatch, ml[b], po[b]);
#pragma unroll
                for (uint32_t b = 0; b < N; ++b)
                    if (base + b * kBatch < ranges) fold(base + b * kBatch, ml[b], po[b]);
            };
            if (ranges <= kBatch) {
                merge(std::integral_constant<uint32_t, 1>{}, 0u);
            } else if (ranges <= 2 * kBatch) {
                merge(std::integral_constant<uint32_t, 2>{}, 0u);
            } else {
                for (uint32_t base = 0; base < ranges; base += 4 * kBatch) merge(std::integral_constant<uint32_t, 4>{}, base);
            }
            const float inv_l = 1.0f / L;
            if (live) {
                uint16_t* dst = a.out + (size_t)(h0 + h) * a.v_dim + 2 * d2;
                st_u16<FUSED>(dst, f32_to_bf16_bits(o0 * inv_l));
                st_u16<FUSED>(dst + 1, f32_to_bf16_bits(o1 * inv_l));
            }
        }
    }
    FK_SDPA_STAMP(9);
}

// The context length of a stand-alone launch: ONE unconditional load (a load under a branch would be waited for at
// the join, ahead of the cache reads it is meant to overlap) through a GLOBAL pointer -- the device scalar, or the
// immediate's own place in the kernel-argument segment.  (Selected as generic pointers the two make a flat load,
// and a flat load's completion can only be awaited with vmcnt(0): every cache row requested behind it would be
// waited for with it.)
__device__ __forceinline__ uint32_t sdpa_load_kv_len(const SdpaArgs& a) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef const __attribute__((address_space(1))) uint32_t* global_u32;
    const global_u32 imm = (global_u32)((uintptr_t)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(SdpaArgs, kv_len_imm));
    const global_u32 dev = (global_u32)(uintptr_t)a.kv_len_ptr;
    return *(a.kv_len_ptr ? dev : imm);
#else
    return a.kv_len_ptr ? *a.kv_len_ptr : a.kv_len_imm;
#endif
}

template <int GT, int KVQ = 0, int ROW = 0>
__global__ __launch_bounds__(kSdpaBlock, GT == 8 ? 1 : 2) void sdpa_decode_kernel(const SdpaArgs a) {
    extern __shared__ __align__(16) float lds[];
    // One unconditional load (the immediate is read from the kernel-argument segment
    // when there is no device scalar): a load under a branch would be waited for at
    // the join, ahead of the cache reads it is meant to overlap.
    kernarg_warm<(int)sizeof(SdpaArgs)>();
    const uint32_t kv_len0 = sdpa_load_kv_len(a);
    if (a.rows <= 1) {
        sdpa_block<GT, false, SdpaArgs, KVQ, false, false, ROW>(a, kv_len0, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.z, lds);
        return;
    }
    // Several active rows (multi-token verification, chunked prefill): grid.z carries
    // (row, head tile).  Row r is the token at position kv_len0 - 1 + r: it attends to
    // kv_len0 + r cache rows (causal inside the group), with its own q, out and workspace.
    const uint32_t gz_count = gridDim.z / a.rows;
    const uint32_t tr = blockIdx.z / gz_count, gz = blockIdx.z - tr * gz_count;
    SdpaArgs r = a;
    r.q = a.q + (size_t)tr * a.n_heads * a.qk_dim;
    r.out = a.out + (size_t)tr * a.n_heads * a.v_dim;
    r.partials = a.partials + (size_t)tr * a.n_heads * a.n_splits * (a.v_dim + 2);
    r.counters = a.counters + (size_t)tr * a.n_kv * gz_count;
    sdpa_block<GT, false, SdpaArgs, KVQ, false, false, ROW>(r, kv_len0, blockIdx.x, blockIdx.y, gz, gz_count, lds, tr);
}

// RoPE (+ head norm) of q and of the new k row, the cache append and the attention in one
// launch: a.q / a.k_new / a.v_new are the raw projection outputs of the token at position
// kv_len - 1, a.k / a.v the cache it is appended to.
// KVQ: a quantised cache; the new rows are quantised by the block whose range holds them.
template <int GT, bool FASTHEAD, int KVQ = 0, int ROW = 0>
__global__ __launch_bounds__(kSdpaBlock, GT == 8 ? 1 : 2) void sdpa_rope_store_kernel(const SdpaArgs a) {
    extern __shared__ __align__(16) float lds[];
    kernarg_warm<(int)sizeof(SdpaArgs)>();
    const uint32_t kv_len0 = sdpa_load_kv_len(a);
    sdpa_block<GT, 2, SdpaArgs, KVQ, FASTHEAD, false, ROW>(a, kv_len0, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.z, lds);
}

}  // namespace fk
