// One new row of a quantised KV cache by one wave: the key's RMSNorm and rotation in fp32 (not rounded to bf16 before it is
// quantised), then per group the MLX-affine quantiser's arithmetic statement for statement (see quantize_affine_kernel).
// Shared by the store kernel and the attention that appends the row itself.
#pragma once
#include "fk_device.hpp"
#include "rope_device.hpp"

namespace fk {

// `tab` (optional): (cos, sin) per pair at this position, the values rope_rotate would compute.
__device__ __forceinline__ void kv_key_row(const uint16_t* src, const uint16_t* nw, float* row, uint32_t dim, uint32_t rope_dims, uint32_t pos,
                                           float base_log2, float eps, uint32_t lane, const float* tab) {
    float r = 1.f;
    if (nw) {
        float ss = 0.f;
        for (uint32_t d = lane; d < dim; d += kWave) {
            const float x = bf16_bits_to_f32(src[d]);
            ss = fmaf(x, x, ss);
        }
        ss = wave_sum(ss);
        r = 1.0f / sqrtf(ss / (float)dim + eps);
    }
    auto value = [&](uint32_t d) {
        const float x = bf16_bits_to_f32(src[d]);
        return nw ? round_bf16(bf16_bits_to_f32(nw[d]) * round_bf16(x * r)) : x;
    };
    const uint32_t half = rope_dims / 2;
    for (uint32_t d = lane; d < half; d += kWave) {
        float lo, hi;
        if (tab) {
            const float vlo = value(d), vhi = value(d + half), cs = tab[2 * d], sn = tab[2 * d + 1];
            lo = vlo * cs - vhi * sn;
            hi = vhi * cs + vlo * sn;
        } else {
            rope_rotate(value(d), value(d + half), d, half, pos, base_log2, lo, hi);
        }
        row[d] = lo;
        row[d + half] = hi;
    }
    for (uint32_t d = 2 * half + lane; d < dim; d += kWave) row[d] = value(d);
}

// row -> codes; meta(group, scale bits, bias bits) from lane 0.  The row is complete in LDS; every lane derives the same scale
// and bias.
template <typename META>
__device__ __forceinline__ void kv_quantize_row(const float* row, uint8_t* codes, uint32_t dim, uint32_t group, uint32_t bits, uint32_t lane,
                                                META&& meta) {
    const int mask = (1 << bits) - 1;
    for (uint32_t g = 0; g < dim / group; ++g) {
        const float* x = row + g * group;
        float vmin = INFINITY, vmax = -INFINITY;
        for (uint32_t i = lane; i < group; i += kWave) {
            vmin = fminf(vmin, x[i]);
            vmax = fmaxf(vmax, x[i]);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            vmin = fminf(vmin, __shfl_xor(vmin, o, kWave));
            vmax = fmaxf(vmax, __shfl_xor(vmax, o, kWave));
        }
        const float scale_abs = fmaxf((vmax - vmin) / (float)mask, 1.0e-7f);
        const bool lo_anchor = fabsf(vmin) > fabsf(vmax);
        float scale = lo_anchor ? scale_abs : -scale_abs;
        const float edge = lo_anchor ? vmin : vmax;
        const float q0 = roundf(edge / scale);
        const bool at_zero = (q0 == 0.0f);
        scale = at_zero ? scale : (edge / q0);
        const float bias = at_zero ? 0.0f : edge;
        const float inv_scale = (scale != 0.0f) ? (1.0f / scale) : 0.0f;
        for (uint32_t i = lane; i < group; i += kWave) {
            int qi = (int)roundf((x[i] - bias) * inv_scale);
            qi = qi < 0 ? 0 : (qi > mask ? mask : qi);
            codes[g * group + i] = (uint8_t)qi;
        }
        if (lane == 0) meta(g, f32_to_bf16_bits(scale), f32_to_bf16_bits(bias));
    }
}

// codes (complete in LDS) -> packed words
template <typename WORD>
__device__ __forceinline__ void kv_pack_row(const uint8_t* codes, uint32_t dim, uint32_t bits, uint32_t lane, WORD&& put) {
    const uint32_t per_word = 32u / bits;
    for (uint32_t wi = lane; wi < dim / per_word; wi += kWave) {
        uint32_t word = 0;
        for (uint32_t el = 0; el < per_word; ++el) word |= (uint32_t)codes[wi * per_word + el] << (el * bits);
        put(wi, word);
    }
}

}  // namespace fk
