// Loads straight from memory into LDS, and matrix sums kept in the AGPR half of the register file: what the prompt kernels
// (qgemm_dma.hip, sdpa_prefill.hip) share.
#pragma once
#include <type_traits>

#include "fk_device.hpp"

namespace fk {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// f(integral_constant<int, 0>) .. f(integral_constant<int, N - 1>): every index is a constant, whatever the unroller thinks of
// the body (an accumulator indexed by a loop variable goes to scratch).
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

// 16 (4) bytes per lane from `base + off` (`ptr`) to LDS at `to` + 16 (4) * lane; counted in vmcnt.  As statements the
// compiler does not look into: its own form waits for every such load in flight ahead of each LDS read.  m0, which the
// statement writes, is an output (the compiler refuses it as a clobber).
__device__ __forceinline__ void dma16(uint32_t to, uint32_t off, const void* base) {
    uint32_t m0;
    asm volatile("s_mov_b32 %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3" : "=&{m0}"(m0) : "s"(to), "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ void dma16(uint32_t to, const unsigned char* ptr) {
    uint32_t m0;
    asm volatile("s_mov_b32 %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off" : "=&{m0}"(m0) : "s"(to), "v"(ptr) : "memory");
}
__device__ __forceinline__ void dma4(uint32_t to, const unsigned char* ptr) {
    uint32_t m0;
    asm volatile("s_mov_b32 %0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, off" : "=&{m0}"(m0) : "s"(to), "v"(ptr) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// a finished sum, where it is used (a plain read lets the compiler copy all of them out at once)
__device__ __forceinline__ f32x4_t take(const f32x4_t& acc) {
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v[r]) : "a"(acc[r]));
    return f32x4_t{v[0], v[1], v[2], v[3]};
}
// (the statements of those files hide matrix instructions from the hazard recogniser: sums are read behind this)
__device__ __forceinline__ void settle_matrix_ops() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

}  // namespace fk
