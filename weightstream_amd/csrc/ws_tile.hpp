// Helpers of the tile kernels (gemm_tile.hip, moe_tile.hip): LDS reads at
// constant offsets that the compiler does not see as memory accesses (ordered
// by lds_wait / lds_ready, see lds_read_b128), conversions piece by piece,
// direct global -> LDS copies.
#pragma once

#include <utility>

#include "ws_device.hpp"

namespace ws {
namespace tile {

typedef unsigned int u32x2v __attribute__((ext_vector_type(2)));

template <int OFF>
__device__ __forceinline__ u32x2v rd64(uint32_t a) {
    u32x2v v;
    __asm__ volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF));
    return v;
}
template <int OFF>
__device__ __forceinline__ u32x4v rd128(uint32_t a) {
    u32x4v v;
    __asm__ volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF));
    return v;
}
template <int OFF>
__device__ __forceinline__ uint32_t rd32(uint32_t a) {
    uint32_t v;
    __asm__ volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF));
    return v;
}
template <int OFF>
__device__ __forceinline__ uint32_t rd8(uint32_t a) {
    uint32_t v;
    __asm__ volatile("ds_read_u8 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF));
    return v;
}
template <class F, int... I>
__device__ __forceinline__ void seq(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
#define WS_SEQ(n, name) std::make_integer_sequence<int, (n)>{}

// piece P (0..3) of a fragment: two e4m3 bytes of q, or two e2m1 nibbles of
// the word f, times the scale s, as two bf16
template <int P>
__device__ __forceinline__ uint32_t cvt8(u32x2v q, float s) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(q[P >> 1], s, P & 1));
}
template <int P>
__device__ __forceinline__ uint32_t cvt4(uint32_t f, float s) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(f, s, P));
}
// nothing is scheduled across: the interleaving written below is the one run
__device__ __forceinline__ void pin() { __builtin_amdgcn_sched_barrier(0); }

// direct global -> LDS copies, 16 or 4 bytes per lane, to lane-consecutive LDS
__device__ __forceinline__ void dma16(const uint8_t *src, uint8_t *dst) {
    __builtin_amdgcn_global_load_lds((const void *)src,
                                     (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
}
__device__ __forceinline__ void dma4(const uint8_t *src, uint8_t *dst) {
    __builtin_amdgcn_global_load_lds((const void *)src,
                                     (__attribute__((address_space(3))) void *)dst, 4, 0, 0);
}

}  // namespace tile
}  // namespace ws
