// Pieces of the f32-accuracy GEMM shared by its kernels (gemm_hp.hip) and the row kernels that
// produce its input (prompt.hip): the fp16-pair split and the packed operand layout.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace larql {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

// v - (f32) the low / high f16 half of h2, one v_fma_mix_f32 (the half widened inside the
// instruction; written out because the compiler otherwise emits a conversion and a subtract)
__device__ __forceinline__ float sub_f16_lo(float v, uint32_t h2) {
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h2), "v"(v));
    return r;
}
__device__ __forceinline__ float sub_f16_hi(float v, uint32_t h2) {
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h2), "v"(v));
    return r;
}

// {a, b} -> hi pair {fp16(a), fp16(b)} and lo pair {fp16(a - hi_a), fp16(b - hi_b)}
__device__ __forceinline__ void hp_split2(float a, float b, uint32_t& hi, uint32_t& lo) {
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, f16x2));
    const float la = sub_f16_lo(a, hi), lb = sub_f16_hi(b, hi);
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){la, lb}, f16x2));
}

// Eight f32 values -> their hi and lo operands.
__device__ __forceinline__ void hp_split8(const float (&v)[8], v4u& hi, v4u& lo) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; i++) hp_split2(v[2 * i], v[2 * i + 1], h[i], l[i]);
    hi = v4u{h[0], h[1], h[2], h[3]};
    lo = v4u{l[0], l[1], l[2], l[3]};
}

// Packed operands XP[token tile][k-step][hi, lo][64 lanes][16 B]: lane 16 g + i of k-step ks
// holds elements 32 ks + 8 g .. + 7 of token i of the tile times the token's power of two, in the
// order masks of a weight dword give its nibbles, (0, 4), (2, 6), (1, 5), (3, 7).  The index of
// the hi part of token m's eight elements e8 = 4 ks + g; the lo part is 64 further.
__device__ __forceinline__ size_t hp_packed_at(int m, int e8, int K) {
    return ((static_cast<size_t>(m >> 4) * (K / 32) + (e8 >> 2)) * 2) * 64 + 16 * (e8 & 3) + (m & 15);
}

// Eight elements x[0 .. 7] times sc -> packed at o.
__device__ __forceinline__ void hp_pack8(const float* x, float sc, v4u* o) {
    const floatx4 a = *reinterpret_cast<const floatx4*>(x), b = *reinterpret_cast<const floatx4*>(x + 4);
    const float e[8] = {a.x * sc, b.x * sc, a.z * sc, b.z * sc, a.y * sc, b.y * sc, a.w * sc, b.w * sc};
    v4u hi, lo;
    hp_split8(e, hi, lo);
    o[0] = hi;
    o[64] = lo;
}

}  // namespace larql
