// Shared by the kernels whose lanes each continue one f32 fma chain with the other operand's values
// as scalar operands: the gate scores (knn.hip) and the f32 products (f32_gemm.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace larql {

typedef float floatx4_t __attribute__((ext_vector_type(4)));

// Floats at wave-uniform addresses, read with scalar loads.
typedef const float __attribute__((address_space(4))) * scalar_f32_ptr;

// At most N vector memory operations of the wave still in flight.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// acc[q] += v[i] x_q[k0 + i] for i = 0 .. 15 in order, x_q the row q (< QW) at X + q sq of a k-minor
// matrix: 16 consecutive floats per row as scalar operands, four rows' chains side by side.
template <int QW>
__device__ __forceinline__ void lane_fma16(float (&acc)[QW], const float (&v)[16], scalar_f32_ptr X, size_t sq, int k0) {
    constexpr int G = QW < 4 ? QW : 4;
#pragma unroll
    for (int q0 = 0; q0 < QW; q0 += G) {
#pragma unroll
        for (int i = 0; i < 16; i++)
#pragma unroll
            for (int q = q0; q < q0 + G; q++) acc[q] = fmaf(v[i], X[q * sq + k0 + i], acc[q]);
    }
}

}  // namespace larql
