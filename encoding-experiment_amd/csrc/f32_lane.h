// Shared by the kernels whose lanes each continue one f32 fma chain with the other operand's values
// as scalar operands: the gate scores (knn.hip) and the f32 products (f32_gemm.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace larql {

typedef float floatx4_t __attribute__((ext_vector_type(4)));

// A query block of a k: QW consecutive floats at a wave-uniform address, read with scalar loads.
typedef const float __attribute__((address_space(4))) * scalar_f32_ptr;

// At most N vector memory operations of the wave still in flight.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The scalar operands' layout: XT[b][k][qw] = element k of query qw b + i (at X + q sq + k sk) for
// q < Q and k < K, else +0; b < Qp / qw, k < Kp (f32_gemm.hip).
void launch_queries_t(const float* X, size_t sq, size_t sk, float* XT, int Q, int K, int Kp, int Qp, int qw,
                      hipStream_t s);

}  // namespace larql
