// f32-accuracy GEMMs of quantized weights: Y[M x N] = X[M x K] . deq(W)^T from f32 X, for the
// chains of projections of the prompt pass and for small batches (Q4_K and Q6_K).
//
// Every f32 activation x is split into two fp16 parts, hi = fp16(x) and lo = fp16(x - hi) (x -
// hi exact in f32), x = hi + lo to ~2^-22 of x or 2^-40 of the row's largest element, whichever is
// more (lo's smallest step), and the products run on v_mfma_f32_16x16x32_f16 with
// f32 accumulation against fp16 weight operands that are exact integers.  Single fp16 operands
// (2^-11) compounded past the 1e-3 bar through 8 and 16 layers; bf16 pairs (2^-16 per product)
// doubled the error.  fp16's range is made safe per token: the row statistics hold the power of
// two that puts the row's largest |x| in [2^14, 2^15); the packing multiplies by it and the
// epilogue divides it out, both exact.  An infinite operand gives NaN (its lo part is inf - inf).
//
// Two launches: x_pack_kernel writes X once as ready-made operands (1 KB per 16 tokens, k-step
// of 32 and part), and the GEMM streams them into LDS by buffer loads that need no registers,
// while each wave turns its own weight rows into operands in registers.
#include <algorithm>
#include <type_traits>

#include "decode.h"
#include "device_common.h"
#include "gemm_hp.h"
#include "larql_hip_internal.h"

namespace larql {

namespace {

constexpr int kPkWaves = 4;             // waves per workgroup, side by side along N
constexpr int kPkR = 4;                 // 16-row weight tiles per wave
constexpr int kPkRows = 16 * kPkR * kPkWaves;  // 256 weight rows per workgroup
constexpr int kPkThreads = 64 * kPkWaves;

// One workgroup per row: the row's exponent and (with xs) scaled sub-block sums
// (gemm_row_stats).
__global__ __launch_bounds__(256) void row_exp_kernel(const float* __restrict__ X, int K, int* __restrict__ e,
                                                      float* __restrict__ xs) {
    gemm_row_stats(X + static_cast<size_t>(blockIdx.x) * K, K, e + blockIdx.x,
                   xs ? xs + static_cast<size_t>(blockIdx.x) * (K / 32) : nullptr);
}

// X [M x K] -> the packed operands (hp_packed_at), each token times its power of two; tokens past
// M are zeros.  Grid (K / 128, token tiles); wave w = k-step w of the workgroup's four.
__global__ __launch_bounds__(256) void x_pack_kernel(const float* __restrict__ X, const int* __restrict__ xe,
                                                     v4u* __restrict__ XP, int M, int K) {
    const int lane = threadIdx.x & 63, ks = blockIdx.x * 4 + (threadIdx.x >> 6), g = lane >> 4;
    const int m = blockIdx.y * 16 + (lane & 15), mc = min(m, M - 1);
    if (ks >= K / 32) return;
    const float* p = X + static_cast<size_t>(mc) * K + 32 * ks + 8 * g;
    const floatx4 a = *reinterpret_cast<const floatx4*>(p), b = *reinterpret_cast<const floatx4*>(p + 4);
    const float sc = m < M ? ldexpf(1.0f, xe[mc]) : 0.0f;
    float e[8] = {a.x, b.x, a.z, b.z, a.y, b.y, a.w, b.w};
#pragma unroll
    for (int k = 0; k < 8; k++) e[k] = m < M ? e[k] * sc : 0.0f;
    v4u hi, lo;
    hp_split8(e, hi, lo);
    v4u* o = XP + hp_packed_at(m, 4 * ks + g, K);
    o[0] = hi;
    o[64] = lo;
}

// At most N vector memory operations of the wave still in flight.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 16 bytes per lane from a buffer straight into LDS, at dst + 16 lane (dst wave-uniform).  (The
// host pass, which only needs the kernel's stub, refuses the builtin's 16-byte size.)
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, v4u* dst, uint32_t voff, uint32_t soff) {
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
#endif
}

// The A operands of one k-step (hi, lo of TT token tiles, 8 KB apart), read and waited for in
// one block: the compiler does not track the loads that fill the LDS ring by stage, so its own
// reads would wait for every load in flight.
template <int TT>
__device__ __forceinline__ void read_a(uint32_t a, int t, v4u (&h)[TT], v4u (&l)[TT]) {
    const uint32_t at = a + 2048u * t;
    if constexpr (TT == 1) {
        asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:1024\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(h[0]), "=&v"(l[0])
                     : "v"(at)
                     : "memory");
    } else if constexpr (TT == 2) {
        asm volatile(
            "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:1024\n\t"
            "ds_read_b128 %2, %4 offset:8192\n\tds_read_b128 %3, %4 offset:9216\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(h[0]), "=&v"(l[0]), "=&v"(h[1]), "=&v"(l[1])
            : "v"(at)
            : "memory");
    } else if constexpr (TT == 3) {
        asm volatile(
            "ds_read_b128 %0, %6\n\tds_read_b128 %1, %6 offset:1024\n\t"
            "ds_read_b128 %2, %6 offset:8192\n\tds_read_b128 %3, %6 offset:9216\n\t"
            "ds_read_b128 %4, %6 offset:16384\n\tds_read_b128 %5, %6 offset:17408\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(h[0]), "=&v"(l[0]), "=&v"(h[1]), "=&v"(l[1]), "=&v"(h[2]), "=&v"(l[2])
            : "v"(at)
            : "memory");
    } else {
        asm volatile(
            "ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:1024\n\t"
            "ds_read_b128 %2, %8 offset:8192\n\tds_read_b128 %3, %8 offset:9216\n\t"
            "ds_read_b128 %4, %8 offset:16384\n\tds_read_b128 %5, %8 offset:17408\n\t"
            "ds_read_b128 %6, %8 offset:24576\n\tds_read_b128 %7, %8 offset:25600\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(h[0]), "=&v"(l[0]), "=&v"(h[1]), "=&v"(l[1]), "=&v"(h[2]), "=&v"(l[2]), "=&v"(h[3]), "=&v"(l[3])
            : "v"(at)
            : "memory");
    }
}

// The eight codes of a nibble dword as fp16 pairs, code times 2^-24 (elements 0, 4, 2, 6) or 2^-20
// (1, 5, 3, 7): a nibble in the low byte of a half is a subnormal, exact in an fp16 product.
__device__ __forceinline__ void nibble_pairs(uint32_t w, f16x2 (&o)[4]) {
    const uint32_t w8 = w >> 8;
    o[0] = __builtin_bit_cast(f16x2, w & 0x000F000Fu);
    o[1] = __builtin_bit_cast(f16x2, w8 & 0x000F000Fu);
    o[2] = __builtin_bit_cast(f16x2, w & 0x00F000F0u);
    o[3] = __builtin_bit_cast(f16x2, w8 & 0x00F000F0u);
}

__device__ __forceinline__ half8 operand8(f16x2 a, f16x2 b, f16x2 c, f16x2 d) {
    return __builtin_bit_cast(half8, v4u{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                         __builtin_bit_cast(uint32_t, c), __builtin_bit_cast(uint32_t, d)});
}

// 4 x 4 transpose of a lane's dwords across the four lane groups: lane group g gets dword g of
// lane groups 0 .. 3.
__device__ __forceinline__ v4u transpose4(v4u q) {
    const auto a02 = __builtin_amdgcn_permlane32_swap(q.x, q.z, false, false);
    const auto a13 = __builtin_amdgcn_permlane32_swap(q.y, q.w, false, false);
    const auto r01 = __builtin_amdgcn_permlane16_swap(a02[0], a13[0], false, false);
    const auto r23 = __builtin_amdgcn_permlane16_swap(a02[1], a13[1], false, false);
    return v4u{r01[0], r01[1], r23[0], r23[1]};
}

struct PkArgs {
    const uint8_t* qs;    // Q4_K nibbles, Q6_K blocks
    const uint8_t* hdr;   // Q4_K headers (Q6_K: unused)
    const v4u* XP;        // packed X (x_pack_kernel)
    const int* xe;        // row exponents
    const float* xs;      // scaled sub-block sums (Q4_K)
    float* Y;             // output, or the split partials
    size_t ypart;         // floats between the outputs of two splits
    int M, N, K, ntiles, mtiles, sb_per, ldy, gx, gy, gz;
};

// Measured, Q4_K [28672 x 4096] (kernel trace): 512 tokens 242-250 us (481-497
// TFLOP/s; MFMA busy 46% of the cycles, VALU 18%, 1.5 waves per SIMD; 311 us when each workgroup split f32 tokens into pairs itself and one wave per SIMD
// waited for its own loads and LDS reads), 24 tokens 30 us (the call 83 us on the fp16 GEMM).  The
// codes by masks take 13 VALU per eight weights; made fp16 integers by a byte permute and an fma per
// pair, 14 (two 8B-shape layers, 512 tokens: 1137 us against 1164; bit-identical).  Left subnormal
// (11 VALU), the codes cost the sums of the matrix cores three bits: 1.9e-6 from 64 bits at K =
// 4096 against 2.3e-7, at the same speed.
//
// 16 TT tokens x 256 weight rows per workgroup: wave w owns 64 rows (kPkR tiles), all waves
// share the token operands.  A unit is 128 k (half a super-block, four k-steps of one 32-element
// sub-block): its operands (8 KB per token tile) are loaded into a two-slot LDS ring while the
// unit before it is multiplied.
//
// Q4_K: w = d s_j q - dmin m_j, so per super-block and token
//   sum_k x_k w_k = d sum_j s_j (sum_{k in j} x_k q_k) - dmin sum_j m_j X_j,  X_j = sum_{k in j} x_k.
// s_j q <= 945 is exact in fp16, the weight operand of both products (x hi and lo, both
// exact in f32; only the split's 2^-22 is lost), a fresh accumulator per super-block, added into
// the total times d.  The min term follows the K loop: the sub-block sums X_j 2^(e - 5) against
// -32 dmin m_j per row, both as fp16 pairs (three products), 32 sub-blocks per k-step.  A lane's
// 16-byte nibble load holds one sub-block, transposed across the lane groups.
//
// Q6_K: w = d sc (q - 32) per 16-element group; sc (q - 32) reaches 4096, past fp16's exact
// integers, so it is split exactly, hi = fp16(sc (q - 32)) and lo the rest (at most 1): three
// products per super-block accumulator (the dropped x_lo w_lo is ~2^-23 of it).
template <int FMT, int TT>
__global__ __launch_bounds__(kPkThreads, 2) void pk_gemm_kernel(PkArgs a) {
    constexpr bool kQ4K = FMT == LARQL_Q4_K, kQ6K = FMT == LARQL_Q6_K;
    static_assert(kQ4K || kQ6K, "Q4_K or Q6_K");
    // an operand's unit: Q4_K s_j q times 2^-14, Q6_K weights at a quarter
    constexpr float kUnit = kQ6K ? 4.0f : 16384.0f;
    // weight loads per wave of a unit of each parity
    constexpr int kWLoads0 = (kQ6K ? 4 : 2) * kPkR, kWLoads1 = 2 * kPkR;
    __shared__ __align__(1024) v4u As[2][TT * 8 * 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int M = a.M, N = a.N, K = a.K;
    // Workgroup -> (weight block bx, token block by, K split bz), a 1-D grid: the gy token
    // blocks of one (bx, bz) get consecutive ids that are equal mod 8, i.e. one XCD (ids go
    // round-robin over the 8) at about the same time, so a weight block is fetched into
    // that XCD's L2 once for all tokens; ids past the gx gz pairs (rounded up to 8) exit.
    const int L = static_cast<int>(blockIdx.x), slot = L >> 3, by = slot % a.gy;
    const int grp = (slot / a.gy) * 8 + (L & 7);
    if (grp >= a.gx * a.gz) return;
    const int bx = grp % a.gx, bz = grp / a.gx;
    const int mt0 = by * TT, nt0 = (bx * kPkWaves + wave) * kPkR;
    // split bz of K: super-blocks [bz sb_per, (bz + 1) sb_per), two units of 128 k each, sums to Y[bz]
    const int u0 = 2 * bz * a.sb_per, u1 = min(K / 128, u0 + 2 * a.sb_per), last = u1 - 1;
    float* Y = a.Y + bz * a.ypart;

    // raw buffer loads: the wave-uniform part of each offset in the scalar operand, the lane's in
    // the vector operand; a buffer starts at the wave's first tile, so offsets stay small
    // whatever the weight's or X's size
    const int nks = K / 32;
    const uint32_t qtile = kQ6K ? static_cast<uint32_t>(K / 256) * static_cast<uint32_t>(kQ6Block) : 8u * K;
    const uint32_t htile = K;  // headers, 256 bytes per super-block (Q6_K: none)
    const int ntc = min(nt0, a.ntiles - 1), have = min(kPkR, a.ntiles - ntc), mhave = min(TT, a.mtiles - mt0);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<v4u*>(a.XP) + static_cast<size_t>(mt0) * nks * 128, 0,
        static_cast<int>(static_cast<uint32_t>(mhave) * nks * 2048u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(a.qs) + static_cast<size_t>(ntc) * qtile, 0, static_cast<int>(have * qtile), 0x00020000);
    const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(a.hdr) + static_cast<size_t>(ntc) * htile, 0, kQ4K ? static_cast<int>(have * htile) : 0, 0x00020000);
    uint32_t qo[kPkR], ho[kPkR];
#pragma unroll
    for (int j = 0; j < kPkR; j++) {  // (tiles past the last re-read it; their rows are not stored)
        qo[j] = static_cast<uint32_t>(min(j, have - 1)) * qtile;
        ho[j] = static_cast<uint32_t>(min(j, have - 1)) * htile;
    }
    // the lane's part: tile-major, 16 bytes a lane, the header of row c
    const uint32_t ql = lane * 16u, hl = c * 16u;
    // load instruction n = wave 2 TT + i of a unit: token tile n / 8, KB n % 8 of its 8 KB (k-step
    // t = (n % 8) / 2, part n % 2).  Q4_K: unit u is k-steps 4 u + t; Q6_K: 8 (u / 2) + 2 t +
    // u % 2 (the sub-blocks whose codes one load of the block layout holds)
    uint32_t xo[2 * TT];
#pragma unroll
    for (int i = 0; i < 2 * TT; i++) {
        const int n = wave * 2 * TT + i;
        xo[i] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(min(n >> 3, mhave - 1)) * nks * 2048u +
                                               (kQ6K ? ((n >> 1) & 3) * 4096u + (n & 1) * 1024u : (n & 7) * 1024u));
    }
    auto load_x = [&](int u, int b) __attribute__((always_inline)) {
        const uint32_t uo = kQ6K ? static_cast<uint32_t>(u >> 1) * 16384u + (u & 1) * 2048u : static_cast<uint32_t>(u) * 8192u;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2 * TT; i++) load_lds16(rx, &As[b][(wave * 2 * TT + i) * 64], lane * 16u, xo[i] + uo);
        __builtin_amdgcn_sched_barrier(0);
    };
    struct Wu {
        v4u q[kPkR];
        v2u h[kPkR];  // Q4_K: {d | dmin << 16, scales of the unit's sub-blocks}; Q6_K: high bits
    };
    // Q6_K: scales (int8 x 4 of the lane's 64 elements) and d of the super-block in progress and
    // of the one requested
    uint32_t sc6[kPkR], sc6n[kPkR], d6n[kPkR];
    // (each group of loads kept whole and in program order: the waits count the loads issued
    // after the one they need)
    auto load_w = [&](int u, auto hc, Wu& w) __attribute__((always_inline)) {
        constexpr int h = decltype(hc)::value;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kPkR; j++) {
            if constexpr (kQ4K) {
                w.q[j] = __builtin_bit_cast(
                    v4u, __builtin_amdgcn_raw_buffer_load_b128(rq, ql, qo[j] + static_cast<uint32_t>(u) * 1024u, 2));
                const uint32_t hso = ho[j] + static_cast<uint32_t>(u >> 1) * 256u;
                if constexpr (h) w.h[j].y = __builtin_amdgcn_raw_buffer_load_b32(rh, hl, hso + 8u, 0);
                else w.h[j] = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(rh, hl, hso, 0));
            } else {
                const uint32_t bo = qo[j] + static_cast<uint32_t>(u >> 1) * static_cast<uint32_t>(kQ6Block);
                w.q[j] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rq, ql, bo + h * 1024u, 2));
                w.h[j] = __builtin_bit_cast(
                    v2u, __builtin_amdgcn_raw_buffer_load_b64(rq, ql, bo + static_cast<uint32_t>(kQ6Qh) + 8u * h, 0));
                if constexpr (h == 0) {
                    sc6n[j] = __builtin_amdgcn_raw_buffer_load_b32(rq, lane * 4u, bo + static_cast<uint32_t>(kQ6Sc), 0);
                    d6n[j] = __builtin_amdgcn_raw_buffer_load_b16(rq, c * 2u, bo + static_cast<uint32_t>(kQ6D), 0);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    floatx4 acc[kPkR][TT], dp[kPkR][TT];
    float dsb[kPkR];  // d of the super-block in progress (row c)
#pragma unroll
    for (int j = 0; j < kPkR; j++) {
        dsb[j] = 0.f;
#pragma unroll
        for (int i = 0; i < TT; i++) acc[j][i] = dp[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    if constexpr (kQ6K) {
#pragma unroll
        for (int j = 0; j < kPkR; j++) sc6[j] = sc6n[j] = d6n[j] = 0;
    }
    const uint32_t lds0 =
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)&As[0][0])) + lane * 16u;

    // unit of buffer b: k-step t = sub-block 4 h + t, lane (g, token c) takes its elements 8 g ..
    auto compute = [&](int b, auto hc, const Wu& w) __attribute__((always_inline)) {
        constexpr int h = decltype(hc)::value;
        v4u n[kPkR], nh[kQ6K ? kPkR : 1];
        uint32_t s6[kPkR];
#pragma unroll
        for (int j = 0; j < kPkR; j++) {
            n[j] = transpose4(w.q[j]);
            if constexpr (kQ4K) {
                s6[j] = w.h[j].y & 0x3F3F3F3Fu;
                if constexpr (h == 0) dsb[j] = h2f(w.h[j].x & 0xFFFFu);
            }
            if constexpr (kQ6K) {
                // of lane group t's two high-bit words the one of this lane's 16-element group, and
                // of its scales those of its sub-block 2 t + h in the low bytes
                nh[j] = transpose4(v4u{w.h[j].x, w.h[j].x, w.h[j].y, w.h[j].y});
                if constexpr (h == 0) {
                    sc6[j] = sc6n[j];
                    dsb[j] = h2f(d6n[j] & 0xFFFFu);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            v4u ah[TT], al[TT];
            read_a<TT>(lds0 + static_cast<uint32_t>(b) * (TT * 8192u), t, ah, al);
#pragma unroll
            for (int j = 0; j < kPkR; j++) {
                const uint32_t word = n[j][t];
                half8 B, Bl;
                if constexpr (kQ4K) {
                    // the scale of sub-block 4h + t in both halves
                    const f16x2 sv =
                        __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, s6[j], 0x04000400u + 0x00010001u * t)) -
                        f16x2{1024.0f16, 1024.0f16};
                    f16x2 q[4];
                    nibble_pairs(word, q);
                    // (2^10 times, so that no operand but zero is subnormal; odd codes are 16 times theirs)
                    const f16x2 se = sv * f16x2{1024.0f16, 1024.0f16}, so = sv * f16x2{64.0f16, 64.0f16};
                    B = operand8(q[0] * se, q[1] * se, q[2] * so, q[3] * so);
                } else {
                    const uint32_t hb = nh[j][t] >> (4 * (g & 1));
                    const uint32_t lo = (word & 0x0F0F0F0Fu) | ((hb & 0x03030303u) << 4);
                    const uint32_t hi = ((word >> 4) & 0x0F0F0F0Fu) | (((hb >> 2) & 0x03030303u) << 4);
                    // the scale of this lane's 16-element group: byte 2 h + g / 2 of lane group t's
                    // word, the weights at a quarter
                    const int scw = __builtin_amdgcn_ds_bpermute(4 * (16 * t + c), static_cast<int>(sc6[j]));
                    const _Float16 sf = static_cast<_Float16>(static_cast<int8_t>(scw >> (16 * h + 8 * (g >> 1))));
                    const f16x2 sv = f16x2{sf, sf} * f16x2{0.25f16, 0.25f16};
                    f16x2 bh[4], bl[4];
                    auto pr = [&](uint32_t codes, uint32_t sel, f16x2& oh, f16x2& ol) __attribute__((always_inline)) {
                        const f16x2 q = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, codes, sel)) -
                                        f16x2{1056.0f16, 1056.0f16};
                        oh = q * sv;
                        ol = __builtin_elementwise_fma(q, sv, -oh);
                    };
                    pr(lo, 0x04020400u, bh[0], bl[0]);
                    pr(lo, 0x04030401u, bh[1], bl[1]);
                    pr(hi, 0x04020400u, bh[2], bl[2]);
                    pr(hi, 0x04030401u, bh[3], bl[3]);
                    B = operand8(bh[0], bh[1], bh[2], bh[3]);
                    Bl = operand8(bl[0], bl[1], bl[2], bl[3]);
                }
                const bool fresh = h == 0 && t == 0;  // an accumulator per super-block
#pragma unroll
                for (int i = 0; i < TT; i++)
                    dp[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(half8, ah[i]), B, fresh ? floatx4{0.f, 0.f, 0.f, 0.f} : dp[j][i], 0, 0, 0);
                if constexpr (kQ6K) {
#pragma unroll
                    for (int i = 0; i < TT; i++)
                        dp[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, ah[i]), Bl, dp[j][i], 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < TT; i++)
                    dp[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, al[i]), B, dp[j][i], 0, 0, 0);
            }
        }
        if constexpr (h == 1) {  // the super-block's sum times d (row c)
#pragma unroll
            for (int j = 0; j < kPkR; j++) {
                const float d = dsb[j] * kUnit;
#pragma unroll
                for (int i = 0; i < TT; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[j][i][r] = fmaf(d, dp[j][i][r], acc[j][i][r]);
            }
        }
    };

    // Stage of unit u: its operands have landed (this wave's loads, then everyone's: everything
    // older than the weight loads of unit u + 1), and every wave has read unit u - 1, whose slot
    // the loads of unit u + 1 overwrite.  The weights of unit u + 2 are requested once those of
    // unit u are used up.
    Wu w0, w1;
    load_w(u0, std::integral_constant<int, 0>{}, w0);
    load_x(u0, 0);
    load_w(min(u0 + 1, last), std::integral_constant<int, 1>{}, w1);
    auto stage = [&](int u, auto hc, Wu& w) __attribute__((always_inline)) {
        constexpr int h = decltype(hc)::value;
        wait_vmcnt<h ? kWLoads0 : kWLoads1>();  // (the loads of unit u + 1)
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        load_x(min(u + 1, last), h ^ 1);
        compute(h, hc, w);
        load_w(min(u + 2, last), hc, w);
    };
    for (int u = u0; u < u1; u += 2) {
        stage(u, std::integral_constant<int, 0>{}, w0);
        stage(u + 1, std::integral_constant<int, 1>{}, w1);
    }
    wait_vmcnt<0>();  // nothing may land in LDS after the workgroup has ended

    if constexpr (kQ4K) {
        // min term over super-blocks [SB0, SB1), four per k-step: lane group g takes super-block
        // q + g, its eight sub-blocks in order (token side: scaled sums; row side: -32 dmin m_j)
        const int SB0 = u0 >> 1, SB1 = u1 >> 1;
        for (int q = SB0; q < SB1; q += 4) {
            const int sb = q + g, sbc = min(sb, SB1 - 1);
            const bool sv = sb < SB1;
            v4u ah[TT], al[TT];
#pragma unroll
            for (int i = 0; i < TT; i++) {
                const int tok = (mt0 + i) * 16 + c;
                const floatx4* p =
                    reinterpret_cast<const floatx4*>(a.xs + static_cast<size_t>(min(tok, M - 1)) * nks + 8 * sbc);
                const floatx4 x0 = p[0], x1 = p[1];
                const bool ok = sv && tok < M;
                float v[8];
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = ok ? x0[k] : 0.f, v[4 + k] = ok ? x1[k] : 0.f;
                hp_split8(v, ah[i], al[i]);
            }
            v4u hd[kPkR];
#pragma unroll
            for (int j = 0; j < kPkR; j++)
                hd[j] = __builtin_bit_cast(
                    v4u, __builtin_amdgcn_raw_buffer_load_b128(rh, hl + static_cast<uint32_t>(sbc) * 256u, ho[j], 0));
#pragma unroll
            for (int j = 0; j < kPkR; j++) {
                // -32 dmin m_j (32: small minima keep their low parts above fp16's smallest step);
                // a row with |dmin| past fp16's range of that takes -dmin m_j / 16 and its sums
                // 2^-9 times as large for the time being
                const float dmin = sv ? h2f(hd[j].x >> 16) : 0.f;
                float nd = -32.0f * dmin, back = 1.0f;
                const bool wide = __builtin_amdgcn_ballot_w64(fabsf(dmin) >= 128.0f) != 0;
                if (wide) {
                    float mx = fabsf(dmin);
                    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
                    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
                    if (mx >= 128.0f) nd = -0.0625f * dmin, back = 512.0f;
#pragma unroll
                    for (int i = 0; i < TT; i++) acc[j][i] *= 1.0f / back;
                }
                float cm[8];
#pragma unroll
                for (int k = 0; k < 8; k++)
                    cm[k] = nd * static_cast<float>((hd[j].w >> (8 * (k & 3) + 4 * (k >> 2))) & 0xFu);
                v4u bh, bl;
                hp_split8(cm, bh, bl);
                const half8 Bh = __builtin_bit_cast(half8, bh), Bl = __builtin_bit_cast(half8, bl);
#pragma unroll
                for (int i = 0; i < TT; i++) {
                    const half8 Ah = __builtin_bit_cast(half8, ah[i]), Al = __builtin_bit_cast(half8, al[i]);
                    acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ah, Bh, acc[j][i], 0, 0, 0);
                    acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ah, Bl, acc[j][i], 0, 0, 0);
                    acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Al, Bh, acc[j][i], 0, 0, 0);
                }
                if (wide) {
#pragma unroll
                    for (int i = 0; i < TT; i++) acc[j][i] *= back;
                }
            }
        }
    }

    // D lane (g, c) holds tokens 4g .. 4g + 3 of weight row c of each 16 x 16 tile
    int ex[TT][4];  // (all requested before the first is used)
#pragma unroll
    for (int i = 0; i < TT; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) ex[i][r] = a.xe[min((mt0 + i) * 16 + 4 * g + r, M - 1)];
#pragma unroll
    for (int i = 0; i < TT; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = (mt0 + i) * 16 + 4 * g + r;
            const float inv = ldexpf(1.0f, -ex[i][r]);
            float* y = Y + static_cast<size_t>(m) * a.ldy + nt0 * 16 + c;
#pragma unroll
            for (int j = 0; j < kPkR; j++)
                if (m < M && (nt0 + j) * 16 + c < N) y[16 * j] = acc[j][i][r] * inv;
        }
}

// Weights of the token rows whose outputs are summed again from the f32 inputs: a token with an
// infinite or NaN element, whose packed operands give NaN although its products with nonzero
// weights are infinite, or one whose sum overflows on the way.
struct PlainRows {
    const uint8_t* qs;
    const uint4* hdr;
    const float* X;
    int K;
};

__device__ __forceinline__ bool not_finite(float v) { return !(fabsf(v) <= 3.4028235e38f); }

// Scale and minimum of sub-block j under header h (Q4_K).
__device__ __forceinline__ float2 q4k_sub_scale(const uint4& h, int j) {
    return make_float2(h2f(h.x & 0xFFFFu) * static_cast<float>(((j < 4 ? h.y : h.z) >> (8 * (j & 3))) & 0x3Fu),
                       h2f(h.x >> 16) * static_cast<float>((h.w >> (8 * (j & 3) + 4 * (j >> 2))) & 0xFu));
}

// Products of the elements of x (row `x`, the wave's) that are not finite with V weight rows from
// `col` on, summed; the finite elements change nothing.  found: whether there is one; odd: whether a
// scale or minimum of the lane's weight rows is not finite (its rows need every product).  `live`: the
// lane's outputs count.  All lanes of the wave call it.
template <int V>
__device__ __forceinline__ void q4k_infinite_products(const PlainRows& pl, const float* x, int col, bool live, float (&t)[V],
                                                      bool& found, bool& odd) {
    const int lane = threadIdx.x & 63, S = pl.K / 256;
    found = odd = false;
#pragma unroll
    for (int k = 0; k < V; k++) t[k] = 0.f;
    const float4* xp = reinterpret_cast<const float4*>(x) + lane;
    float4 next = xp[0];
    for (int sb = 0; sb < S; sb++) {
        const float v[4] = {next.x, next.y, next.z, next.w};
        next = xp[64 * min(sb + 1, S - 1)];
#pragma unroll
        for (int k = 0; k < V; k++) {
            const uint32_t dm = pl.hdr[q4k_hdr_index(col + k, sb, S)].x;
            odd |= (dm & 0x7C00u) == 0x7C00u || (dm & 0x7C000000u) == 0x7C000000u;
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            for (uint64_t at = __builtin_amdgcn_ballot_w64(not_finite(v[e])); at; at &= at - 1) {
                const int src = __builtin_ctzll(at), el = 4 * src + e, j = el >> 5;
                const float xv = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v[e]), src));
                found = true;
                bool done = true;
#pragma unroll
                for (int k = 0; k < V; k++) {
                    const float2 sc = q4k_sub_scale(pl.hdr[q4k_hdr_index(col + k, sb, S)], j);
                    const uint32_t b = pl.qs[q4k_sub_offset(col + k, sb, j, S) + ((el & 31) >> 1)];
                    t[k] = fmaf(fmaf(sc.x, static_cast<float>(el & 1 ? b >> 4 : b & 15u), -sc.y), xv, t[k]);
                    done &= isnan(t[k]);
                }
                if (!__builtin_amdgcn_ballot_w64(live && !done)) return;  // (NaN stays NaN)
            }
        }
    }
}

// The dot of weight row `row` and x as a plain f32 sum, by the whole wave (a sub-block per lane).
__device__ __forceinline__ float q4k_plain_dot(const PlainRows& pl, const float* x, int row) {
    const int S = pl.K / 256;
    float acc = 0.f;
    for (int b = threadIdx.x & 63; b < 8 * S; b += 64) {
        const int sb = b >> 3, j = b & 7;
        const float2 sc = q4k_sub_scale(pl.hdr[q4k_hdr_index(row, sb, S)], j);
        const uint4 q = *reinterpret_cast<const uint4*>(pl.qs + q4k_sub_offset(row, sb, j, S));
        const float* xe = x + 32 * b;
#pragma unroll 1
        for (int k = 0; k < 4; k++) {
            uint32_t w = k == 0 ? q.x : k == 1 ? q.y : k == 2 ? q.z : q.w;
#pragma unroll
            for (int i = 0; i < 8; i++, w >>= 4)
                acc = fmaf(fmaf(sc.x, static_cast<float>(w & 15u), -sc.y), xe[8 * k + i], acc);
        }
    }
    return wave_sum(acc);
}

// Y = sum over the splits of the partial products, in split order (deterministic); four
// splits' loads at a time.  N a multiple of V and rows aligned to V floats: V columns per thread.
// PLAIN: an output that is not finite is summed again from the f32 inputs, by its wave: one infinite
// token of six, [14336 x 4096], 31 us the call (21 without; 1300 with a thread's serial sum for each
// output), of four, [4096 x 14336], 55 us (25; 4550).
template <int V, bool PLAIN>
__global__ void sum_splits_kernel(const float* __restrict__ P, float* __restrict__ Y, size_t n, int splits, int N,
                                  int ldy, PlainRows pl) {
    const size_t i0 = (blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x) * V;
    if (!PLAIN && i0 >= n) return;
    const size_t i = PLAIN ? (i0 < n ? i0 : n - V) : i0;  // (PLAIN: the last wave stays whole)
    typedef float fv __attribute__((ext_vector_type(V)));
    fv a = *reinterpret_cast<const fv*>(P + i);
    for (int z = 1; z < splits; z += 4) {
        fv v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = *reinterpret_cast<const fv*>(P + min(z + k, splits - 1) * n + i);
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (z + k < splits) a += v[k];
    }
    const size_t r = i / N, col = i % N;
    if constexpr (PLAIN) {
        bool bad = false;
#pragma unroll
        for (int k = 0; k < V; k++) bad |= not_finite(a[k]);
        uint64_t left = __builtin_amdgcn_ballot_w64(bad);
        while (left) {  // a token row of the wave at a time
            const uint32_t ru = __builtin_amdgcn_readlane(static_cast<uint32_t>(r), __builtin_ctzll(left));
            const float* x = pl.X + static_cast<size_t>(ru) * pl.K;
            const bool mine = bad && static_cast<uint32_t>(r) == ru;
            left &= ~__builtin_amdgcn_ballot_w64(mine);
            float t[V];
            bool found, odd;
            q4k_infinite_products<V>(pl, x, static_cast<int>(col), mine, t, found, odd);
#pragma unroll
            for (int k = 0; k < V; k++) {
                if (mine && found && !odd && not_finite(a[k])) a[k] = t[k];
                uint64_t each = __builtin_amdgcn_ballot_w64(mine && (!found || odd) && not_finite(a[k]));
                for (; each; each &= each - 1) {
                    const int src = __builtin_ctzll(each);
                    const float y = q4k_plain_dot(pl, x, __builtin_amdgcn_readlane(static_cast<int>(col) + k, src));
                    if ((threadIdx.x & 63) == src) a[k] = y;
                }
            }
        }
        if (i0 >= n) return;
    }
    *reinterpret_cast<fv*>(Y + r * ldy + col) = a;
}

// Token tiles per workgroup (the fewest workgroups of at most four, evenly filled) and K-splits
// (1..16, whole super-blocks each): the splits with the least modelled time, rounds of workgroups
// over the CUs x super-blocks per workgroup, ~2.2 / 3.0 / 3.6 / 4.1 us each at 1 .. 4 token tiles
// (workgroups past one per CU are counted as a further round), plus, when split, the partial sums
// written and summed ((splits + 1) m N floats at ~5 TB/s, and a launch).
struct PkPlan {
    int tt, splits, sb_per;
    double ns;  // the modelled time of the GEMM and its sums
};
PkPlan pk_plan(const DevWeight& w, size_t m) {
    const int S = static_cast<int>(w.cols / 256);
    const long most = w.format == LARQL_Q4_K ? 4 : 3;  // (four would spill for Q6_K)
    const long cus = current_device_cus(), mt = static_cast<long>((m + 15) / 16), gy = (mt + most - 1) / most;
    PkPlan best{static_cast<int>((mt + gy - 1) / gy), 1, S, -1.0};
    constexpr double kUnit[5] = {0, 2200, 3000, 3600, 4100};  // ns
    const double unit = kUnit[best.tt] * (w.format == LARQL_Q6_K ? 1.5 : 1.0);
    const long wgs = static_cast<long>((w.rows + kPkRows - 1) / kPkRows) * ((mt + best.tt - 1) / best.tt);
    for (int s = 1; s <= 16 && s <= S; s++) {
        const int per = (S + s - 1) / s, eff = (S + per - 1) / per;
        double cost = static_cast<double>((wgs * eff + cus - 1) / cus) * per * unit;
        if (eff > 1) cost += 3000.0 + (eff + 1) * static_cast<double>(m) * static_cast<double>(w.rows) * 0.0008;
        if (best.ns < 0 || cost < best.ns) best.splits = eff, best.sb_per = per, best.ns = cost;
    }
    return best;
}

size_t align4(size_t n) { return (n + 3) & ~size_t{3}; }

}  // namespace

// Q4_K operands of 2 GiB and more (X in f32, the nibbles), which the GEMM refuses.
static bool q4k_gemm_above_2gib(const DevWeight& w, size_t m) {
    return w.format == LARQL_Q4_K && (m > 0x7FFFFFFF / (4 * w.cols) || w.rows_pad > 0x7FFFFFFF / (w.cols / 2));
}

size_t gemm_x_pack_floats(size_t m, size_t cols) { return (m + 15) / 16 * 16 * cols; }

// workspace: the K-split partials (when split), and for a caller without packed rows those and
// their statistics
static size_t part_floats_of(const PkPlan& p, const DevWeight& w, size_t m, bool plain, bool packed) {
    const size_t parts = align4(p.splits > 1 || plain ? p.splits * m * w.rows : 0);
    return packed ? parts + 4 : parts + align4(gemm_row_stats_floats(m, w.cols)) + gemm_x_pack_floats(m, w.cols) + 4;
}
size_t gemm_f32_part_floats(const DevWeight& w, size_t m, bool plain, bool packed) {
    return part_floats_of(pk_plan(w, m), w, m, plain, packed);
}

size_t gemm_row_stats_floats(size_t m, size_t cols) { return m + 4 + m * (cols / 32); }

GemmRowStats gemm_row_stats_at(float* ws, size_t m, size_t /*cols*/) {
    // the exponents, then the sub-block sums from a 16-byte boundary (float4 reads)
    const uintptr_t at = reinterpret_cast<uintptr_t>(ws + m);
    return {reinterpret_cast<int*>(ws), reinterpret_cast<float*>((at + 15) & ~uintptr_t{15}), nullptr};
}

void launch_gemm_row_stats(const float* X, size_t m, size_t cols, const GemmRowStats& st, hipStream_t s) {
    if (m == 0) return;
    if (cols % 32 != 0 || cols > 0x7FFFFFFF) fail(LARQL_HIP_ERR_INVALID, "GEMM row statistics: cols must be a multiple of 32");
    row_exp_kernel<<<dim3(static_cast<unsigned>(m)), dim3(256), 0, s>>>(X, static_cast<int>(cols), st.xe, st.xs);
    LARQL_HIP_CHECK(hipGetLastError());
}

void launch_gemm_x_pack(const float* X, size_t m, size_t cols, const GemmRowStats& st, hipStream_t s) {
    if (m == 0) return;
    const size_t mt = (m + 15) / 16;
    if (cols % 32 != 0 || !st.xp || !st.xe || m > 0x7FFFFFFF / cols)
        fail(LARQL_HIP_ERR_INVALID, "GEMM operand packing: bad arguments");
    // (grid y is at most 65535 tiles: longer batches in several launches)
    for (size_t t = 0; t < mt; t += 65535) {
        const size_t nt = mt - t < 65535 ? mt - t : 65535, r0 = 16 * t;
        x_pack_kernel<<<dim3(static_cast<unsigned>((cols + 127) / 128), static_cast<unsigned>(nt)), dim3(256), 0, s>>>(
            X + r0 * cols, st.xe + r0, reinterpret_cast<v4u*>(st.xp + r0 * cols), static_cast<int>(m - r0),
            static_cast<int>(cols));
        LARQL_HIP_CHECK(hipGetLastError());
    }
}

void launch_gemm_pack_rows(const float* X, size_t m, size_t cols, const GemmRowStats& st, hipStream_t s) {
    if (cols > static_cast<size_t>(kFusedRowMax)) {
        launch_gemm_row_stats(X, m, cols, st, s);
        launch_gemm_x_pack(X, m, cols, st, s);
        return;
    }
    if (m > 0x7FFFFF00) fail(LARQL_HIP_ERR_INVALID, "GEMM operand packing: too many tokens");
    ResidRows r;
    r.hin = X;
    r.st = st;
    r.m = static_cast<int>(m);
    r.n = static_cast<int>(cols);
    launch_resid_norm_stats_rows(r, s);
}

// Q4_K batches small enough that this GEMM beats the fp16 one (prefill.hip), whose workgroups
// are 256 tokens whatever the batch: ~2.2 us per super-block of K and round of 80-row
// workgroups, against the plan's time and its two other launches.  Measured [14336 x 4096]: 6
// tokens 22.6 against 39.5 us, 64 tokens 41 against 42, 96 tokens 49 against 45; [4096 x 14336]:
// 6 tokens 30 against 125, 192 tokens 83 against 145; [10240 x 2560]: 32 tokens 22 against 28,
// 64 tokens 31 against 28.
size_t gemm_f32_small_batch(const DevWeight& w, size_t m, size_t rows) {
    if (w.format != LARQL_Q4_K || m < 2 || m > kSmallBatchMax || q4k_gemm_above_2gib(w, m)) return 0;
    const size_t wgs = ((w.rows_pad / 16 + 4) / 5) * ((m + 255) / 256), cus = static_cast<size_t>(current_device_cus());
    const double other = 6500.0 + static_cast<double>((wgs + cus - 1) / cus) * static_cast<double>(w.cols / 256) * 2200.0;
    const PkPlan p = pk_plan(w, m);
    return 1.45 * p.ns + 8000.0 < other ? part_floats_of(p, w, std::max(m, rows), true, false) : 0;
}

void launch_gemm_f32(const DevWeight& w, const float* X, float* Y, size_t m, float* part, size_t part_floats,
                     hipStream_t s, size_t ldy, const GemmRowStats* pre, GemmSplits* defer, bool plain) {
    if (ldy == 0) ldy = w.rows;
    if (ldy < w.rows || ldy > 0x7FFFFFFF) fail(LARQL_HIP_ERR_INVALID, "f32 GEMM: bad output row stride");
    if (defer && ldy != w.rows) fail(LARQL_HIP_ERR_INVALID, "f32 GEMM: deferred split sums need dense output rows");
    if (w.format != LARQL_Q4_K && w.format != LARQL_Q6_K) fail(LARQL_HIP_ERR_UNSUPPORTED, "f32 GEMM: Q4_K or Q6_K weights");
    if (pre && (!pre->xe || (w.format == LARQL_Q4_K && !pre->xs)))
        fail(LARQL_HIP_ERR_INVALID, "f32 GEMM: incomplete row statistics");
    if (m == 0) return;
    if (m > 0x7FFFFFFF / w.cols) fail(LARQL_HIP_ERR_INVALID, "f32 GEMM: too many tokens");
    if (q4k_gemm_above_2gib(w, m)) fail(LARQL_HIP_ERR_UNSUPPORTED, "f32 GEMM: operands above 2 GiB");
    const PkPlan p = pk_plan(w, m);
    if (plain && (w.format != LARQL_Q4_K || defer)) fail(LARQL_HIP_ERR_INVALID, "f32 GEMM: plain sums of Q4_K outputs only");
    if (!part || part_floats < gemm_f32_part_floats(w, m, plain, pre && pre->xp)) fail(LARQL_HIP_ERR_INVALID, "f32 GEMM: workspace too small");
    const bool parts = p.splits > 1 || plain;  // the GEMM writes partial products, summed after it
    float* at = part + align4(parts ? p.splits * m * w.rows : 0);
    GemmRowStats st;
    if (pre) {
        st = *pre;
    } else {
        st = gemm_row_stats_at(at, m, w.cols);
        if (w.format != LARQL_Q4_K) st.xs = nullptr;
    }
    if (!st.xp) {
        const uintptr_t xp = reinterpret_cast<uintptr_t>(at + align4(gemm_row_stats_floats(m, w.cols)));
        st.xp = reinterpret_cast<float*>((xp + 15) & ~uintptr_t{15});
        if (pre) launch_gemm_x_pack(X, m, w.cols, st, s);
        else launch_gemm_pack_rows(X, m, w.cols, st, s);
    }
    PkArgs a{};
    a.qs = w.qs;
    a.hdr = reinterpret_cast<const uint8_t*>(w.hdr);
    a.XP = reinterpret_cast<const v4u*>(st.xp);
    a.xe = st.xe;
    a.xs = st.xs;
    a.Y = parts ? part : Y;
    a.ypart = m * w.rows;
    a.M = static_cast<int>(m);
    a.N = static_cast<int>(w.rows);
    a.K = static_cast<int>(w.cols);
    a.ntiles = static_cast<int>(w.rows_pad / 16);
    a.mtiles = static_cast<int>((m + 15) / 16);
    a.sb_per = p.sb_per;
    a.ldy = static_cast<int>(parts ? w.rows : ldy);
    a.gx = static_cast<int>((w.rows + kPkRows - 1) / kPkRows);
    a.gy = (a.mtiles + p.tt - 1) / p.tt;
    a.gz = p.splits;
    const size_t grid = (static_cast<size_t>(a.gx) * a.gz + 7) / 8 * 8 * a.gy;
    if (grid > 0x7FFFFFFF) fail(LARQL_HIP_ERR_INVALID, "f32 GEMM: grid too large");
    auto go = [&](auto f, auto t) {
        pk_gemm_kernel<decltype(f)::value, decltype(t)::value>
            <<<dim3(static_cast<unsigned>(grid)), dim3(kPkThreads), 0, s>>>(a);
    };
    auto fmt = [&](auto f) {
        if (p.tt == 1) go(f, std::integral_constant<int, 1>{});
        else if (p.tt == 2) go(f, std::integral_constant<int, 2>{});
        else if (p.tt == 3) go(f, std::integral_constant<int, 3>{});
        else if constexpr (decltype(f)::value == LARQL_Q4_K) go(f, std::integral_constant<int, 4>{});
    };
    if (w.format == LARQL_Q4_K) fmt(std::integral_constant<int, LARQL_Q4_K>{});
    else fmt(std::integral_constant<int, LARQL_Q6_K>{});
    LARQL_HIP_CHECK(hipGetLastError());
    if (defer) *defer = {p.splits > 1 ? part : nullptr, p.splits};
    if (parts && !defer) {
        const size_t n = m * w.rows;
        const int N = static_cast<int>(w.rows), ld = static_cast<int>(ldy);
        const PlainRows pl{w.qs, w.hdr, X, static_cast<int>(w.cols)};
        auto sum = [&](auto v) {
            constexpr int V = decltype(v)::value;
            const dim3 g(static_cast<unsigned>((n / V + 255) / 256)), b(256);
            if (plain) sum_splits_kernel<V, true><<<g, b, 0, s>>>(part, Y, n, p.splits, N, ld, pl);
            else sum_splits_kernel<V, false><<<g, b, 0, s>>>(part, Y, n, p.splits, N, ld, pl);
        };
        if (N % 4 == 0 && ld % 4 == 0 && reinterpret_cast<uintptr_t>(Y) % 16 == 0) sum(std::integral_constant<int, 4>{});
        else sum(std::integral_constant<int, 1>{});
        LARQL_HIP_CHECK(hipGetLastError());
    }
}

}  // namespace larql
