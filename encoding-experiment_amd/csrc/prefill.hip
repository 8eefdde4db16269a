// Quantized prefill: Y[M x N] = X[M x K] . deq(W)^T for a Q4_K weight W [N x K],
// M tokens at once (M = 512 in the prefill workload).
//
// Reference semantics: the trait's prefill (LC/src/backend.rs:143-152) runs, per token,
// the Q4_K matvec (LC/src/cpu/ops/q4k_matvec.rs:31-90; the Metal prefill is that matvec
// in a loop over positions, LC/src/metal/prefill.rs:21-110).  Here the M matvecs are one
// GEMM on the matrix cores, v_mfma_f32_16x16x32_f16 with f32 accumulation:
//   * x16_pack_kernel converts X to fp16 once, laid out as ready-made A operands:
//     one 1 KB block (64 lanes x 8 halves) per (16 tokens, super-block, half, step);
//   * the GEMM (q4k_gemm_shared_kernel) streams the tile-major Q4_K weights and
//     dequantizes each 16-row tile and k-step once per 256 tokens into fp16 B operands in
//     LDS, w = (1024 + q) * (d sc_j) - (1024 d sc_j + dmin m_j) in one f32 fma per element,
//     rounded to fp16 (the same value as d sc_j q - dmin m_j, to ~2^-14 d sc_j);
//   * each of its eight waves multiplies its own 32 tokens, A operands straight from the
//     packed X into registers, by the shared B operands of 80 weight rows.
// The MFMA k order within a step is free as long as A and B agree: lane (g, c) of step s
// in half h supplies elements 8s + {0,4,1,5,2,6,3,7} of sub-block 4h + g (the order in
// which the nibble bytes unpack), and x16_pack_kernel writes X in that order.
// fp16 operands carry 11 significant bits: over K = 2560 random terms the error is
// ~1e-4 of max|Y|, inside the 1e-3 bar.
#include <type_traits>

#include "device_common.h"
#include "larql_hip_internal.h"

namespace larql {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

constexpr int kMt = 4;  // the packed X is padded to kMt tiles of 16 tokens

// X [M x K] f32 -> XP[mt][sb][h][s][lane] (uint4 = 8 halves); rows >= M are zeros.
// Workgroup (sb, mt): the 16 x 256 block of X, read row-major into LDS, written out as
// its 512 operand uint4 in order.
__global__ __launch_bounds__(256) void x16_pack_kernel(const float* __restrict__ X, v4u* __restrict__ XP, int M,
                                                       int K) {
    __shared__ float xs[16][256 + 4];
    const int sb = blockIdx.x, S = gridDim.x, mt = blockIdx.y, tid = threadIdx.x;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int idx = tid + 256 * r, row = idx >> 6, c4 = idx & 63;
        const size_t m = static_cast<size_t>(mt) * 16 + row;
        const float4 v = m < static_cast<size_t>(M)
                             ? *reinterpret_cast<const float4*>(X + m * K + 256 * sb + 4 * c4)
                             : make_float4(0.f, 0.f, 0.f, 0.f);
        *reinterpret_cast<float4*>(&xs[row][4 * c4]) = v;
    }
    __syncthreads();
    auto pk = [](float lo, float hi) __attribute__((always_inline)) {
        return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<_Float16>(lo))) |
               (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<_Float16>(hi))) << 16);
    };
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int t = tid + 256 * q, h = t >> 8, s = (t >> 6) & 3, lane = t & 63;
        const int g = lane >> 4, i = lane & 15;
        const float* p = &xs[i][32 * (4 * h + g) + 8 * s];
        const float4 a = *reinterpret_cast<const float4*>(p);
        const float4 b = *reinterpret_cast<const float4*>(p + 4);
        // element order 0, 4, 1, 5, 2, 6, 3, 7
        const v4u out = {pk(a.x, b.x), pk(a.y, b.y), pk(a.z, b.z), pk(a.w, b.w)};
        XP[(static_cast<size_t>(mt) * S + sb) * 512 + t] = out;
    }
}

// Two weights from a dword holding two fp16 values v: (v * sc + c) in f32, each rounded
// to fp16 (v_fma_mix, fp16 source operand with f32 scale and offset).
__device__ __forceinline__ uint32_t mix2(uint32_t p, float sc, float c) {
    uint32_t r;
    asm("v_fma_mixlo_f16 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=&v"(r) : "v"(p), "v"(sc), "v"(c));
    asm("v_fma_mixhi_f16 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(r) : "v"(p), "v"(sc), "v"(c));
    return r;
}

// (m & x) | magic for a magic with no bits under m.
__device__ __forceinline__ uint32_t bfi(uint32_t m, uint32_t x, uint32_t magic) {
    uint32_t r;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "v"(m), "v"(x), "s"(magic));
    return r;
}

// Scale and offsets of one sub-block for the two nibble positions of a byte: the low
// nibble q becomes the fp16 1024 + q, the high nibble (left in place) 1024 + 16 q, so
//   w = (1024 + q) sc - (1024 sc + mn) = (1024 + 16 q) (sc / 16) - (64 sc + mn).
struct SubScale {
    float sc, c_lo, sc16, c_hi;
};

// Eight weights (elements 8s + 0, 4, 1, 5, 2, 6, 3, 7) from the nibble dword of step s;
// byte i holds elements 2i (low nibble) and 2i + 1 (high nibble).
__device__ __forceinline__ half8 deq8(uint32_t u, const SubScale& k, uint32_t m_lo, uint32_t m_hi) {
    constexpr uint32_t kMagic = 0x64006400u;  // fp16 1024 in both halves
    const uint32_t u8 = u >> 8;
    v4u r;
    r.x = mix2(bfi(m_lo, u, kMagic), k.sc, k.c_lo);     // elements 0, 4
    r.y = mix2(bfi(m_hi, u, kMagic), k.sc16, k.c_hi);   // 1, 5
    r.z = mix2(bfi(m_lo, u8, kMagic), k.sc, k.c_lo);    // 2, 6
    r.w = mix2(bfi(m_hi, u8, kMagic), k.sc16, k.c_hi);  // 3, 7
    return __builtin_bit_cast(half8, r);
}

// ── fp16 operands with the dequantization shared by the workgroup ─────────
// 256 tokens x 80 weight rows per workgroup (grid 128 x 2 = one workgroup per CU at
// M = 512, N = 10240), eight waves, two per SIMD (one wave's loads wait while the other
// multiplies).  Each unit (half super-block, 128 k, four k-steps of 32) is dequantized
// once: wave w turns k-step w % 4 of tiles 0-2 (w < 4) or 3-4 (w >= 4) into fp16 B
// operands in LDS, then every wave multiplies its own 32 tokens (two A tiles from the
// packed X, straight into registers) by the B operands of all four steps.  Per unit and
// SIMD: five 8-weight dequantizations and their scales against 80 MFMAs, where a wave that
// dequantizes its own rows for its own 64 tokens does twenty.
constexpr int kShTiles = 5;                   // 16-row weight tiles per workgroup
constexpr int kShWaves = 8;
constexpr int kShThreads = 64 * kShWaves;
constexpr int kShMt = 2;                      // 16-token tiles per wave
constexpr int kShTok = 16 * kShMt * kShWaves;  // 256 tokens per workgroup
constexpr int kShDq = 3;                      // most tiles one wave dequantizes per unit

__global__ __launch_bounds__(kShThreads) void q4k_gemm_shared_kernel(const uint8_t* __restrict__ qs,
                                                                     const v4u* __restrict__ hdr,
                                                                     const v4u* __restrict__ XP, float* __restrict__ Y,
                                                                     int M, int N, int K, int ntiles, int mtiles) {
    __shared__ v4u Bs[3][kShTiles][4][64];  // B operands of three units (60 KB)
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int S = K / 256;
    const int n = 2 * S;  // units: (super-block u / 2, half u % 2)
    const int nt0 = blockIdx.x * kShTiles;
    const int mtw = blockIdx.y * (kShTok / 16) + wave * kShMt;  // first 16-token tile of this wave
    const int step = wave & 3;                                  // the k-step this wave dequantizes
    const int dj0 = wave < 4 ? 0 : 3, dn = wave < 4 ? 3 : 2;    // and its tiles dj0 .. dj0 + dn - 1

    // qs block (sb 0, half 0) of dequantized tile jj, offset to this wave's dword of the
    // lane's 16-byte nibble slot, and the tile's header block
    uint32_t qo[kShDq], ho[kShDq];
#pragma unroll
    for (int jj = 0; jj < kShDq; jj++) {
        const uint32_t t = static_cast<uint32_t>(min(nt0 + dj0 + min(jj, dn - 1), ntiles - 1));
        qo[jj] = __builtin_amdgcn_readfirstlane(t * S * 2048u + 4u * step);
        ho[jj] = __builtin_amdgcn_readfirstlane(t * S * 256u);
    }
    // Every load is a raw buffer load: the wave-uniform part of the offset in the scalar
    // operand, the lane's byte offset in the vector operand, so no vector ALU goes to
    // addresses.  All offsets are in range (tiles clamped, units below n).
    const uint32_t lo16 = lane * 16u, lc16 = c * 16u;
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(qs), 0, static_cast<int>(static_cast<uint32_t>(ntiles) * S * 2048u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<v4u*>(hdr), 0, static_cast<int>(static_cast<uint32_t>(ntiles) * S * 256u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<v4u*>(XP), 0, static_cast<int>(static_cast<uint32_t>(mtiles) * n * 4096u), 0x00020000);
    // A tile i of this wave: XP[(mt n + u) 256 + s 64 + lane], mt clamped into the packed X
    // (tiles past it hold tokens >= M, whose rows are not stored)
    uint32_t xo[kShMt];
#pragma unroll
    for (int i = 0; i < kShMt; i++)
        xo[i] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(min(mtw + i, mtiles - 1)) * n * 4096u);

    struct Au {
        v4u v[kShMt][4];  // [tile][k-step]
    };
    auto load_a = [&a_rs = rx, &xo, lo16](int u, Au& a) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kShMt; i++)
#pragma unroll
            for (int s = 0; s < 4; s++)
                a.v[i][s] = __builtin_bit_cast(
                    v4u, __builtin_amdgcn_raw_buffer_load_b128(a_rs, lo16, xo[i] + u * 4096u + s * 1024u, 0));
    };
    struct Wu {
        uint32_t q[kShDq];
        v4u hd[kShDq];
    };
    auto load_w = [&qo, &ho, rq, rh, lo16, lc16](int u, Wu& w) __attribute__((always_inline)) {
#pragma unroll
        for (int jj = 0; jj < kShDq; jj++) {
            w.q[jj] = __builtin_amdgcn_raw_buffer_load_b32(rq, lo16, qo[jj] + u * 1024u, 0);
            w.hd[jj] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rh, lc16, ho[jj] + (u >> 1) * 256u, 0));
        }
    };
    uint32_t m_lo = 0x000F000Fu, m_hi = 0x00F000F0u;
    asm volatile("" : "+v"(m_lo), "+v"(m_hi));  // keep the masks in VGPRs
    // this wave's k-step of unit u for its tiles -> LDS buffer b
    auto dequant = [&](int u, const Wu& w, int b) __attribute__((always_inline)) {
        const int h = u & 1;
#pragma unroll
        for (int jj = 0; jj < kShDq; jj++) {
            if (jj >= dn) break;
            const float d = h2f(w.hd[jj].x & 0xFFFFu), dmin = h2f(w.hd[jj].x >> 16);
            const uint32_t scw = h ? w.hd[jj].z : w.hd[jj].y;
            const float sc = d * static_cast<float>((scw >> (8 * g)) & 0x3Fu);
            const float mn = dmin * static_cast<float>((w.hd[jj].w >> (8 * g + 4 * h)) & 0xFu);
            SubScale k;
            k.sc = sc;
            // -(1024 sc + mn) as one fma with negated operands (no separate negation)
            k.c_lo = __builtin_fmaf(-1024.f, sc, -mn);
            k.sc16 = sc * 0.0625f;
            k.c_hi = __builtin_fmaf(-64.f, sc, -mn);
            Bs[b][dj0 + jj][step][lane] = __builtin_bit_cast(v4u, deq8(w.q[jj], k, m_lo, m_hi));
        }
    };
    floatx4 acc[kShMt][kShTiles];
#pragma unroll
    for (int i = 0; i < kShMt; i++)
#pragma unroll
        for (int j = 0; j < kShTiles; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const bool live = mtw < mtiles;  // wave-uniform: this wave has tokens to multiply
    // the B operands of step s + 1 are read from LDS before the MFMAs of step s are issued
    auto mfma = [&](const Au& a, int b) __attribute__((always_inline)) {
        if (!live) return;
        v4u bq[2][kShTiles];
#pragma unroll
        for (int j = 0; j < kShTiles; j++) bq[0][j] = Bs[b][j][0][lane];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (s < 3) {
#pragma unroll
                for (int j = 0; j < kShTiles; j++) bq[(s + 1) & 1][j] = Bs[b][j][s + 1][lane];
            }
            __builtin_amdgcn_sched_barrier(0);  // keep those reads ahead of this step's MFMAs
#pragma unroll
            for (int i = 0; i < kShMt; i++)
#pragma unroll
                for (int j = 0; j < kShTiles; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a.v[i][s]),
                                                                       __builtin_bit_cast(half8, bq[s & 1][j]),
                                                                       acc[i][j], 0, 0, 0);
        }
    };

    // Three-unit ring: unit u multiplies from LDS buffer u % 3 and A registers u % 3 and
    // was dequantized from weight registers u % 3.  In the stage of unit u the wave first
    // dequantizes unit u + 1 (its weights were requested two stages before) into buffer
    // (u + 1) % 3, requests the weights of unit u + 3, multiplies unit u, then requests the
    // A tiles of unit u + 3 into the registers it just used.  A barrier ends each stage:
    // buffer (u + 1) % 3 is complete, and the buffer the next stage overwrites was last
    // read two stages before.  Loads past the last unit re-read it (unused).
    Au a0, a1, a2;
    Wu w0, w1, w2;
    load_w(0, w0);
    load_a(0, a0);
    load_w(min(1, n - 1), w1);
    load_a(min(1, n - 1), a1);
    load_w(min(2, n - 1), w2);
    load_a(min(2, n - 1), a2);
    dequant(0, w0, 0);
    __syncthreads();
    auto stage = [&](int u, int b, Au& a, const Wu& wn, Wu& wr) __attribute__((always_inline)) {
        if (u + 1 < n) dequant(u + 1, wn, b == 2 ? 0 : b + 1);
        load_w(min(u + 3, n - 1), wr);
        mfma(a, b);
        load_a(min(u + 3, n - 1), a);
        __syncthreads();
    };
    int u = 0;
    for (; u + 3 <= n; u += 3) {
        stage(u, 0, a0, w1, w0);
        stage(u + 1, 1, a1, w2, w1);
        stage(u + 2, 2, a2, w0, w2);
    }
    if (u < n) stage(u, 0, a0, w1, w0);
    if (u + 1 < n) stage(u + 1, 1, a1, w2, w1);

    // D lane (g, c) holds rows 4g .. 4g + 3 of column c of each 16 x 16 tile
    if (!live) return;
#pragma unroll
    for (int i = 0; i < kShMt; i++)
#pragma unroll
        for (int j = 0; j < kShTiles; j++) {
            const int col = (nt0 + j) * 16 + c;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = (mtw + i) * 16 + 4 * g + r;
                if (m < M && col < N) Y[static_cast<size_t>(m) * N + col] = acc[i][j][r];
            }
        }
}

}  // namespace

size_t q4k_gemm_ws_bytes(size_t m, size_t cols) {
    const size_t m_pad = (m + 16 * kMt - 1) / (16 * kMt) * (16 * kMt);
    return m_pad * cols * sizeof(uint16_t);
}

void launch_q4k_gemm(const DevWeight& w, const float* X, float* Y, size_t m, void* ws, hipStream_t s) {
    if (w.format != LARQL_Q4_K) fail(LARQL_HIP_ERR_UNSUPPORTED, "prefill GEMM: Q4_K weights only");
    if (m == 0) return;
    if (!ws) fail(LARQL_HIP_ERR_INVALID, "prefill GEMM: no workspace");
    if (m > 0x7FFFFFFF / w.cols) fail(LARQL_HIP_ERR_INVALID, "prefill GEMM: too many tokens");
    const size_t mtiles = (m + 16 * kMt - 1) / (16 * kMt) * kMt;  // 16-token tiles, padded
    // the kernel addresses X, the nibbles and the headers with 31-bit buffer offsets
    if (mtiles * 16 * w.cols * 2 > 0x7FFFFFFF || w.rows_pad * (w.cols / 2) > 0x7FFFFFFF)
        fail(LARQL_HIP_ERR_UNSUPPORTED, "prefill GEMM: operands above 2 GiB");
    x16_pack_kernel<<<dim3(static_cast<unsigned>(w.cols / 256), static_cast<unsigned>(mtiles)), dim3(256), 0, s>>>(
        X, static_cast<v4u*>(ws), static_cast<int>(m), static_cast<int>(w.cols));
    LARQL_HIP_CHECK(hipGetLastError());
    const size_t ntiles = w.rows_pad / 16;
    const dim3 grid(static_cast<unsigned>((ntiles + kShTiles - 1) / kShTiles),
                    static_cast<unsigned>((mtiles * 16 + kShTok - 1) / kShTok));
    q4k_gemm_shared_kernel<<<grid, dim3(kShThreads), 0, s>>>(
        w.qs, reinterpret_cast<const v4u*>(w.hdr), static_cast<const v4u*>(ws), Y, static_cast<int>(m),
        static_cast<int>(w.rows), static_cast<int>(w.cols), static_cast<int>(ntiles), static_cast<int>(mtiles));
    LARQL_HIP_CHECK(hipGetLastError());
}

}  // namespace larql
