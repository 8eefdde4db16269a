// f32 matrix products of the trait: ComputeBackend::matmul (C = A . B) and matmul_transb
// (C = A . B^T), LC/src/backend.rs:27-31 (the Metal backend runs both as tiled sgemm
// kernels, LC/src/metal/f32_ops.rs:93-140).
//
// Every element of C is one f32 fma chain over k = 0 .. K-1 starting from +0, the
// canonical order of the gate-score kernel, so a product is reproducible bit for bit and
// equals the oracle's chain; the reference CPU path (matrixmultiply's blocked sgemm) sums in
// its own order, within f32 rounding of this one.
//
// Two forms: lanes (a chain per lane, the other side's values as scalar operands), and 256 x 64
// tiles for large products.
#include <algorithm>
#include <type_traits>

#include "device_common.h"
#include "f32_lane.h"
#include "larql_hip_internal.h"

namespace larql {

namespace {

constexpr int kGThreads = 256;
constexpr int kGTileR = 256, kGTileC = 64, kGKs = 16;

// Workgroup tile: 256 "rows" (operand R) x 64 "columns" (operand C), thread tile 8 x 8,
// K in LDS stages of 16 (double-buffered, the next stage's global loads held in registers
// while the current one is consumed).  Each operand may be k-minor in memory (a row of K
// floats per row / column) or k-major (a row of the other dimension per k); the LDS tiles
// are k-major either way.  The launcher puts the larger of m and n on the 256 side and
// stores C transposed when it swaps them.  Loads are scalar and predicated (any K, any
// alignment); rows and columns past the matrix are clamped duplicates, never stored.
template <bool R_KMAJOR, bool C_KMAJOR, bool OUT_T>
__global__ __launch_bounds__(kGThreads) void f32_gemm_kernel(const float* __restrict__ R, size_t ldr,
                                                             const float* __restrict__ Cm, size_t ldc,
                                                             float* __restrict__ out, size_t ldo, int Rn, int Cn,
                                                             int K) {
    __shared__ float Rs[2][kGKs][kGTileR];
    __shared__ float Cs[2][kGKs][kGTileC];
    const int tid = threadIdx.x;
    const int r0 = blockIdx.y * kGTileR, c0 = blockIdx.x * kGTileC;
    const int tr = tid & 31, tc = tid >> 5;  // rows r0 + 8 tr .., columns c0 + 8 tc ..

    // R stage: k-minor, thread = row r0 + tid, 16 consecutive k; k-major, thread =
    // (rows r0 + 4 (tid & 63) .. + 3, k 4 (tid >> 6) .. + 3)
    float rv[16];
    auto rload = [&](int k0) __attribute__((always_inline)) {
        if constexpr (!R_KMAJOR) {
            const float* p = R + static_cast<size_t>(min(r0 + tid, Rn - 1)) * ldr;
#pragma unroll
            for (int i = 0; i < 16; i++) rv[i] = k0 + i < K ? p[k0 + i] : 0.f;
        } else {
            const int rr = 4 * (tid & 63), kk = 4 * (tid >> 6);
#pragma unroll
            for (int a = 0; a < 4; a++)
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    const int k = k0 + kk + a;
                    rv[4 * a + b] = k < K ? R[static_cast<size_t>(k) * ldr + min(r0 + rr + b, Rn - 1)] : 0.f;
                }
        }
    };
    auto rstore = [&](int buf) __attribute__((always_inline)) {
        if constexpr (!R_KMAJOR) {
#pragma unroll
            for (int i = 0; i < 16; i++) Rs[buf][i][tid] = rv[i];
        } else {
            const int rr = 4 * (tid & 63), kk = 4 * (tid >> 6);
#pragma unroll
            for (int a = 0; a < 4; a++)
                *reinterpret_cast<float4*>(&Rs[buf][kk + a][rr]) =
                    make_float4(rv[4 * a], rv[4 * a + 1], rv[4 * a + 2], rv[4 * a + 3]);
        }
    };
    // C stage: k-minor, thread = (column c0 + (tid & 63), k 4 (tid >> 6) .. + 3); k-major,
    // thread = (columns c0 + 4 (tid & 15) .. + 3, k tid >> 4)
    float cv[4];
    auto cload = [&](int k0) __attribute__((always_inline)) {
        if constexpr (!C_KMAJOR) {
            const float* p = Cm + static_cast<size_t>(min(c0 + (tid & 63), Cn - 1)) * ldc;
            const int kk = k0 + 4 * (tid >> 6);
#pragma unroll
            for (int i = 0; i < 4; i++) cv[i] = kk + i < K ? p[kk + i] : 0.f;
        } else {
            const int k = k0 + (tid >> 4), cc = 4 * (tid & 15);
#pragma unroll
            for (int i = 0; i < 4; i++)
                cv[i] = k < K ? Cm[static_cast<size_t>(k) * ldc + min(c0 + cc + i, Cn - 1)] : 0.f;
        }
    };
    auto cstore = [&](int buf) __attribute__((always_inline)) {
        if constexpr (!C_KMAJOR) {
            const int kk = 4 * (tid >> 6);
#pragma unroll
            for (int i = 0; i < 4; i++) Cs[buf][kk + i][tid & 63] = cv[i];
        } else {
            *reinterpret_cast<float4*>(&Cs[buf][tid >> 4][4 * (tid & 15)]) = make_float4(cv[0], cv[1], cv[2], cv[3]);
        }
    };

    float acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) acc[i][j] = 0.f;

    const int nk = (K + kGKs - 1) / kGKs;
    if (nk > 0) {
        rload(0);
        cload(0);
        rstore(0);
        cstore(0);
    }
    __syncthreads();
    for (int s = 0; s < nk; s++) {
        const int b = s & 1;
        if (s + 1 < nk) {
            rload((s + 1) * kGKs);
            cload((s + 1) * kGKs);
        }
        // the last stage runs only its real k: no padded term enters a chain
        const int kend = min(kGKs, K - s * kGKs);
#pragma unroll 2
        for (int k = 0; k < kend; k++) {
            const float4 ra = *reinterpret_cast<const float4*>(&Rs[b][k][tr * 8]);
            const float4 rb = *reinterpret_cast<const float4*>(&Rs[b][k][tr * 8 + 4]);
            const float4 ca = *reinterpret_cast<const float4*>(&Cs[b][k][tc * 8]);
            const float4 cb = *reinterpret_cast<const float4*>(&Cs[b][k][tc * 8 + 4]);
            const float rw[8] = {ra.x, ra.y, ra.z, ra.w, rb.x, rb.y, rb.z, rb.w};
            const float cw[8] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
                for (int j = 0; j < 8; j++) acc[i][j] = fmaf(cw[j], rw[i], acc[i][j]);
        }
        // buffer b ^ 1 was last read in stage s - 1, before that stage's barrier
        if (s + 1 < nk) {
            rstore(b ^ 1);
            cstore(b ^ 1);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int r = r0 + tr * 8 + i;
        if (r >= Rn) continue;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int c = c0 + tc * 8 + j;
            if (c >= Cn) continue;
            if constexpr (OUT_T) out[static_cast<size_t>(c) * ldo + r] = acc[i][j];
            else out[static_cast<size_t>(r) * ldo + c] = acc[i][j];
        }
    }
}

// ── few rows on one side, or too few tiles to fill the GPU ────────────────
// The larger of m and n ("rows") goes over the lanes, one fma chain each, the other side's QW values
// at a k come as scalar operands (scalar loads of X as it lies): 64 rows x QW NW columns per workgroup, so a
// product fills the GPU with waves where 256 x 64 tiles would leave most CUs idle.  K_MAJOR rows
// (element k of row r at k ld + r) are read as they lie, a 256-byte line per k, 16 k ahead.
// Others are staged by global_load_lds, E floats a lane (4 where rows are 16-byte aligned, else 1),
// 64 rows x 32 k in a ring of three stages; the E-float chunk j of row r sits in slot
// j ^ (r mod the chunks of a row), so neighbouring lanes reading the same k of their rows touch
// different banks.  The ring is read and waited for in one asm block, since the compiler does not
// track by stage the loads that fill it.
// Bound: the chains' and the scalar loads' latency in few waves, fp32 VALU issue in many.  One row
// by [10240 x 2560] 71 us (755 in tiles: 40 of them), 7 by [12000 x 2600] 116 (903), by [2600 x
// 12000] 119 (541), 16 by [1000 x 2000] 48 (575), 512 by [12000 x 2600] 836 us, 38 TFLOP/s (1317).
constexpr int kLaneNd = 3;

template <int E>
__device__ __forceinline__ void lane_ring16(uint32_t row, uint32_t swz, int h, float (&v)[16]) {
    if constexpr (E == 4) {
        floatx4_t q[4];
        const uint32_t a0 = row + ((16u * (4 * h)) ^ swz), a1 = row + ((16u * (4 * h + 1)) ^ swz),
                       a2 = row + ((16u * (4 * h + 2)) ^ swz), a3 = row + ((16u * (4 * h + 3)) ^ swz);
        asm volatile(
            "ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(q[0]), "=&v"(q[1]), "=&v"(q[2]), "=&v"(q[3])
            : "v"(a0), "v"(a1), "v"(a2), "v"(a3)
            : "memory");
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = q[i >> 2][i & 3];
    } else {
#pragma unroll
        for (int g = 0; g < 2; g++) {
            uint32_t a[8];
#pragma unroll
            for (int i = 0; i < 8; i++) a[i] = row + ((4u * (16 * h + 8 * g + i)) ^ swz);
            asm volatile(
                "ds_read_b32 %0, %8\n\tds_read_b32 %1, %9\n\tds_read_b32 %2, %10\n\tds_read_b32 %3, %11\n\t"
                "ds_read_b32 %4, %12\n\tds_read_b32 %5, %13\n\tds_read_b32 %6, %14\n\tds_read_b32 %7, %15\n\t"
                "s_waitcnt lgkmcnt(0)"
                : "=&v"(v[8 * g]), "=&v"(v[8 * g + 1]), "=&v"(v[8 * g + 2]), "=&v"(v[8 * g + 3]), "=&v"(v[8 * g + 4]),
                  "=&v"(v[8 * g + 5]), "=&v"(v[8 * g + 6]), "=&v"(v[8 * g + 7])
                : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7])
                : "memory");
        }
    }
}

// E floats per lane straight into LDS, at dst + E lane (dst wave-uniform).
template <int E>
__device__ __forceinline__ void load_lds(const float* src, float* dst) {
    const auto* g = (const __attribute__((address_space(1))) void*)src;
    auto* l = (__attribute__((address_space(3))) void*)dst;
    if constexpr (E == 4) __builtin_amdgcn_global_load_lds(g, l, 16, 0, 0);
    else __builtin_amdgcn_global_load_lds(g, l, 4, 0, 0);
}

template <int QW, int NW, bool K_MAJOR, bool X_KMAJOR, bool OUT_T, int E>
__global__ __launch_bounds__(64 * NW) void f32_lane_gemm_kernel(const float* __restrict__ G, size_t ld,
                                                                const float* __restrict__ X, size_t ldx,
                                                                float* __restrict__ out, size_t ldo, int R, int K, int Q) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // (waves past the last column repeat the last QW of the Q >= QW: the same values again)
    const int r0 = blockIdx.x * 64, q0 = min((static_cast<int>(blockIdx.y) * NW + wave) * QW, Q - QW);
    // column q0 + q at k: X k-minor, x[q ldx + k]; k-major, x[k ldx + q]
    const scalar_f32_ptr x = (scalar_f32_ptr)(reinterpret_cast<uintptr_t>(X) +
                                              sizeof(float) * (X_KMAJOR ? static_cast<size_t>(q0) : q0 * ldx));
    float acc[QW];
#pragma unroll
    for (int q = 0; q < QW; q++) acc[q] = 0.f;
    // 16 k (or n < 16) from k0 on, whose values of its row the lane holds
    auto full = [&](int k0, const float (&v)[16]) __attribute__((always_inline)) {
        if constexpr (X_KMAJOR) {
#pragma unroll
            for (int i = 0; i < 16; i++)
#pragma unroll
                for (int q = 0; q < QW; q++) acc[q] = fmaf(v[i], x[static_cast<size_t>(k0 + i) * ldx + q], acc[q]);
        } else {
            lane_fma16<QW>(acc, v, x, ldx, k0);
        }
    };
    auto part = [&](int k0, int n, const float (&v)[16]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 15; i++)
            if (i < n)
#pragma unroll
                for (int q = 0; q < QW; q++)
                    acc[q] = fmaf(v[i], X_KMAJOR ? x[static_cast<size_t>(k0 + i) * ldx + q] : x[q * ldx + k0 + i], acc[q]);
    };
    if constexpr (K_MAJOR) {
        const float* p = G + min(r0 + lane, R - 1);
        float v[16], w[16];
        auto load = [&](int k0, float (&o)[16]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 16; i++) o[i] = p[static_cast<size_t>(min(k0 + i, K - 1)) * ld];
        };
        load(0, v);
        int k0 = 0;
        for (; k0 + 32 <= K; k0 += 32) {
            load(k0 + 16, w);
            full(k0, v);
            load(k0 + 32, v);
            full(k0 + 16, w);
        }
        if (k0 + 16 <= K) {
            load(k0 + 16, w);
            full(k0, v);
            k0 += 16;
            part(k0, K - k0, w);
        } else {
            part(k0, K - k0, v);
        }
    } else {
        constexpr int kChunks = 32 / E, kRowsPer = 64 / kChunks;  // chunks of a staged row, rows of a load
        constexpr int kPer = kChunks / NW;                        // loads per wave and stage
        static_assert(kPer * NW == kChunks, "the waves split a stage's loads evenly");
        __shared__ __align__(128) float ring[kLaneNd][64 * 32];
        const float* gp[kPer];
        uint32_t kk[kPer];
#pragma unroll
        for (int i = 0; i < kPer; i++) {
            const int r = kRowsPer * (kPer * wave + i) + lane / kChunks;
            gp[i] = G + static_cast<size_t>(min(r0 + r, R - 1)) * ld;
            kk[i] = E * ((lane % kChunks) ^ (r % kChunks));
        }
        auto gload = [&](int st, int slot) __attribute__((always_inline)) {
            // (a chunk past the row re-reads its last one: staged, never used)
#pragma unroll
            for (int i = 0; i < kPer; i++)
                load_lds<E>(gp[i] + min(32 * st + static_cast<int>(kk[i]), K - E), &ring[slot][64 * E * (kPer * wave + i)]);
        };
        const uint32_t mine = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
                                  (__attribute__((address_space(3))) void*)&ring[0][0])) + 128u * lane;
        const uint32_t swz = 4u * E * (lane % kChunks);
        const int ns = (K + 31) / 32, last = ns - 1;
#pragma unroll
        for (int d = 0; d < kLaneNd - 1; d++) gload(min(d, last), d);
        int slot = 0;
        for (int st = 0; st < ns; st++) {
            // stage st has landed (this wave's loads, then everyone's), and every wave is past
            // stage st - 1, whose slot the next loads overwrite
            wait_vmcnt<kPer * (kLaneNd - 2)>();
            if constexpr (NW > 1) asm volatile("s_barrier" ::: "memory");
            gload(min(st + kLaneNd - 1, last), slot == 0 ? kLaneNd - 1 : slot - 1);
            const uint32_t row = mine + static_cast<uint32_t>(slot) * 8192u;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int k0 = 32 * st + 16 * h;
                float v[16];
                if (k0 >= K) break;
                lane_ring16<E>(row, swz, h, v);
                if (k0 + 16 <= K) full(k0, v);
                else part(k0, K - k0, v);
            }
            slot = slot + 1 == kLaneNd ? 0 : slot + 1;
        }
        wait_vmcnt<0>();  // nothing may land in LDS after the workgroup has ended
    }
    const int r = r0 + lane;
    if (r >= R) return;
#pragma unroll
    for (int q = 0; q < QW; q++) {
        if constexpr (OUT_T) out[static_cast<size_t>(r) * ldo + q0 + q] = acc[q];
        else out[static_cast<size_t>(q0 + q) * ldo + r] = acc[q];
    }
}

template <bool RK, bool CK, bool OT>
void launch_gemm(const float* R, size_t ldr, const float* Cm, size_t ldc, float* out, size_t ldo, size_t Rn,
                 size_t Cn, size_t K, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>((Cn + kGTileC - 1) / kGTileC),
                    static_cast<unsigned>((Rn + kGTileR - 1) / kGTileR));
    f32_gemm_kernel<RK, CK, OT><<<grid, dim3(kGThreads), 0, s>>>(R, ldr, Cm, ldc, out, ldo, static_cast<int>(Rn),
                                                                 static_cast<int>(Cn), static_cast<int>(K));
    LARQL_HIP_CHECK(hipGetLastError());
}

// Whether the lanes' form runs a product of `rows` x `q` (rows >= q) whose rows are k-minor or
// k-major.  The tiles take k-minor rows a float at a time per thread: lanes up to two tiles per
// CU (512 x [12000 x 2600], 376 tiles: 836 us in lanes, 1317 in tiles); k-major rows below three
// tiles for four CUs (100 x [2600 x 12000], 94 tiles: 353 us in lanes, 541 in tiles; 300 columns,
// 235 tiles: 609 and 540).
bool lane_form(size_t rows, size_t q, size_t k, bool k_major) {
    const size_t tiles = (rows + kGTileR - 1) / kGTileR * ((q + kGTileC - 1) / kGTileC);
    const size_t cus = static_cast<size_t>(current_device_cus());
    return k > 0 && (k_major ? 4 * tiles < 3 * cus : tiles < 2 * cus);
}

// Columns per wave (at most q) and waves per workgroup.
struct LanePlan {
    int qw, nw;
};
LanePlan lane_plan(size_t q) {
    if (q <= 2) return {static_cast<int>(q), 1};
    if (q <= 16) return {2, q <= 4 ? 2 : q <= 8 ? 4 : 8};
    if (q <= 32) return {4, 8};
    return {8, 8};
}
template <bool KM, bool XK, bool OT, int E>
void launch_lane(const float* G, size_t ld, const float* X, size_t ldx, float* out, size_t ldo, int R, int K, int Q, hipStream_t s) {
    const LanePlan p = lane_plan(static_cast<size_t>(Q));
    const unsigned gx = static_cast<unsigned>((R + 63) / 64);
    const size_t per = static_cast<size_t>(p.qw) * p.nw, blocks = (Q + per - 1) / per;
    auto go = [&](auto qw, auto nw) {
        constexpr int QW = decltype(qw)::value, NW = decltype(nw)::value;
        for (size_t y = 0; y < blocks; y += 65535) {  // (grid y is at most 65535)
            // (a last launch of fewer than QW columns starts earlier: the same values again)
            const size_t q0 = std::min(y * per, static_cast<size_t>(Q - QW));
            f32_lane_gemm_kernel<QW, NW, KM, XK, OT, E>
                <<<dim3(gx, static_cast<unsigned>(blocks - y < 65535 ? blocks - y : 65535)), dim3(64 * NW), 0, s>>>(
                    G, ld, X + (XK ? q0 : q0 * ldx), ldx, out + (OT ? q0 : q0 * ldo), ldo, R, K, Q - static_cast<int>(q0));
        }
    };
    using std::integral_constant;
    const integral_constant<int, 1> c1;
    const integral_constant<int, 2> c2;
    const integral_constant<int, 4> c4;
    const integral_constant<int, 8> c8;
    if (p.qw == 1) go(c1, c1);
    else if (p.qw == 2 && p.nw == 1) go(c2, c1);
    else if (p.qw == 2 && p.nw == 2) go(c2, c2);
    else if (p.qw == 2 && p.nw == 4) go(c2, c4);
    else if (p.qw == 2) go(c2, c8);
    else if (p.qw == 4) go(c4, c8);
    else go(c8, c8);
    LARQL_HIP_CHECK(hipGetLastError());
}

}  // namespace

void launch_f32_matmul(const float* A, const float* B, float* C, size_t m, size_t k, size_t n, bool transpose_b,
                       hipStream_t s) {
    if (m == 0 || n == 0) return;
    if (m > 0x7FFFFFFFu || n > 0x7FFFFFFFu || k > 0x7FFFFFFFu || (m + kGTileR - 1) / kGTileR > 65535 ||
        (n + kGTileR - 1) / kGTileR > 65535)
        fail(LARQL_HIP_ERR_INVALID, "matmul: dimensions too large");
    const bool swap = m > n;  // A's rows over the lanes
    const size_t rows = swap ? m : n, q = swap ? n : m;
    if (lane_form(rows, q, k, !swap && !transpose_b)) {
        const int R = static_cast<int>(rows), K = static_cast<int>(k), Q = static_cast<int>(q);
        const float* G = swap ? A : B;
        const bool al16 = k % 4 == 0 && reinterpret_cast<uintptr_t>(G) % 16 == 0;
        if (!swap && !transpose_b) launch_lane<true, false, false, 1>(B, n, A, k, C, n, R, K, Q, s);
        else if (!swap && al16) launch_lane<false, false, false, 4>(B, k, A, k, C, n, R, K, Q, s);
        else if (!swap) launch_lane<false, false, false, 1>(B, k, A, k, C, n, R, K, Q, s);
        else if (transpose_b && al16) launch_lane<false, false, true, 4>(A, k, B, k, C, n, R, K, Q, s);
        else if (transpose_b) launch_lane<false, false, true, 1>(A, k, B, k, C, n, R, K, Q, s);
        else if (al16) launch_lane<false, true, true, 4>(A, k, B, n, C, n, R, K, Q, s);
        else launch_lane<false, true, true, 1>(A, k, B, n, C, n, R, K, Q, s);
        return;
    }
    // A [m][k] is k-minor; B is [n][k] (k-minor, transpose_b) or [k][n] (k-major).  The
    // larger of m and n goes on the 256 side; C [m][n] is stored transposed when n is there.
    if (transpose_b) {
        if (m >= n) launch_gemm<false, false, false>(A, k, B, k, C, n, m, n, k, s);
        else launch_gemm<false, false, true>(B, k, A, k, C, n, n, m, k, s);
    } else {
        if (m >= n) launch_gemm<false, true, false>(A, k, B, n, C, n, m, n, k, s);
        else launch_gemm<true, false, true>(B, n, A, k, C, n, n, m, k, s);
    }
}

}  // namespace larql
