// Q4_0 x Q8 and Q8_0 x Q8 products for many activation rows (the prompt pass of Q8_0 / Q4_0
// layers, the walk FFN's pair batch beyond 8 positions): out[t][n] = sum over the 32-element
// blocks b, in order, of (float)isum_b * (s_w * s_x), isum_b an exact int32 dot (the order of
// LC/csrc/q4_dot.c:58-89 and LC/src/cpu/ops/q8_matvec.rs:44-57; product and sum rounded
// separately), bit for bit what the matvec kernels give row by row.
//
// v_mfma_i32_16x16x32_i8 takes one block of 16 tokens x 16 weight rows: D lane (g, c) holds the
// dots of tokens 4 g .. 4 g + 3 and weight row c, whose four chains the lane continues.  A
// workgroup is 16 TT tokens x 64 R weight rows, wave w owning R tiles; the tokens' codes (in the
// order the weight unpack gives) and scales are staged in LDS, four blocks per stage, the next
// stage's loads in registers meanwhile.
// Bound: the reference's four operations per (row, token, block) (conversion, two products, sum) in
// few waves (two [14336 x 4096] at 96 rows: 34,800 VALU operations per SIMD in 196,000 cycles, 1.3
// waves per SIMD, 11% MFMA): Q4_0 [14336 x 4096] 29 us at 32 tokens, 65 at 128 (230 TOP/s), against 53 and
// 204 us in passes of eight tokens that each stream the weights; the two matrices of a walk FFN
// layer at 96 tokens 82 us.
#include <type_traits>

#include "device_common.h"
#include "larql_hip_internal.h"

#pragma clang fp contract(off)

namespace larql {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kIgWaves = 4, kIgThreads = 64 * kIgWaves;

// Bytes of the codes minus 8 (signed), without borrows between bytes.
__device__ __forceinline__ uint32_t nib_s8(uint32_t w4) { return ((w4 | 0x80808080u) - 0x08080808u) ^ 0x80808080u; }

__device__ __forceinline__ long pack64(uint32_t lo, uint32_t hi) {
    return static_cast<long>((static_cast<uint64_t>(hi) << 32) | lo);
}

struct IgArgs {
    const void* qs[kIntGemmMats];  // weights of one shape and their scales
    const void* sc[kIntGemmMats];
    float* out;                    // of the first weight; the others' ostep floats apart
    ptrdiff_t ostep;
    const int8_t* X8;  // [M][K] codes
    const float* XS;   // [M][K / 32] scales
    int M, N, nb, ntiles, ldo, gx, gy, gz;
};

// Q4_0: lane (g, c) loads block 4 u + g of row c (row-major nibbles), and a 4 x 4 transpose
// across the lane groups gives it dword g (elements 8 g ..) of each of the four blocks: even
// elements in the low nibbles, odd in the high.  Q8_0: lane (g, c) loads piece g of row c of a
// block pair (16 bytes: block g / 2, half g % 2); swapping two dwords between the wave's halves
// gives it eight bytes of each block, 16 (g & 1) + 8 (g >> 1) on.
template <int FMT, int TT, int R>
__global__ __launch_bounds__(kIgThreads) void int_gemm_kernel(IgArgs a) {
    constexpr bool kQ40 = FMT == LARQL_Q4_0;
    __shared__ __align__(16) v2u As[2][TT][2][64][2];  // [tile][block pair][lane][block of the pair]
    __shared__ __align__(16) float Xs[2][4][16 * TT];  // token scales of the four blocks
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int M = a.M, N = a.N, nb = a.nb, K = 32 * nb;
    // the gy token blocks of one (weight block, matrix) on one XCD back to back (as the
    // f32-accuracy GEMM's grid)
    const int L = static_cast<int>(blockIdx.x), slot = L >> 3, by = slot % a.gy;
    const int grp = (slot / a.gy) * 8 + (L & 7);
    if (grp >= a.gx * a.gz) return;
    const int bx = grp % a.gx, bz = grp / a.gx;
    const int t0 = by * 16 * TT, nt0 = (bx * kIgWaves + wave) * R;
    const uint8_t* qs = static_cast<const uint8_t*>(a.qs[bz]);
    float* out = a.out + bz * a.ostep;

    // raw buffer loads (the launcher keeps the weights below 2 GiB): lane part + uniform part
    const uint32_t qbytes = static_cast<uint32_t>(a.ntiles) * 16u * (kQ40 ? static_cast<uint32_t>(K / 2) : static_cast<uint32_t>(K));
    const uint32_t sbytes = static_cast<uint32_t>(a.ntiles) * 16u * static_cast<uint32_t>(nb) * (kQ40 ? 2u : 4u);
    const __amdgpu_buffer_rsrc_t rq =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(qs), 0, static_cast<int>(qbytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.sc[bz]), 0, static_cast<int>(sbytes), 0x00020000);
    uint32_t qo[R], so[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
        const uint32_t t = static_cast<uint32_t>(min(nt0 + j, a.ntiles - 1));
        qo[j] = __builtin_amdgcn_readfirstlane(t * 16u * (kQ40 ? K / 2 : K));
        so[j] = __builtin_amdgcn_readfirstlane(t * 16u * nb * (kQ40 ? 2u : 4u));
    }
    const uint32_t ql = kQ40 ? static_cast<uint32_t>(c) * (K / 2) + 16u * g : lane * 16u;
    const uint32_t sl = kQ40 ? static_cast<uint32_t>(c) * (2u * nb) : c * 8u;
    struct Wu {
        v4u q[R][kQ40 ? 1 : 2];
        v2u s[R][kQ40 ? 1 : 2];  // Q4_0: four f16 scales; Q8_0: f32 scale pairs
    };
    auto load_w = [&](int u, Wu& w) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < R; j++) {
            if constexpr (kQ40) {
                w.q[j][0] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rq, ql, qo[j] + u * 64u, 0));
                w.s[j][0] = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(rs, sl, so[j] + u * 8u, 0));
            } else {
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    w.q[j][p] = __builtin_bit_cast(
                        v4u, __builtin_amdgcn_raw_buffer_load_b128(rq, ql, qo[j] + (2 * u + p) * 1024u, 0));
                    w.s[j][p] = __builtin_bit_cast(
                        v2u, __builtin_amdgcn_raw_buffer_load_b64(rs, sl, so[j] + (2 * u + p) * 128u, 0));
                }
            }
        }
    };
    // staging: thread = token tid % 64 (clamped into the tile and the batch; tokens past M give
    // rows that are not stored), block tid / 64 of the stage
    const int st = min(lane, 16 * TT - 1), sb = wave, sm = min(t0 + st, M - 1);
    const int8_t* xp = a.X8 + static_cast<size_t>(sm) * K + 32 * sb;
    const float* xsp = a.XS + static_cast<size_t>(sm) * nb + sb;
    struct Xu {
        v4u v[2];
        float s;
    };
    auto load_x = [&](int u, Xu& x) __attribute__((always_inline)) {
        const v4u* p = reinterpret_cast<const v4u*>(xp + 128 * static_cast<size_t>(u));
        x.v[0] = p[0];
        x.v[1] = p[1];
        x.s = xsp[4 * u];
    };
    auto store_x = [&](int b, const Xu& x) __attribute__((always_inline)) {
        if (lane >= 16 * TT) return;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            v2u o;
            if constexpr (kQ40) {
                const uint32_t d0 = x.v[q >> 1][2 * (q & 1)], d1 = x.v[q >> 1][2 * (q & 1) + 1];
                o.x = __builtin_amdgcn_perm(d1, d0, 0x06040200u);
                o.y = __builtin_amdgcn_perm(d1, d0, 0x07050301u);
            } else {
                o.x = x.v[q & 1][2 * (q >> 1)];
                o.y = x.v[q & 1][2 * (q >> 1) + 1];
            }
            As[b][st >> 4][sb >> 1][16 * q + (st & 15)][sb & 1] = o;
        }
        Xs[b][sb][st] = x.s;
    };
    floatx4 acc[R][TT];
#pragma unroll
    for (int j = 0; j < R; j++)
#pragma unroll
        for (int i = 0; i < TT; i++) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};

    auto compute = [&](int b, const Wu& w) __attribute__((always_inline)) {
        uint32_t n[R][4];
        if constexpr (kQ40) {
#pragma unroll
            for (int j = 0; j < R; j++) {
                const v4u q = w.q[j][0];
                const auto a02 = __builtin_amdgcn_permlane32_swap(q.x, q.z, false, false);
                const auto a13 = __builtin_amdgcn_permlane32_swap(q.y, q.w, false, false);
                const auto r01 = __builtin_amdgcn_permlane16_swap(a02[0], a13[0], false, false);
                const auto r23 = __builtin_amdgcn_permlane16_swap(a02[1], a13[1], false, false);
                n[j][0] = r01[0], n[j][1] = r01[1], n[j][2] = r23[0], n[j][3] = r23[1];
            }
        }
#pragma unroll
        for (int p = 0; p < 2; p++) {
            v4u av[TT];
#pragma unroll
            for (int i = 0; i < TT; i++) av[i] = *reinterpret_cast<const v4u*>(&As[b][i][p][lane][0]);
            long B[R][2];
            float ws[R][2];
#pragma unroll
            for (int j = 0; j < R; j++) {
                if constexpr (kQ40) {
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const uint32_t wd = n[j][2 * p + e];
                        B[j][e] = pack64(nib_s8(wd & 0x0F0F0F0Fu), nib_s8((wd >> 4) & 0x0F0F0F0Fu));
                        ws[j][e] = h2f(w.s[j][0][p] >> (16 * e));
                    }
                } else {
                    const v4u q = w.q[j][p];
                    const auto xz = __builtin_amdgcn_permlane32_swap(q.x, q.z, false, false);
                    const auto yw = __builtin_amdgcn_permlane32_swap(q.y, q.w, false, false);
                    B[j][0] = pack64(xz[0], yw[0]);
                    B[j][1] = pack64(xz[1], yw[1]);
                    ws[j][0] = __uint_as_float(w.s[j][p].x);
                    ws[j][1] = __uint_as_float(w.s[j][p].y);
                }
            }
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int i = 0; i < TT; i++) {
                    const floatx4 xs = *reinterpret_cast<const floatx4*>(&Xs[b][2 * p + e][16 * i + 4 * g]);
                    const long A = e ? pack64(av[i].z, av[i].w) : pack64(av[i].x, av[i].y);
#pragma unroll
                    for (int j = 0; j < R; j++) {
                        const v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(A, B[j][e], v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const float cs = ws[j][e] * xs[r];
                            const float pr = static_cast<float>(d[r]) * cs;
                            acc[j][i][r] = acc[j][i][r] + pr;
                        }
                    }
                }
        }
    };

    // stage u in LDS slot u % 2, the loads of the D stages after it in registers
    constexpr int D = TT * R <= 3 ? 4 : 2;
    const int ns = nb / 4, last = ns - 1;
    Wu w[D];
    Xu x[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        load_x(min(d, last), x[d]);
        load_w(min(d, last), w[d]);
    }
    store_x(0, x[0]);
    load_x(min(D, last), x[0]);
    lds_barrier();
    for (int u = 0; u < ns; u += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (u + d >= ns) break;
            store_x((d + 1) & 1, x[(d + 1) % D]);
            load_x(min(u + d + 1 + D, last), x[(d + 1) % D]);
            compute(d & 1, w[d]);
            load_w(min(u + d + D, last), w[d]);
            lds_barrier();
        }
    }
#pragma unroll
    for (int i = 0; i < TT; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int t = t0 + 16 * i + 4 * g + r;
            float* y = out + static_cast<size_t>(t) * a.ldo + nt0 * 16 + c;
#pragma unroll
            for (int j = 0; j < R; j++)
                if (t < M && (nt0 + j) * 16 + c < N) y[16 * j] = acc[j][i][r];
        }
}

template <int FMT, int TT>
void launch_tt(const IgArgs& a, int R, unsigned grid, hipStream_t s) {
    if (R == 1) int_gemm_kernel<FMT, TT, 1><<<dim3(grid), dim3(kIgThreads), 0, s>>>(a);
    else int_gemm_kernel<FMT, TT, 2><<<dim3(grid), dim3(kIgThreads), 0, s>>>(a);
}

template <int FMT>
void launch_fmt(const IgArgs& a, int TT, int R, unsigned grid, hipStream_t s) {
    if (TT == 1) launch_tt<FMT, 1>(a, R, grid, s);
    else if (TT == 2) launch_tt<FMT, 2>(a, R, grid, s);
    else if (TT == 3) launch_tt<FMT, 3>(a, R, grid, s);
    else launch_tt<FMT, 4>(a, R, grid, s);
}

}  // namespace

bool int_gemm_takes(const DevWeight& w) {
    return (w.format == LARQL_Q4_0 || w.format == LARQL_Q8_0) && w.cols % 128 == 0 && w.rows_pad % 64 == 0 &&
           w.rows_pad * w.cols <= 0x7FFFFFFF;
}

namespace {
// Token tiles and weight tiles per wave: the least modelled time, rounds of workgroups over
// the CUs times a workgroup's VALU operations per block (16 per 16 x 16 tile, ~12 to unpack a
// weight tile, ~30 of loop, staging and waits)
struct IgPlan {
    int TT, R;
    long rounds;
};
IgPlan ig_plan(long ntiles, size_t m, int mats) {
    const long cus = current_device_cus(), mt = (static_cast<long>(m) + 15) / 16;
    IgPlan p{1, 1, 1};
    double best = -1;
    for (int r = 1; r <= 2; r++)
        for (int t = 1; t <= 4; t++) {
            const long wgs = (ntiles + 4L * r - 1) / (4L * r) * ((mt + t - 1) / t) * mats;
            const double cost = static_cast<double>((wgs + cus - 1) / cus) * (r * (16.0 * t + 12.0) + 30.0);
            if (best < 0 || cost < best) best = cost, p = {t, r, (wgs + cus - 1) / cus};
        }
    return p;
}

void launch_ig(IgArgs& a, int fmt, hipStream_t s) {
    const auto [TT, R, rounds] = ig_plan(a.ntiles, static_cast<size_t>(a.M), a.gz);
    a.gx = (a.ntiles + 4 * R - 1) / (4 * R);
    a.gy = ((a.M + 15) / 16 + TT - 1) / TT;
    const unsigned grid = static_cast<unsigned>((static_cast<long>(a.gx) * a.gz + 7) / 8 * 8 * a.gy);
    if (fmt == LARQL_Q4_0) launch_fmt<LARQL_Q4_0>(a, TT, R, grid, s);
    else launch_fmt<LARQL_Q8_0>(a, TT, R, grid, s);
    LARQL_HIP_CHECK(hipGetLastError());
}
}  // namespace

// Measured, rows 2048 .. 20000 (one matrix or two), 9 .. 33 activation rows: a line in the workgroup's
// tiles per block and round.
double int_gemm_us(const DevWeight& w, size_t m, int mats) {
    const IgPlan p = ig_plan(static_cast<long>(w.rows_pad / 16), m, mats);
    return 3.4 + static_cast<double>(w.cols / 32) * static_cast<double>(p.rounds) * (p.R * (16 * p.TT + 12) + 12.5) * 0.0031;
}

void launch_int_gemm(const DevWeight& w, const DevWeight* w2, const int8_t* q8x, const float* q8s, float* out,
                     float* out2, size_t m, size_t ldo, hipStream_t s) {
    if (m == 0) return;
    if (ldo == 0) ldo = w.rows;
    if (!int_gemm_takes(w) || (w2 && (w2->format != w.format || w2->rows != w.rows || w2->cols != w.cols)))
        fail(LARQL_HIP_ERR_INVALID, "int GEMM: Q4_0 or Q8_0 weights of one shape, cols a multiple of 128");
    if (ldo < w.rows || ldo > 0x7FFFFFFF || m > 0x7FFFFFFF / w.cols) fail(LARQL_HIP_ERR_INVALID, "int GEMM: bad sizes");
    IgArgs a{};
    a.qs[0] = w.qs;
    a.sc[0] = w.d;
    a.out = out;
    if (w2) {
        a.qs[1] = w2->qs;
        a.sc[1] = w2->d;
        a.ostep = out2 - out;
    }
    a.X8 = q8x;
    a.XS = q8s;
    a.M = static_cast<int>(m);
    a.N = static_cast<int>(w.rows);
    a.nb = static_cast<int>(w.cols / 32);
    a.ntiles = static_cast<int>(w.rows_pad / 16);
    a.ldo = static_cast<int>(ldo);
    a.gz = w2 ? 2 : 1;
    launch_ig(a, w.format, s);
}

void launch_int_gemm_q4_layers(const void* const* nib, const void* const* scales, int layers, const int8_t* X8,
                               const float* XS, float* S, int F, int K, int Q, hipStream_t s) {
    if (layers < 1 || layers > kIntGemmMats || K % 128) fail(LARQL_HIP_ERR_INVALID, "int GEMM: bad layers");
    IgArgs a{};
    for (int l = 0; l < layers; l++) a.qs[l] = nib[l], a.sc[l] = scales[l];
    a.out = S;
    a.ostep = static_cast<ptrdiff_t>(Q) * F;
    a.X8 = X8;
    a.XS = XS;
    a.M = Q;
    a.N = F;
    a.nb = K / 32;
    a.ntiles = static_cast<int>(pad_rows(static_cast<size_t>(F)) / 16);
    a.ldo = F;
    a.gz = layers;
    launch_ig(a, LARQL_Q4_0, s);
}

}  // namespace larql
