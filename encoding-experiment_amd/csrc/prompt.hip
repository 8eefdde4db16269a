// Row kernels of the batched prompt pass (prefill_q4, LC/src/backend.rs:139-152): the
// per-position operations of a Llama layer applied to all M positions of a prompt at
// once, around the Q4_K GEMMs (prefill.hip) and the prompt-mode attention (decode.hip).
// Each follows the decode step's arithmetic for one position:
//   * RMSNorm  (LI/src/residual.rs:17-33): rms = sqrt(sum(x^2) in f64 / n + eps) rounded
//     to f32, y = (x * (1 / rms)) * w — the fused-norm prologue of the matvecs;
//   * RoPE of K (LI/src/attention/rope.rs:22-55) with the cos/sin table, K and V rounded
//     to fp16 (RNE) into the cache rows of their positions;
//   * residual add (LI/src/forward/layer.rs:88-92) and act(gate) * up
//     (LI/src/ffn/mod.rs:87-103) over gate/up rows interleaved as the fused weight emits them;
//   * the layer variants of FullPipelineLayer (LC/src/pipeline.rs:76-115): norm weight
//     offset, the post-norm residual h + norm(v) (LI/src/attention/block.rs:139-150,
//     LI/src/forward/layer.rs:76-87), the parameter-free per-head V-norm
//     (LI/src/residual.rs:86-110) and the layer scalar.  These kernels also serve the
//     decode step (one row).
#include "decode.h"
#include "gemm_hp.h"
#include "matvec_common.h"

#include <type_traits>

namespace larql {

namespace {

// sum(x^2) of n floats in f64 by a 256-thread workgroup -> rms as the CPU path rounds it
// (LI/src/residual.rs:24).
__device__ __forceinline__ float row_rms(const float* __restrict__ x, int n, double eps, double* red) {
    double ss = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) ss += static_cast<double>(x[i]) * x[i];
    ss = wave_sum_d(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const double tot = (red[0] + red[1]) + (red[2] + red[3]);
    return static_cast<float>(sqrt(tot / static_cast<double>(n) + eps));
}

// Grid M rows; 256 threads.  y = (x * (1 / rms)) * (off + w), or without a weight
// (w == null) y = x * (1 / rms) (LI/src/residual.rs:25-29: weight None -> 1.0).
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const float* __restrict__ X, const float* __restrict__ w,
                                                           float off, float* __restrict__ Y, int n, double eps) {
    __shared__ double red[4];
    const float* x = X + static_cast<size_t>(blockIdx.x) * n;
    float* y = Y + static_cast<size_t>(blockIdx.x) * n;
    const float inv = 1.0f / row_rms(x, n, eps, red);
    if (w) {
        for (int i = threadIdx.x; i < n; i += 256) y[i] = (x[i] * inv) * (off + w[i]);
    } else {
        for (int i = threadIdx.x; i < n; i += 256) y[i] = x[i] * inv;
    }
}

// Post-norm residual, grid M rows: out = (h + norm(v, w)) * scale (scale 1 = none).
__global__ __launch_bounds__(256) void resid_norm_rows_kernel(const float* __restrict__ H, const float* __restrict__ V,
                                                              const float* __restrict__ w, float off, float scale,
                                                              float* __restrict__ OUT, int n, double eps) {
    __shared__ double red[4];
    const size_t r = static_cast<size_t>(blockIdx.x) * n;
    const float* v = V + r;
    const float inv = 1.0f / row_rms(v, n, eps, red);
    for (int i = threadIdx.x; i < n; i += 256) {
        const float nv = w ? (v[i] * inv) * (off + w[i]) : v[i] * inv;
        OUT[r + i] = (H[r + i] + nv) * scale;
    }
}

// Parameter-free RMS norm of each V head in place: grid (M rows, num_kv heads), one wave;
// head h of row p starts at X + p * ld + h * hd.
__global__ __launch_bounds__(64) void vnorm_rows_kernel(float* __restrict__ X, int ld, int hd, double eps) {
    float* v = X + static_cast<size_t>(blockIdx.x) * ld + static_cast<size_t>(blockIdx.y) * hd;
    double ss = 0.0;
    for (int i = threadIdx.x; i < hd; i += 64) ss += static_cast<double>(v[i]) * v[i];
    ss = wave_sum_d(ss);
    const float rms = static_cast<float>(sqrt(ss / static_cast<double>(hd) + eps));
    for (int i = threadIdx.x; i < hd; i += 64) v[i] = v[i] / rms;
}

// Thread per (position p, kv element j): K RoPE'd at p, K and V to fp16 in the cache.
__global__ void rope_kv_rows_kernel(const float* __restrict__ QKV, int M, int p0, int ld, int q_dim, int kv_dim,
                                    int hd, int half, const float2* __restrict__ rope, __half* __restrict__ kc,
                                    __half* __restrict__ vc, int num_kv) {
    const size_t t = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x;
    if (t >= static_cast<size_t>(M) * kv_dim) return;
    const int p = static_cast<int>(t / kv_dim), j = static_cast<int>(t - static_cast<size_t>(p) * kv_dim);
    const int kvh = j / hd, d = j - kvh * hd, pos = p0 + p;
    const float* row = QKV + static_cast<size_t>(p) * ld;
    const float* k = row + q_dim + kvh * hd;
    const float2* cs = rope + static_cast<size_t>(pos) * half;
    float kr = k[d];
    if (d < half) kr = rope_low(k[d], k[d + half], cs[d]);
    else if (d < 2 * half) kr = rope_high(k[d - half], k[d], cs[d - half]);
    kc[(static_cast<size_t>(pos) * num_kv + kvh) * hd + d] = __float2half_rn(kr);
    vc[((static_cast<size_t>(pos >> 3) * num_kv + kvh) * hd + d) * 8 + (pos & 7)] =
        __float2half_rn(row[q_dim + kv_dim + j]);
}

__global__ void add_rows_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ out,
                                size_t n, float scale) {
    const size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x;
    if (i < n) out[i] = (a[i] + b[i]) * scale;
}

// GU rows [M][2 inter] with gate and up interleaved (2i, 2i + 1) -> act [M][inter].
__global__ void gated_pair_rows_kernel(const float* __restrict__ GU, float* __restrict__ act, size_t n, int kind) {
    const size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x;
    if (i < n) act[i] = gated_act(kind, GU[2 * i], GU[2 * i + 1]);
}

// act[i] = act(G[i]) * U[i] (gate and up in separate buffers).
__global__ void gated_mul_kernel(const float* __restrict__ G, const float* __restrict__ U, float* __restrict__ act,
                                 size_t n, int kind) {
    const size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x;
    if (i < n) act[i] = gated_act(kind, G[i], U[i]);
}

// ── Fused row kernels of the prompt pass ─────────────────────────────────
// One workgroup per row; the row stays in LDS (kFusedRowMax floats at most) between the
// steps, and each thread's loads of a chunk are issued together (indices clamped into
// the row, so no load sits under a branch), so a row costs one round trip to memory per
// chunk and two workgroup barriers instead of a dependent load per element.

// Workgroup -> row, the 16 rows of a token tile on one XCD (workgroup i runs on XCD i % 8): the
// packed operands of a tile share 128-byte lines, which that XCD's L2 then fills whole.  Grids
// are whole groups of 128 rows.
__device__ __forceinline__ int tile_row() {
    const int j = static_cast<int>(blockIdx.x) >> 3;
    return ((j >> 4) * 8 + (static_cast<int>(blockIdx.x) & 7)) * 16 + (j & 15);
}

// The statistics of row r (n floats in LDS, written by all threads) into st: its exponent and,
// with st.xs, its scaled sub-block sums, the arithmetic of gemm_row_stats, whose maximum is
// order-free and whose sums run per sub-block in one thread; with st.xp the row packed.  m:
// this thread's max |x|; wm: one float per wave.
template <int NT>
__device__ __forceinline__ void lds_row_out(const float* row, int n, int r, float m, float* wm, const GemmRowStats& st) {
    const int t = threadIdx.x;
    m = wave_max(m);
    if ((t & 63) == 0) wm[t >> 6] = m;
    __syncthreads();
    m = wm[0];
#pragma unroll
    for (int k = 1; k < NT / 64; k++) m = fmaxf(m, wm[k]);
    const int ev = (m > 0.f && m <= 3.4e38f) ? min(120, max(-120, 14 - ilogbf(m))) : 0;
    if (t == 0) st.xe[r] = ev;
    if (st.xp) {
        const float sc = ldexpf(1.0f, ev);
        for (int e8 = t; e8 < n / 8; e8 += NT) hp_pack8(row + 8 * e8, sc, reinterpret_cast<v4u*>(st.xp) + hp_packed_at(r, e8, n));
    }
    if (!st.xs) return;
    float* xs = st.xs + static_cast<size_t>(r) * (n / 32);
    const double sc = ldexp(1.0, ev - 5);
    for (int j = t; j < n / 32; j += NT) {
        const float4* p = reinterpret_cast<const float4*>(row + 32 * j);
        double sum[2] = {0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float4 v = p[k];
            sum[k & 1] += (static_cast<double>(v.x) + static_cast<double>(v.y)) +
                          (static_cast<double>(v.z) + static_cast<double>(v.w));
        }
        xs[j] = static_cast<float>((sum[0] + sum[1]) * sc);
    }
}

// f64 sum of ss over the NT threads, wave by wave.
template <int NT>
__device__ __forceinline__ double block_sum_d(double ss, double* red) {
    ss = wave_sum_d(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    double tot = red[0];
#pragma unroll
    for (int k = 1; k < NT / 64; k++) tot += red[k];
    return tot;
}

// The step between two projections, per row of n floats, in the arithmetic of the separate
// kernels (f64 sums of squares in another order):
//   y = the projection row, its partial products summed in split order (sum_splits_kernel),
//       several splits' loads at a time;
//   POST: y = (y / rms(y)) * (poff + pw)                             (resid_norm_rows_kernel);
//   h = (hin + y) * scale, or hin itself without a projection        (add_rows_kernel);
//   x = norm ? (h * (1 / rms(h))) * (off + w) : h                    (rmsnorm_rows_kernel);
// h to hout (if given), x as its statistics and packed operands (if st.xe).
// NT threads: 256 where there are rows enough to fill the GPU, else 1024 (fewer elements per thread
// to wait for in turn: 9.3 -> 7.3 us per launch at 24 rows of 4096; 11.2 -> 13.0 at 512 rows).
template <int NT, bool POST>
__global__ __launch_bounds__(NT) void resid_norm_stats_rows_kernel(ResidRows a) {
    constexpr int kRowChunk = 4096 / NT, kZ = NT == 256 ? 4 : 8;  // elements per thread and chunk, splits' loads together
    __shared__ __align__(16) float row[kFusedRowMax];
    __shared__ double red[2][NT / 64];
    __shared__ float wm[NT / 64];
    const int t = threadIdx.x, ri = tile_row(), n = a.n;
    if (ri >= a.m) return;
    const size_t r = static_cast<size_t>(ri) * n;
    double ss = 0.0;
    float m = 0.f;
    float w0[kRowChunk];  // the norm weights of the first chunk, requested with its rows
    for (int c0 = 0; c0 < n; c0 += NT * kRowChunk) {
        float y[kRowChunk], h[kRowChunk];
#pragma unroll
        for (int q = 0; q < kRowChunk; q++) {
            const size_t i = r + min(c0 + t + NT * q, n - 1);
            y[q] = a.P ? a.P[i] : 0.f;
            h[q] = POST ? 0.f : a.hin[i];
        }
        if (c0 == 0) {
#pragma unroll
            for (int q = 0; q < kRowChunk; q++) w0[q] = a.w ? a.w[min(t + NT * q, n - 1)] : 0.f;
        }
        for (int z = 1; z < a.splits; z += kZ) {
            float v[kZ][kRowChunk];
#pragma unroll
            for (int k = 0; k < kZ; k++)
#pragma unroll
                for (int q = 0; q < kRowChunk; q++)
                    v[k][q] = a.P[min(z + k, a.splits - 1) * a.pstride + r + min(c0 + t + NT * q, n - 1)];
#pragma unroll
            for (int k = 0; k < kZ; k++)
                if (z + k < a.splits)
#pragma unroll
                    for (int q = 0; q < kRowChunk; q++) y[q] += v[k][q];
        }
#pragma unroll
        for (int q = 0; q < kRowChunk; q++) {
            const int i = c0 + t + NT * q;
            if (i < n) {
                const float hv = POST ? y[q] : (a.P ? (h[q] + y[q]) * a.scale : h[q]);
                if (!POST && a.hout) a.hout[r + i] = hv;
                row[i] = hv;
                ss += static_cast<double>(hv) * hv;
                m = fmaxf(m, fabsf(hv));
            }
        }
    }
    if constexpr (POST) {  // (a thread's own elements of `row` throughout)
        const double tot = block_sum_d<NT>(ss, red[0]);
        const float inv = 1.0f / static_cast<float>(sqrt(tot / static_cast<double>(n) + a.eps));
        ss = 0.0, m = 0.f;
        for (int c0 = 0; c0 < n; c0 += NT * kRowChunk) {
            float h[kRowChunk], wv[kRowChunk];
#pragma unroll
            for (int q = 0; q < kRowChunk; q++) {
                const int i = min(c0 + t + NT * q, n - 1);
                h[q] = a.hin[r + i];
                wv[q] = a.pw ? a.pw[i] : 0.f;
            }
#pragma unroll
            for (int q = 0; q < kRowChunk; q++) {
                const int i = c0 + t + NT * q;
                if (i < n) {
                    const float nv = a.pw ? (row[i] * inv) * (a.poff + wv[q]) : row[i] * inv;
                    const float hv = (h[q] + nv) * a.scale;
                    if (a.hout) a.hout[r + i] = hv;
                    row[i] = hv;
                    ss += static_cast<double>(hv) * hv;
                    m = fmaxf(m, fabsf(hv));
                }
            }
        }
    }
    if (!a.norm && !a.st.xe) return;  // (uniform)
    if (a.norm) {
        const double tot = block_sum_d<NT>(ss, red[1]);
        const float inv = 1.0f / static_cast<float>(sqrt(tot / static_cast<double>(n) + a.norm_eps));
        m = 0.f;
        for (int c0 = 0; c0 < n; c0 += NT * kRowChunk) {
            float wv[kRowChunk];
#pragma unroll
            for (int q = 0; q < kRowChunk; q++) wv[q] = c0 == 0 ? w0[q] : (a.w ? a.w[min(c0 + t + NT * q, n - 1)] : 0.f);
#pragma unroll
            for (int q = 0; q < kRowChunk; q++) {
                const int i = c0 + t + NT * q;
                if (i < n) {  // (the thread's own elements of `row`: no barrier needed)
                    const float x = a.w ? (row[i] * inv) * (a.off + wv[q]) : row[i] * inv;
                    row[i] = x;
                    m = fmaxf(m, fabsf(x));
                }
            }
        }
    }
    if (a.st.xe) lds_row_out<NT>(row, n, ri, m, wm, a.st);
}

// act(gate) * up over a row of n outputs (1024 threads) from gate/up rows with the pairs interleaved
// (as gated_pair_rows_kernel; K-split partial products summed in split order): its statistics and
// packed operands for the down projection.
__global__ __launch_bounds__(1024) void gated_stats_rows_kernel(const float* __restrict__ G, size_t pstride, int splits,
                                                                int M, int n, int kind, GemmRowStats st) {
    constexpr int kChunk = 8;
    __shared__ __align__(16) float row[kFusedRowMax];
    __shared__ float wm[16];
    const int t = threadIdx.x, ri = tile_row();
    if (ri >= M) return;
    const size_t r = static_cast<size_t>(ri) * n;
    float m = 0.f;
    for (int c0 = 0; c0 < n; c0 += 1024 * kChunk) {
        float2 v[kChunk];
#pragma unroll
        for (int q = 0; q < kChunk; q++) v[q] = reinterpret_cast<const float2*>(G)[r + min(c0 + t + 1024 * q, n - 1)];
        for (int z = 1; z < splits; z += 2) {
            float2 p[2][kChunk];
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int q = 0; q < kChunk; q++)
                    p[k][q] = reinterpret_cast<const float2*>(G + min(z + k, splits - 1) * pstride)[r + min(c0 + t + 1024 * q, n - 1)];
#pragma unroll
            for (int k = 0; k < 2; k++)
                if (z + k < splits)
#pragma unroll
                    for (int q = 0; q < kChunk; q++) v[q].x += p[k][q].x, v[q].y += p[k][q].y;
        }
#pragma unroll
        for (int q = 0; q < kChunk; q++) {
            const int i = c0 + t + 1024 * q;
            if (i < n) {
                const float x = gated_act(kind, v[q].x, v[q].y);
                row[i] = x;
                m = fmaxf(m, fabsf(x));
            }
        }
    }
    lds_row_out<1024>(row, n, ri, m, wm, st);
}

unsigned blocks(size_t n) { return static_cast<unsigned>((n + 255) / 256); }

}  // namespace

void launch_rmsnorm_rows(const float* X, const float* w, float off, float* Y, size_t m, size_t n, double eps,
                         hipStream_t s) {
    if (m == 0) return;
    rmsnorm_rows_kernel<<<dim3(static_cast<unsigned>(m)), dim3(256), 0, s>>>(X, w, off, Y, static_cast<int>(n), eps);
    LARQL_HIP_CHECK(hipGetLastError());
}

void launch_resid_norm_rows(const float* H, const float* V, const float* w, float off, float scale, float* out,
                            size_t m, size_t n, double eps, hipStream_t s) {
    if (m == 0) return;
    resid_norm_rows_kernel<<<dim3(static_cast<unsigned>(m)), dim3(256), 0, s>>>(H, V, w, off, scale, out,
                                                                                static_cast<int>(n), eps);
    LARQL_HIP_CHECK(hipGetLastError());
}

void launch_vnorm_rows(float* X, size_t m, size_t ld, int num_heads, int hd, double eps, hipStream_t s) {
    if (m == 0 || num_heads == 0) return;
    vnorm_rows_kernel<<<dim3(static_cast<unsigned>(m), static_cast<unsigned>(num_heads)), dim3(64), 0, s>>>(
        X, static_cast<int>(ld), hd, eps);
    LARQL_HIP_CHECK(hipGetLastError());
}

void launch_rope_kv_rows(const float* QKV, size_t m, size_t p0, size_t q_dim, size_t kv_dim, int hd, int rdim,
                         const float2* rope, __half* kc, __half* vc, int num_kv, hipStream_t s) {
    const size_t n = m * kv_dim;
    if (n == 0) return;
    rope_kv_rows_kernel<<<dim3(blocks(n)), dim3(256), 0, s>>>(
        QKV, static_cast<int>(m), static_cast<int>(p0), static_cast<int>(q_dim + 2 * kv_dim), static_cast<int>(q_dim),
        static_cast<int>(kv_dim), hd, rdim / 2, rope, kc, vc, num_kv);
    LARQL_HIP_CHECK(hipGetLastError());
}

void launch_add_rows(const float* a, const float* b, float* out, size_t n, hipStream_t s, float scale) {
    if (n == 0) return;
    add_rows_kernel<<<dim3(blocks(n)), dim3(256), 0, s>>>(a, b, out, n, scale);
    LARQL_HIP_CHECK(hipGetLastError());
}

void launch_gated_mul(const float* G, const float* U, float* act, size_t n, int kind, hipStream_t s) {
    if (n == 0) return;
    gated_mul_kernel<<<dim3(blocks(n)), dim3(256), 0, s>>>(G, U, act, n, kind);
    LARQL_HIP_CHECK(hipGetLastError());
}

static dim3 tile_rows_grid(size_t m) { return dim3(static_cast<unsigned>((m + 127) / 128 * 128)); }

void launch_resid_norm_stats_rows(const ResidRows& a, hipStream_t s) {
    if (a.m == 0) return;
    if (a.m > 0x7FFFFF00 || a.splits < 1 || a.n % 32 != 0 || a.n > kFusedRowMax || !a.hin || (a.post && !a.P) ||
        (a.st.xp && !a.st.xe))
        fail(LARQL_HIP_ERR_INVALID, "fused residual and norm rows: bad arguments");
    auto go = [&](auto nt) {
        constexpr int NT = decltype(nt)::value;
        if (a.post) resid_norm_stats_rows_kernel<NT, true><<<tile_rows_grid(a.m), dim3(NT), 0, s>>>(a);
        else resid_norm_stats_rows_kernel<NT, false><<<tile_rows_grid(a.m), dim3(NT), 0, s>>>(a);
    };
    if (a.m >= current_device_cus()) go(std::integral_constant<int, 256>{});
    else go(std::integral_constant<int, 1024>{});
    LARQL_HIP_CHECK(hipGetLastError());
}

void launch_gated_stats_rows(const float* G, size_t pstride, int splits, size_t m, size_t n, int kind,
                             const GemmRowStats& st, hipStream_t s) {
    if (m == 0) return;
    if (m > 0x7FFFFF00 || splits < 1 || n % 32 != 0 || n > static_cast<size_t>(kFusedRowMax) || !st.xe)
        fail(LARQL_HIP_ERR_INVALID, "fused gated rows: bad arguments");
    gated_stats_rows_kernel<<<tile_rows_grid(m), dim3(1024), 0, s>>>(G, pstride, splits, static_cast<int>(m),
                                                                     static_cast<int>(n), kind, st);
    LARQL_HIP_CHECK(hipGetLastError());
}

void launch_gated_pair_rows(const float* GU, float* act, size_t n, int kind, hipStream_t s) {
    if (n == 0) return;
    gated_pair_rows_kernel<<<dim3(blocks(n)), dim3(256), 0, s>>>(GU, act, n, kind);
    LARQL_HIP_CHECK(hipGetLastError());
}

}  // namespace larql
