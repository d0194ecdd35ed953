// Kernels of the denoising step around the blocks (the transformer's outer
// forward and the sampler), all in f32:
//   linear_f32: the bias-free global linears (img_in, the timestep embedder,
//     modulation.1, norm_out.linear, proj_out, txt_in) over f32 weights,
//     src/quantized_transformer.rs:14-33, 43-54, 56-81, 213-228, 288-310;
//   rows_rmsnorm: txt_in's ZeroCenterRMSNorm (weight + 1 applied at upload);
//   rows_ln_scale: norm_out = LayerNorm(x) * (1 + scale) (:300-309);
//   euler: FlowMatchEuler::step (src/scheduler.rs:54-66);
//   cfg: neg + scale * (cond - neg) (src/pipeline.rs:180-186).
// Weights are dequantized to f32 once at upload and accumulation is f32, as the
// reference's F32 matmuls. A forward reads about 0.4 GB of them (modulation.1
// alone is 4 hidden x hidden), so the linears are split by their row count:
//   up to ROWS_MAX rows (one timestep per batch entry): one wave per output
//     column streams its weight row (linear_rows_kernel);
//   more rows (img_in, proj_out, txt_in): f32 matrix instructions over tiles
//     whose k range the workgroup's waves share (linear_mfma_kernel);
//   widths or addresses that do not allow 16 B loads: linear_any_kernel.
#include <algorithm>

#include "device_common.h"
#include "kernels.h"

namespace qimm {
namespace {

constexpr int LT = 64;  // output tile (rows x columns) per workgroup
constexpr int LK = 32;  // k chunk staged through LDS
constexpr int LP = LT + 4;

__device__ __forceinline__ float act(float v, int a) {
    if (a == ACT_SILU) return v / (1.0f + expf(-v));
    if (a == ACT_GELU_TANH) {
        const float c = 0.7978845608028654f;  // sqrt(2 / pi)
        return 0.5f * v * (1.0f + tanhf(c * (v + 0.044715f * v * v * v)));
    }
    return v;
}

// y[m, n] = act(sum_k x[m, k] * w[n, k]) for any sizes. 256 threads, each a
// 4 x 4 block of the 64 x 64 tile; x and w chunks are stored k-major in LDS so
// the inner loop reads 4 consecutive rows / columns per thread.
__global__ __launch_bounds__(256) void linear_any_kernel(const float *__restrict__ x, int64_t ldx,
                                                         const float *__restrict__ w, int64_t M, int64_t N,
                                                         int64_t K, int a, float *__restrict__ y, int64_t ldy) {
    __shared__ float xs[LK][LP];
    __shared__ float ws[LK][LP];
    const int t = threadIdx.x, tx = t & 15, ty = t >> 4;
    const int64_t m0 = (int64_t)blockIdx.y * LT, n0 = (int64_t)blockIdx.x * LT;
    float acc[4][4] = {};
    for (int64_t k0 = 0; k0 < K; k0 += LK) {
        // 64 rows x 32 k of each operand: 8 values per thread, k fastest
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int idx = t + 256 * e, r = idx >> 5, kk = idx & 31;
            const int64_t k = k0 + kk;
            const int64_t m = m0 + r, n = n0 + r;
            xs[kk][r] = (m < M && k < K) ? x[m * ldx + k] : 0.f;
            ws[kk][r] = (n < N && k < K) ? w[n * K + k] : 0.f;
        }
        __syncthreads();
#pragma unroll 8
        for (int kk = 0; kk < LK; kk++) {
            const float4 av = *(const float4 *)&xs[kk][4 * ty];
            const float4 bv = *(const float4 *)&ws[kk][4 * tx];
            const float ar[4] = {av.x, av.y, av.z, av.w}, br[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = fmaf(ar[i], br[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t m = m0 + 4 * ty + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t n = n0 + 4 * tx + j;
            if (n < N) y[m * ldy + n] = act(acc[i][j], a);
        }
    }
}

// A few rows (K % 4 == 0): bound by the weight bytes. Wave v of workgroup b
// owns output column 8 b + v: its lanes read the weight row 16 B each, up to
// RU loads in flight per lane before their products, against MB rows of x kept
// in LDS (chunks of RK k); blockIdx.y takes the next MB rows (their weights
// come from the MALL). Measured at K = 4096, one row: 16384 columns 52 us (5.1
// TB/s, a large copy's rate), 4096 columns 17 us; the 64 x 64 tile kernel
// above took 770 us for either (128 dependent k chunks in 64-256 workgroups).
constexpr int ROWS_MAX = 8;  // rows taken by this kernel
constexpr int RK = 4096;     // k per LDS chunk
constexpr int RU = 8;        // 16 B weight loads in flight per lane
template <int MB>
__global__ __launch_bounds__(512) void linear_rows_kernel(const float *__restrict__ x, int64_t ldx,
                                                          const float *__restrict__ w, int64_t M, int64_t N,
                                                          int64_t K, int a, float *__restrict__ y, int64_t ldy) {
    __shared__ __attribute__((aligned(16))) float xs[MB * RK];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t m0 = (int64_t)blockIdx.y * MB, n = (int64_t)blockIdx.x * 8 + wave;
    const float *wr = w + min(n, N - 1) * K;
    float acc[MB] = {};
    for (int64_t k0 = 0; k0 < K; k0 += RK) {
        const int kc = (int)min((int64_t)RK, K - k0);  // a multiple of 4
        if (k0) __syncthreads();
        for (int mb = 0; mb < MB; mb++) {
            const float *xr = x + min(m0 + mb, M - 1) * ldx + k0;
            for (int i = threadIdx.x; i < kc; i += 512) xs[mb * RK + i] = xr[i];
        }
        __syncthreads();
        for (int c0 = 4 * lane; c0 < kc; c0 += 256 * RU) {
            f32x4 wv[RU];
#pragma unroll
            for (int u = 0; u < RU; u++) wv[u] = *(const f32x4 *)(wr + k0 + min(c0 + 256 * u, kc - 4));
#pragma unroll
            for (int u = 0; u < RU; u++) {
                const int c = c0 + 256 * u;
                if (c < kc)
#pragma unroll
                    for (int mb = 0; mb < MB; mb++) {
                        const f32x4 xv = *(const f32x4 *)(xs + mb * RK + c);
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[mb] = fmaf(wv[u][e], xv[e], acc[mb]);
                    }
            }
        }
    }
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        const float v = wave_sum(acc[mb]);
        if (lane == 0 && n < N && m0 + mb < M) y[(m0 + mb) * ldy + n] = act(v, a);
    }
}

// Many rows: f32 matrix instructions (v_mfma_f32_32x32x2 / 16x16x4, f32 operands
// and sums), 64 weight rows (output columns) as the A operand and TB tokens as
// the B operand of a wave. Each wave copies its own runs of 32 k (128 B of
// every row) to its own part of LDS by direct loads and reads its fragments
// from there, so no barrier is needed: reading the operands straight into
// registers, one row per lane, costs a cache lookup per lane (proj_out 47 us
// against 35). The order of k within a run is free as long as both
// operands use it: a lane's 16 B feed four MFMAs. KW waves of the workgroup
// take every KW-th run of one tile and meet in LDS, added in wave order; with
// KW = 1 each of the four waves has 64 columns of its own (small K: img_in,
// bound by its output). The next run lands during the current run's MFMAs.
// TB = 16 doubles the workgroups where 32-token tiles would leave CUs without
// one (proj_out: 64 columns). Measured against the 64 x 64 tile kernel:
// proj_out 64 x 4096 at 1024 tokens 900 -> 35 us (64 of 256 CUs at the f32
// matrix rate: 14), txt_in 4096 x 4096 at 77 tokens 815 -> 68 us, img_in
// 4096 x 64 at 1024 tokens 26 -> 16 us.
template <int TB, int KW>
__global__ __launch_bounds__(KW == 1 ? 256 : 64 * KW) void linear_mfma_kernel(
    const float *__restrict__ x, int64_t ldx, const float *__restrict__ w, int64_t M, int64_t N, int64_t K, int a,
    float *__restrict__ y, int64_t ldy, int vec, int mt, int nt) {
    static_assert(TB == 32 || TB == 16, "one MFMA of tokens");
    constexpr int KS = TB == 32 ? 2 : 4;        // lanes' k groups
    constexpr int RUN = 4 * KS;                 // k of one 16 B read of all groups
    constexpr int NL = 32 / RUN;                // reads per 32-k run
    constexpr int NT = 64 / TB;                 // column tiles of the wave's 64
    constexpr int NR = TB * TB / 64;            // accumulator registers per tile
    constexpr int ROWS = 64 + TB;               // weight rows, then tokens
    typedef float acc_t __attribute__((ext_vector_type(NR)));
    constexpr int PITCH = 68;                   // floats per token row of the partial sums
    constexpr int NWV = KW == 1 ? 4 : KW;
    static_assert(TB * PITCH * 4 <= ROWS * 128, "the sums fit the wave's operand rows");
    __shared__ __attribute__((aligned(16))) uint8_t lds[NWV * ROWS * 128];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & (TB - 1), kg = lane / TB;
    // an n tile's token tiles run together on one XCD, whose L2 then serves
    // their repeated weight reads (workgroups are dealt round-robin over 8)
    const int L = blockIdx.x;
    int mi, ni;
    if ((nt & 7) == 0) {
        mi = (L >> 3) % mt;
        ni = (L >> 3) / mt * 8 + (L & 7);
    } else {
        mi = L % mt;
        ni = L / mt;
    }
    const int64_t m0 = (int64_t)mi * TB;
    const int64_t n0 = ((int64_t)ni * (KW == 1 ? 4 : 1) + (KW == 1 ? wave : 0)) * 64;
    const int runs = (int)((K + 31) / 32);
    uint8_t *own = lds + wave * ROWS * 128;

    // direct load i of a run fills rows 8 i .. 8 i + 7: lane l row 8 i + l / 8 at
    // slot l % 8, which holds chunk (l % 8) ^ key(row) (4 k each; swz_key)
    const float *src[ROWS / 8];
    int chunk[2];
#pragma unroll
    for (int i = 0; i < ROWS / 8; i++) {
        const int row = 8 * i + (lane >> 3);
        src[i] = row < 64 ? w + min(n0 + row, N - 1) * K : x + min(m0 + row - 64, M - 1) * ldx;
        if (i < 2) chunk[i] = 4 * ((lane & 7) ^ swz_key(row));  // the key repeats every 16 rows
    }
    // K % 16 == 0: the last run may be short; chunks past it repeat its start and are not used
    auto dma = [&](int rn) __attribute__((always_inline)) {
        const int64_t k = (int64_t)rn * 32;
#pragma unroll
        for (int i = 0; i < ROWS / 8; i++) {
            const int64_t kc = k + chunk[i & 1] < K ? k + chunk[i & 1] : k;
            __builtin_amdgcn_global_load_lds((const void *)(src[i] + kc), (lds_ptr_t)(own + i * 1024), 16, 0, 0);
        }
    };
    acc_t acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < NR; r++) acc[t][r] = 0.f;
    int rn = KW == 1 ? 0 : wave;
    if (rn < runs) dma(rn);
    for (; rn < runs; rn += KW) {
        __builtin_amdgcn_s_waitcnt(WAIT_VM0);
        f32x4 xv[NL], wv[NL][NT];
#pragma unroll
        for (int l = 0; l < NL; l++) {
            const int c = KS * l + kg;
            xv[l] = *(const f32x4 *)(own + swz(64 + lr, c));
#pragma unroll
            for (int t = 0; t < NT; t++) wv[l][t] = *(const f32x4 *)(own + swz(TB * t + lr, c));
        }
        __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);  // the rows are read: the next run may land
        __builtin_amdgcn_sched_barrier(0);
        if (rn + KW < runs) dma(rn + KW);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int l = 0; l < NL; l++) {
            if ((int64_t)rn * 32 + RUN * l >= K) break;
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    if constexpr (TB == 32)
                        acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[l][t][e], xv[l][e], acc[t], 0, 0, 0);
                    else
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[l][t][e], xv[l][e], acc[t], 0, 0, 0);
                }
        }
    }
    // register r of lane (lr, kg): column TB t + 8 (r / 4) + 4 kg + r % 4 (TB = 32)
    // or TB t + 4 kg + r (TB = 16) of token lr; through LDS to whole row pieces
    float *pw = (float *)own + lr * PITCH;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int j = 0; j < NR / 4; j++)
            *(f32x4 *)(pw + TB * t + (TB == 32 ? 8 * j : 0) + 4 * kg) =
                f32x4{acc[t][4 * j], acc[t][4 * j + 1], acc[t][4 * j + 2], acc[t][4 * j + 3]};
    __syncthreads();
    constexpr int STEP = KW == 1 ? 64 : 64 * KW;
    for (int i = KW == 1 ? lane : (int)threadIdx.x; i < TB * 16; i += STEP) {
        const int m = i >> 4, c = (i & 15) * 4;
        const uint8_t *p = (KW == 1 ? own : lds) + (m * PITCH + c) * 4;
        f32x4 v = *(const f32x4 *)p;
#pragma unroll
        for (int q = 1; q < KW; q++) v += *(const f32x4 *)(p + q * ROWS * 128);
        if (m0 + m >= M) continue;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = act(v[e], a);
        float *yr = y + (m0 + m) * ldy + n0 + c;
        if (vec && n0 + c + 4 <= N) {
            *(f32x4 *)yr = v;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n0 + c + e < N) yr[e] = v[e];
        }
    }
}

// one 256-thread workgroup per row: block sum of v over the row
__device__ __forceinline__ float block_sum(float v, float *red) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

// y = x / sqrt(mean(x^2) + eps) * w   (candle_nn::RmsNorm)
__global__ __launch_bounds__(256) void rows_rmsnorm_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                           int64_t D, float eps, float *__restrict__ y) {
    __shared__ float red[4];
    const float *xr = x + (int64_t)blockIdx.x * D;
    float *yr = y + (int64_t)blockIdx.x * D;
    float ss = 0.f;
    for (int64_t i = threadIdx.x; i < D; i += 256) ss += xr[i] * xr[i];
    ss = block_sum(ss, red);
    const float r = 1.0f / sqrtf(ss / (float)D + eps);
    for (int64_t i = threadIdx.x; i < D; i += 256) yr[i] = xr[i] * r * w[i];
}

// y = (x - mean) / sqrt(var + eps) * (1 + scale[row / rows_per])   (two-pass variance)
__global__ __launch_bounds__(256) void rows_ln_scale_kernel(const float *__restrict__ x,
                                                            const float *__restrict__ scale, int64_t D,
                                                            int64_t rows_per, float eps, float *__restrict__ y) {
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const float *xr = x + row * D;
    const float *sr = scale + (row / rows_per) * D;
    float *yr = y + row * D;
    float s = 0.f;
    for (int64_t i = threadIdx.x; i < D; i += 256) s += xr[i];
    const float mean = block_sum(s, red) / (float)D;
    float v = 0.f;
    for (int64_t i = threadIdx.x; i < D; i += 256) {
        const float d = xr[i] - mean;
        v += d * d;
    }
    const float rstd = 1.0f / sqrtf(block_sum(v, red) / (float)D + eps);
    for (int64_t i = threadIdx.x; i < D; i += 256) yr[i] = (xr[i] - mean) * rstd * (1.0f + sr[i]);
}

__global__ void euler_kernel(float *__restrict__ x, const float *__restrict__ v, int64_t n, float dt) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = x[i] + v[i] * dt;
}

__global__ void cfg_kernel(const float *__restrict__ cond, const float *__restrict__ neg, int64_t n, float s,
                           float *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = neg[i] + (cond[i] - neg[i]) * s;
}

__global__ void zero_sinusoid_kernel(float *__restrict__ out, int64_t n, int width) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (int)(i % width) < width / 2 ? 1.0f : 0.0f;
}

struct Floats {
    float v[256];
};
__global__ void set_floats_kernel(float *__restrict__ dst, Floats f, int n) {
    if ((int)threadIdx.x < n) dst[threadIdx.x] = f.v[threadIdx.x];
}

unsigned grid1(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

hipError_t launch_linear_f32(const float *x, int64_t ldx, const float *w, int64_t m, int64_t n, int64_t k, int act_out,
                             float *y, int64_t ldy, hipStream_t stream) {
    if (m <= 0 || n <= 0) return hipSuccess;
    auto blocks = [](int64_t v, int64_t per) { return (unsigned)((v + per - 1) / per); };
    if (k % 4 == 0 && k > 0 && m <= ROWS_MAX && ((uintptr_t)w & 15) == 0) {
        // the rows of one pass over the weights: as many as there are, at most four (64 KB of x in LDS)
        const dim3 grid(blocks(n, 8), blocks(m, m >= 3 ? 4 : m));
        if (m == 1) linear_rows_kernel<1><<<grid, dim3(512), 0, stream>>>(x, ldx, w, m, n, k, act_out, y, ldy);
        else if (m == 2) linear_rows_kernel<2><<<grid, dim3(512), 0, stream>>>(x, ldx, w, m, n, k, act_out, y, ldy);
        else linear_rows_kernel<4><<<grid, dim3(512), 0, stream>>>(x, ldx, w, m, n, k, act_out, y, ldy);
        return hipGetLastError();
    }
    if (k % 16 == 0 && k > 0 && ldx % 4 == 0 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0 && m <= (1 << 24) && n <= (1 << 20)) {
        const int vec = ldy % 4 == 0 && ((uintptr_t)y & 15) == 0;
        auto go = [&](auto kernel, int tb, int nb, int threads) {
            const unsigned mt = blocks(m, tb), nt = blocks(n, nb);
            kernel<<<dim3(mt * nt), dim3(threads), 0, stream>>>(x, ldx, w, m, n, k, act_out, y, ldy, vec, (int)mt, (int)nt);
        };
        if (k < 512)  // too few 32-k runs to share between waves
            go(linear_mfma_kernel<32, 1>, 32, 256, 256);
        else if ((int64_t)blocks(n, 64) * blocks(m, 32) >= device_cu_count())
            go(linear_mfma_kernel<32, 8>, 32, 64, 512);
        else
            go(linear_mfma_kernel<16, 8>, 16, 64, 512);
        return hipGetLastError();
    }
    const dim3 grid(blocks(n, LT), blocks(m, LT));
    linear_any_kernel<<<grid, dim3(256), 0, stream>>>(x, ldx, w, m, n, k, act_out, y, ldy);
    return hipGetLastError();
}

hipError_t launch_set_floats(float *dst, const float *values, int64_t n, hipStream_t stream) {
    for (int64_t at = 0; at < n; at += 256) {
        Floats f{};
        const int len = (int)std::min<int64_t>(256, n - at);
        std::copy(values + at, values + at + len, f.v);
        set_floats_kernel<<<dim3(1), dim3(256), 0, stream>>>(dst + at, f, len);
    }
    return hipGetLastError();
}

// the t = 0 sinusoid [1 .. 1, 0 .. 0] (src/quantized_transformer.rs:334-343)
hipError_t launch_zero_sinusoid(float *out, int64_t rows, int64_t width, hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    zero_sinusoid_kernel<<<dim3(grid1(rows * width)), dim3(256), 0, stream>>>(out, rows * width, (int)width);
    return hipGetLastError();
}

hipError_t launch_rows_rmsnorm(const float *x, const float *w, int64_t rows, int64_t d, float eps, float *y,
                               hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    rows_rmsnorm_kernel<<<dim3((unsigned)rows), dim3(256), 0, stream>>>(x, w, d, eps, y);
    return hipGetLastError();
}

hipError_t launch_rows_ln_scale(const float *x, const float *scale, int64_t rows, int64_t d, int64_t rows_per,
                                float eps, float *y, hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    rows_ln_scale_kernel<<<dim3((unsigned)rows), dim3(256), 0, stream>>>(x, scale, d, rows_per, eps, y);
    return hipGetLastError();
}

hipError_t launch_euler(float *x, const float *v, int64_t n, float dt, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    euler_kernel<<<dim3(grid1(n)), dim3(256), 0, stream>>>(x, v, n, dt);
    return hipGetLastError();
}

hipError_t launch_cfg(const float *cond, const float *neg, int64_t n, float scale, float *out, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    cfg_kernel<<<dim3(grid1(n)), dim3(256), 0, stream>>>(cond, neg, n, scale, out);
    return hipGetLastError();
}

}  // namespace qimm
