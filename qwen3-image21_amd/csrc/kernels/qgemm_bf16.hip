// Large-M GEMM for gfx950 over bf16 weight rows: C = A (bf16) x W^T with the
// epilogues of the other GEMM kernels. It takes weights stored in bf16 and, for
// quantized weights, the bf16 copy their upload lays out beside the codes (the
// values every decoding kernel multiplies, bit for bit).
//
// Replaces candle's QMatMul::forward (src/quantized_transformer.rs:19-33) on
// the block's token-parallel projections (call sites 133-135, 151, 196, 202).
//
// What bounds it: the matrix pipe at the clock the operand data allows (all-zero
// operands run 1.65-1.85 PFLOP/s, random ones 1.38-1.52). Decoding 32 weights
// per lane and k step beside the MFMAs costs more than reading twice the bytes:
// the decoding kernel of the same tile (qgemm_wide.hip) runs 1.10-1.18, and a
// form of this kernel that decodes in its load phases 1.04-1.17.
//
// 512 threads = 8 waves, two per SIMD: waves w and w + 4 share one. A wave owns
// 128 weight rows x 16 TT tokens (v_mfma_f32_16x16x32_bf16, the weights as the
// A operand); WN x WT waves make the tile, 128 WN rows x 16 TT WT tokens. Both
// operand tiles are copied HBM -> LDS by direct loads (128 B rows of 64 k,
// XOR-swizzled slots), with no staging registers.
//
// A k step is cut into phases of one load part and one MFMA part, a barrier
// after each, and waves 4-7 run one barrier behind waves 0-3: on every SIMD one
// wave multiplies while the other reads its next fragments from LDS and issues
// the direct loads, and the multiplying wave has the higher priority.
//  - TT = 4: four phases (weight half x token half: 16 MFMAs each) over two LDS
//    stages; a quarter of the tile is refilled as soon as both wave groups have
//    read it, so every direct load has at least a whole k step to land.
//  - TT = 2: two phases (weight half x all tokens: 16 MFMAs each), three stages.
// Measured against the decoding kernel (Q4_K, one process, us): at 4096 tokens
// q/k/v 12288 x 4096 366 -> 294, gate_up 24576 x 4096 715 -> 599, 4096 x 12288
// 349 -> 272, 4096 x 4096 126 -> 98; at 3072 tokens q/k/v 326 -> 250; at 2048
// tokens against the 128x128 kernel 4096 x 4096 95 -> 62, 4096 x 12288 (Q6_K)
// 313 -> 172; bf16 weights 12288 x 4096 at 2050 tokens against the four-wave
// kernel of qgemm_large.hip 219 -> 191.
#include <algorithm>
#include <type_traits>

#include "device_common.h"
#include "kernels.h"

namespace qimm {
namespace {

constexpr int BK = 64, ROWB = 128;  // k per step; bytes per LDS row
constexpr int NWAVE = 8;
constexpr int GROUP_TOKENS = 1024;  // tokens whose tiles run together
// Epilogue code of the SwiGLU form that rounds whole Q8_K blocks of the hidden
// state (EpiParams::hmid_q8k): 512 weight rows = 256 hidden columns per tile.
constexpr int EPI_SWIGLU_Q8K = 16;

__device__ __forceinline__ float silu(float g) { return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)); }

// sum / max / min over the four lanes that hold one token's rows (l, l ^ 16, l ^ 32, l ^ 48)
__device__ __forceinline__ float sum_groups(float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}
__device__ __forceinline__ float max_groups(float v) {
    v = fmaxf(v, __shfl_xor(v, 16));
    return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ int min_groups(int v) {
    v = min(v, __shfl_xor(v, 16));
    return min(v, __shfl_xor(v, 32));
}

// Tile shape of an epilogue: waves along the weight rows (the rest along tokens)
template <int EPI>
constexpr int waves_n() {
    return EPI == EPI_SWIGLU_Q8K ? 4 : 2;
}
template <int WN, int TT>
struct Shape {
    static constexpr int WT = NWAVE / WN, BN = 128 * WN, BM = 16 * TT * WT;
    static constexpr int TB = BM * ROWB, WB = BN * ROWB;  // bytes of a stage's token and weight rows
    static constexpr int NS = TT == 4 ? 2 : 3;            // stages
    static constexpr int LDS = NS * (TB + WB);
};

// EPI's epilogue of tile (m0, n0); `head` tiles of 16 * 4 WT tokens first, then,
// with SMALL, tiles of half as many.
template <int EPI, bool SMALL>
__global__ __launch_bounds__(64 * NWAVE, 1) void qgemm_bf16_kernel(const uint16_t *__restrict__ A, int64_t M, int64_t lda,
                                                                 const uint16_t *__restrict__ W, int64_t N, int64_t K,
                                                                 EpiParams ep, int head) {
    constexpr int WN = waves_n<EPI>();
    constexpr int LDS_BYTES = Shape<WN, 4>::LDS > (SMALL ? Shape<WN, 2>::LDS : 0) ? Shape<WN, 4>::LDS : Shape<WN, 2>::LDS;
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS_BYTES];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nt = (int)(N / (128 * WN));
    // a split product (EPI_F32): share blockIdx.y of the k steps, its sums to
    // out [share][M][ldo]
    int KT = (int)(K / BK);
    int64_t k_first = 0;
    if constexpr (EPI == EPI_F32) {
        const int sh = blockIdx.y, n = gridDim.y, k0 = KT * sh / n;
        k_first = (int64_t)k0 * BK;
        KT = KT * (sh + 1) / n - k0;
        ep.out = (float *)ep.out + (int64_t)sh * M * ep.ldo;
    }

    auto tiles = [&](auto tt_, int idx, int mt, int64_t row0) __attribute__((always_inline)) {
        constexpr int TT = decltype(tt_)::value;
        using S = Shape<WN, TT>;
        constexpr int WT = S::WT, BM = S::BM, NS = S::NS, TB = S::TB, WB = S::WB;
        constexpr int GROUP_M = GROUP_TOKENS / BM;
        // XCD-aware order, GROUP_M token tiles at a time
        const int total = mt * nt;
        int L = idx;
        if ((total & 7) == 0) L = (L & 7) * (total >> 3) + (L >> 3);
        const int per_group = GROUP_M * nt, first_m = L / per_group * GROUP_M, gm = min(mt - first_m, GROUP_M);
        const int64_t m0 = row0 + (int64_t)(first_m + (L % per_group) % gm) * BM;
        const int64_t n0 = (int64_t)((L % per_group) / gm) * S::BN;
        const int lane = tid & 63, l16 = lane & 15, lg = lane >> 4;
        const int wn = WT == 4 ? wave >> 2 : wave >> 1, wt = wave & (WT - 1);

        // LDS: token rows of every stage, then weight rows of every stage. A
        // fragment lane reads row l16 of a 16-row tile, chunk 4 ks + lg (8 k).
        uint32_t toff[2], woff[2];
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const uint32_t o = (uint32_t)(l16 * ROWB + (((4 * ks + lg) ^ swz_key(l16)) << 4));
            toff[ks] = wt * 16 * TT * ROWB + o;
            woff[ks] = NS * TB + wn * 128 * ROWB + o;
        }
        // Direct loads: one instruction fills 8 rows, lane l row l / 8 at slot l % 8,
        // which holds chunk (l % 8) ^ key(row). Token part h (of NTP): rows h RT ..
        // of every token wave's 16 TT; weight part h (of 2): rows 64 h .. of every
        // weight wave's 128. Rows past M repeat the last one (outputs not written).
        constexpr int NTP = TT == 4 ? 2 : 1, RT = 16 * TT / NTP;           // token parts, rows per wave and part
        constexpr int TI = WT * RT / 8 / NWAVE, WI = WN * 64 / 8 / NWAVE;  // instructions per wave and part
        static_assert(TI >= 1 && WI >= 1, "every wave loads");
        const char *abase = (const char *)(A + m0 * lda + k_first), *wbase = (const char *)(W + n0 * K + k_first);
        const int mlast = (int)min(M - 1 - m0, (int64_t)BM - 1);
        uint32_t tsrc[NTP][TI], wsrc[WI];
#pragma unroll
        for (int i = 0; i < TI; i++) {
            const int q = TI * wave + i, r = q / (RT / 8) * 16 * TT + q % (RT / 8) * 8 + (lane >> 3);
#pragma unroll
            for (int h = 0; h < NTP; h++)
                tsrc[h][i] = (uint32_t)min(r + h * RT, mlast) * (uint32_t)(2 * lda) + 16 * ((lane & 7) ^ swz_key(r + h * RT));
        }
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const int q = WI * wave + i, r = q / 8 * 128 + q % 8 * 8 + (lane >> 3);
            wsrc[i] = (uint32_t)r * (uint32_t)(2 * K) + 16 * ((lane & 7) ^ swz_key(r));
        }
        auto dma_t = [&](int s, int h, int kt) __attribute__((always_inline)) {
            const char *b = abase + (int64_t)min(kt, KT - 1) * (2 * BK);
#pragma unroll
            for (int i = 0; i < TI; i++) {
                const int q = TI * wave + i, r = q / (RT / 8) * 16 * TT + q % (RT / 8) * 8 + h * RT;
                __builtin_amdgcn_global_load_lds((const void *)(b + tsrc[h][i]), (lds_ptr_t)(lds + s * TB + r * ROWB), 16, 0, 0);
            }
        };
        auto dma_w = [&](int s, int h, int kt) __attribute__((always_inline)) {
            const char *b = wbase + (int64_t)min(kt, KT - 1) * (2 * BK) + (int64_t)h * 64 * 2 * K;
#pragma unroll
            for (int i = 0; i < WI; i++) {
                const int q = WI * wave + i, r = q / 8 * 128 + q % 8 * 8 + h * 64;
                __builtin_amdgcn_global_load_lds((const void *)(b + wsrc[i]), (lds_ptr_t)(lds + NS * TB + s * WB + r * ROWB),
                                                 16, 0, 0);
            }
        };

        f32x4 acc[8][TT];
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int j = 0; j < TT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        bf16x8 wf[4][2], tf[TT][2];  // fragments of one weight half, of all tokens
        auto rd_w = [&](int s, int h) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int ks = 0; ks < 2; ks++)
                    wf[t][ks] = *(const bf16x8 *)(lds + woff[ks] + s * WB + h * 64 * ROWB + t * 16 * ROWB);
        };
        auto rd_t = [&](int s, int h) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < TT / NTP; t++)
#pragma unroll
                for (int ks = 0; ks < 2; ks++)
                    tf[h * (TT / NTP) + t][ks] = *(const bf16x8 *)(lds + toff[ks] + s * TB + h * RT * ROWB + t * 16 * ROWB);
        };
        // Barriers are raw ones: __syncthreads() would wait for every load in flight.
        auto barrier = [&]() __attribute__((always_inline)) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        // One phase: the load part, then the products of weight half i with token
        // part j. `landed` (a count of this wave's newest loads) lets those stay in
        // flight and waits for the older ones: what the next phase reads was issued
        // before them, by every wave, so it is in LDS after the barrier.
        auto phase = [&](auto landed, auto loads, int i, int j) __attribute__((always_inline)) {
            constexpr int n = decltype(landed)::value;
            __builtin_amdgcn_sched_barrier(0);
            loads();
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(WAIT_VM0 | (n & 15) | ((n >> 4) << 14));
            barrier();
            __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int u = 0; u < TT / NTP; u++) {
                        const int jj = j * (TT / NTP) + u;
                        acc[4 * i + t][jj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][ks], tf[jj][ks], acc[4 * i + t][jj], 0, 0, 0);
                    }
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            barrier();
        };
        // A part may be refilled two phases after the phase that reads it: by then
        // both groups have passed the wait that ends their reads.
        if constexpr (TT == 4) {
            using InFlight = std::integral_constant<int, 2 * TI + 2 * WI>;
            dma_t(0, 0, 0);
            dma_w(0, 0, 0);
            dma_t(0, 1, 0);
            dma_w(0, 1, 0);
            dma_t(1, 0, 1);
            dma_w(1, 0, 1);
            __builtin_amdgcn_s_waitcnt(WAIT_VM0 | (TI + WI));  // step 0 has landed
            barrier();
            if (wave >= 4) barrier();  // waves 4-7 run one barrier behind
            // the first token half of a step is read in the last phase of the step
            // before it: 8, 4, 8 and 4 fragment reads per phase instead of 12, 4, 8
            // and none (4096 tokens: 12288 x 4096 307 -> 294 us, 4096 x 12288 285 -> 272)
            rd_t(0, 0);
            auto step = [&](int kt, auto s_) __attribute__((always_inline)) {
                constexpr int s = decltype(s_)::value;
                phase(InFlight{}, [&] { rd_w(s, 0); dma_t(s ^ 1, 1, kt + 1); }, 0, 0);
                phase(InFlight{}, [&] { rd_t(s, 1); dma_w(s ^ 1, 1, kt + 1); }, 0, 1);
                phase(InFlight{}, [&] { rd_w(s, 1); dma_t(s, 0, kt + 2); }, 1, 0);
                phase(InFlight{}, [&] { rd_t(s ^ 1, 0); dma_w(s, 0, kt + 2); }, 1, 1);
            };
            for (int kt = 0; kt < KT; kt += 2) {  // KT is even
                step(kt, std::integral_constant<int, 0>{});
                step(kt + 1, std::integral_constant<int, 1>{});
            }
        } else {
            dma_t(0, 0, 0);
            dma_w(0, 0, 0);
            dma_w(0, 1, 0);
            dma_t(1, 0, 1);
            dma_w(1, 0, 1);
            dma_w(1, 1, 1);
            __builtin_amdgcn_s_waitcnt(WAIT_VM0 | (TI + 2 * WI));
            barrier();
            if (wave >= 4) barrier();
            auto step = [&](int kt, auto s_) __attribute__((always_inline)) {
                constexpr int s = decltype(s_)::value, s2 = (s + 2) % 3;
                phase(std::integral_constant<int, 2 * TI + 3 * WI>{},
                      [&] { rd_t(s, 0); rd_w(s, 0); dma_t(s2, 0, kt + 2); dma_w(s2, 0, kt + 2); }, 0, 0);
                phase(std::integral_constant<int, TI + 3 * WI>{}, [&] { rd_w(s, 1); dma_w(s2, 1, kt + 2); }, 1, 0);
            };
            int kt = 0;
            for (; kt + 3 <= KT; kt += 3) {
                step(kt, std::integral_constant<int, 0>{});
                step(kt + 1, std::integral_constant<int, 1>{});
                step(kt + 2, std::integral_constant<int, 2>{});
            }
            if (kt < KT) step(kt, std::integral_constant<int, 0>{});
            if (kt + 1 < KT) step(kt + 1, std::integral_constant<int, 1>{});
        }
        if (wave < 4) barrier();
        __builtin_amdgcn_s_waitcnt(WAIT_VM0_LGKM0);  // no load into LDS still in flight

        // ---- epilogue: lane (l16, lg) holds of token mw + 16 j + l16 the weight rows
        // nw + 16 i + 4 lg + r (acc[i][j][r]) ----
        const int64_t mw = m0 + wt * 16 * TT + l16, nw = n0 + 128 * wn + 4 * lg;
        if constexpr (EPI == EPI_F32 || EPI == EPI_BF16) {
#pragma unroll
            for (int j = 0; j < TT; j++) {
                const int64_t m = mw + 16 * j;
                if (m >= M) continue;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const f32x4 v = acc[i][j];
                    if constexpr (EPI == EPI_F32)
                        *(f32x4 *)((float *)ep.out + m * ep.ldo + nw + 16 * i) = v;
                    else
                        *(u32x2 *)((uint16_t *)ep.out + m * ep.ldo + nw + 16 * i) =
                            u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
                }
            }
        } else if constexpr (EPI == EPI_RESID) {
            // 16 token rows at a time through the wave's part of LDS, so that the x rows
            // are read and written 512 B at a time, the next 16 rows' x in flight during
            // the current ones' (4096 x 4096 at 4096 tokens 117 -> 110 us against 16 B
            // pieces of 16 rows per access; the plain bf16 epilogue takes 103). x_out may
            // alias x_in: each element is read and written by the same lane.
            constexpr int P = 132;  // floats per staged row
            float *stg = (float *)lds + wave * (16 * P);
            const int64_t mr = m0 + wt * 16 * TT + (lane >> 5), nr = n0 + 128 * wn + 4 * (lane & 31);
            const bool one = m0 / ep.g_rows_per == (min(m0 + BM, M) - 1) / ep.g_rows_per;  // one gate row
            f32x4 xv[2][8], gv{};
            if (one) gv = *(const f32x4 *)(ep.gvec + m0 / ep.g_rows_per * ep.g_stride + nr);
            auto load_x = [&](int j) __attribute__((always_inline)) {
#pragma unroll
                for (int q = 0; q < 8; q++) xv[j & 1][q] = *(const f32x4 *)(ep.x_in + min(mr + 16 * j + 2 * q, M - 1) * N + nr);
            };
            __syncthreads();  // every wave is done with the operand stages
            load_x(0);
#pragma unroll
            for (int j = 0; j < TT; j++) {
                if (j + 1 < TT) load_x(j + 1);
#pragma unroll
                for (int i = 0; i < 8; i++) *(f32x4 *)(stg + l16 * P + 16 * i + 4 * lg) = acc[i][j];
                __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const int64_t m = mr + 16 * j + 2 * q;
                    const f32x4 a = *(const f32x4 *)(stg + (2 * q + (lane >> 5)) * P + 4 * (lane & 31));
                    if (m >= M) continue;
                    const f32x4 gr = one ? gv : *(const f32x4 *)(ep.gvec + m / ep.g_rows_per * ep.g_stride + nr);
                    f32x4 o;
#pragma unroll
                    for (int e = 0; e < 4; e++) o[e] = xv[j & 1][q][e] + gr[e] * a[e];
                    *(f32x4 *)(ep.x_out + m * N + nr) = o;
                }
                __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);  // the rows are read
                __builtin_amdgcn_wave_barrier();
            }
        } else if constexpr (EPI == EPI_SWIGLU || EPI == EPI_SWIGLU_Q8K) {
            // rows interleaved per 64 (gate | up): tiles i < 4 are gate rows, i + 4 the
            // up rows of the same hidden columns hc + 16 i + r
            const int64_t hc = (n0 + 128 * wn) / 2 + 4 * lg;
#pragma unroll
            for (int j = 0; j < TT; j++)
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][j][r] = silu(acc[i][j][r]) * acc[i + 4][j][r];
            if constexpr (EPI == EPI_SWIGLU_Q8K) {
                // candle's Q8_K rounding (quant_act4<256>'s arithmetic): a token's 256
                // columns are the four weight waves' 64: the largest magnitude, then its
                // first column (as column * 2 plus the sign bit), through LDS
                float *red = (float *)lds;            // [WN][BM]
                int *redi = (int *)(lds + WN * BM * 4);  // [WN][BM]
                const int tk = wt * 16 * TT + l16;
                __syncthreads();  // every wave is done with the operand stages
#pragma unroll
                for (int j = 0; j < TT; j++) {
                    float a = 0.f;
#pragma unroll
                    for (int i = 0; i < 4; i++)
#pragma unroll
                        for (int r = 0; r < 4; r++) a = fmaxf(a, fabsf(acc[i][j][r]));
                    a = max_groups(a);
                    if (lg == 0) red[wn * BM + tk + 16 * j] = a;
                }
                __syncthreads();
                float amax[TT];
#pragma unroll
                for (int j = 0; j < TT; j++) {
                    float a = red[tk + 16 * j];
#pragma unroll
                    for (int v = 1; v < WN; v++) a = fmaxf(a, red[v * BM + tk + 16 * j]);
                    amax[j] = a;
                    int f = 0x7fffffff;
#pragma unroll
                    for (int i = 3; i >= 0; i--)
#pragma unroll
                        for (int r = 3; r >= 0; r--) {
                            const float v = acc[i][j][r];
                            const int code = ((64 * wn + 16 * i + 4 * lg + r) << 1) | (v < 0.f ? 1 : 0);
                            f = fabsf(v) == a ? code : f;
                        }
                    f = min_groups(f);
                    if (lg == 0) redi[wn * BM + tk + 16 * j] = f;
                }
                __syncthreads();
#pragma unroll
                for (int j = 0; j < TT; j++) {
                    const int64_t m = mw + 16 * j;
                    int f = redi[tk + 16 * j];
#pragma unroll
                    for (int v = 1; v < WN; v++) f = min(f, redi[v * BM + tk + 16 * j]);
                    float sc, dq;
                    q8k_scales(amax[j], (f & 1) ? -amax[j] : amax[j], sc, dq);
                    if (m >= M) continue;
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        *(u32x2 *)(ep.hmid + m * ep.ldh + hc + 16 * i) = q8k_values4(acc[i][j], sc, dq);
                }
            } else {
#pragma unroll
                for (int j = 0; j < TT; j++) {
                    const int64_t m = mw + 16 * j;
                    if (ep.hmid_q8_0) {
                        // candle's Q8_0 rounding: tiles 2 b and 2 b + 1 are one 32-column block
#pragma unroll
                        for (int b = 0; b < 2; b++) {
                            float a = 0.f;
#pragma unroll
                            for (int i = 2 * b; i < 2 * b + 2; i++)
#pragma unroll
                                for (int r = 0; r < 4; r++) a = fmaxf(a, fabsf(acc[i][j][r]));
                            float sc, dq;
                            q8_0_scales(max_groups(a), sc, dq);
                            if (m < M)
#pragma unroll
                                for (int i = 2 * b; i < 2 * b + 2; i++)
                                    *(u32x2 *)(ep.hmid + m * ep.ldh + hc + 16 * i) = q8_0_values4(acc[i][j], sc, dq);
                        }
                        continue;
                    }
                    if (m >= M) continue;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const f32x4 v = acc[i][j];
                        if (ep.hmid_f32)
                            *(f32x4 *)(ep.hmid_f32 + m * ep.ldh + hc + 16 * i) = v;
                        else
                            *(u32x2 *)(ep.hmid + m * ep.ldh + hc + 16 * i) =
                                u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
                    }
                }
            }
        } else if constexpr (EPI == EPI_QKV) {
            // the wave holds one head (128 fused columns) of its 16 TT tokens
            const int64_t nb = n0 + 128 * wn + ep.n_offset;
            const int sec = (int)(nb / ep.hidden);
            const int64_t head_i = (nb % ep.hidden) / 128;
            const int64_t S = ep.seq, H = ep.heads;
            const uint32_t Su = (uint32_t)S;
            // rows of 128 dims through the wave's own part of LDS (256 B rows, 16 B chunk
            // c of row t at slot c ^ (t % 16)), so that they leave as whole 256 B rows
            uint16_t *stg = (uint16_t *)lds + wave * (16 * TT * 128);
            auto stage = [&](int j, int i, u32x2 v) __attribute__((always_inline)) {
                const int c = (2 * i + (lg >> 1)) ^ l16;
                *(u32x2 *)(stg + (16 * j + l16) * 128 + 8 * c + 4 * (lg & 1)) = v;
            };
            auto store_rows = [&](uint16_t *dst) __attribute__((always_inline)) {
                __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);  // the wave's own rows
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int p = 0; p < 4 * TT; p++) {
                    const int t = 4 * p + lg;
                    const int64_t m = m0 + wt * 16 * TT + t;
                    if (m >= M) continue;
                    const uint32_t b = (uint32_t)m / Su, s = (uint32_t)m % Su;
                    *(u32x4 *)(dst + (((int64_t)b * H + head_i) * S + s) * 128 + 8 * l16) =
                        *(const u32x4 *)(stg + t * 128 + 8 * (l16 ^ (t & 15)));
                }
            };
            __syncthreads();  // every wave is done with the operand stages
            if (sec < 2) {
                // RmsNorm over the head, RoPE on (2 i, 2 i + 1), q also scaled
                const float *nwt = (sec == 0 ? ep.norm_q : ep.norm_k) + 4 * lg;
                const float osc = sec == 0 ? ep.q_scale : 1.0f;
                f32x4 wv[8];
#pragma unroll
                for (int i = 0; i < 8; i++) wv[i] = *(const f32x4 *)(nwt + 16 * i);
#pragma unroll
                for (int j = 0; j < TT; j++) {
                    const uint32_t s = (uint32_t)min(mw + 16 * j, M - 1) % Su;
                    const float *pr = ep.pe + (int64_t)s * 128 + 4 * lg;
                    f32x4 cs[8];
#pragma unroll
                    for (int i = 0; i < 8; i++) cs[i] = *(const f32x4 *)(pr + 16 * i);
                    float ss = 0.f;
#pragma unroll
                    for (int i = 0; i < 8; i++)
#pragma unroll
                        for (int r = 0; r < 4; r++) ss += acc[i][j][r] * acc[i][j][r];
                    const float rs = 1.0f / sqrtf(sum_groups(ss) * (1.0f / 128.0f) + 1e-6f);
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        uint32_t o[2];
#pragma unroll
                        for (int e = 0; e < 2; e++) {
                            const float x0 = acc[i][j][2 * e] * rs * wv[i][2 * e];
                            const float x1 = acc[i][j][2 * e + 1] * rs * wv[i][2 * e + 1];
                            const float co = cs[i][2 * e], sn = cs[i][2 * e + 1];
                            o[e] = pack_bf16x2((x0 * co - x1 * sn) * osc, (x0 * sn + x1 * co) * osc);
                        }
                        stage(j, i, u32x2{o[0], o[1]});
                    }
                }
                store_rows(sec == 0 ? ep.q : ep.k);
            } else {
                // v: rows [B,H,S,128] when v_bhsd is set, then transposed to vt
                // [B,H,128,vt_ld]: d rows of the wave's tokens through LDS
                if (ep.v_bhsd) {
#pragma unroll
                    for (int j = 0; j < TT; j++)
#pragma unroll
                        for (int i = 0; i < 8; i++)
                            stage(j, i, u32x2{pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3])});
                    store_rows(ep.v_bhsd);
                    __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);  // the rows are read
                    __builtin_amdgcn_wave_barrier();
                }
                // d row of 16 TT tokens, its 8-token chunks at slot c ^ (d / 4 % (2 TT)):
                // the 2 B writes of a 16-token tile then spread over the banks
                constexpr int CH = 2 * TT;  // chunks per row
#pragma unroll
                for (int j = 0; j < TT; j++)
#pragma unroll
                    for (int i = 0; i < 8; i++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int d = 16 * i + 4 * lg + r, c = (2 * j + (l16 >> 3)) ^ ((d >> 2) % CH);
                            stg[d * (16 * TT) + 8 * c + (l16 & 7)] = (uint16_t)(pack_bf16x2(acc[i][j][r], 0.f) & 0xffffu);
                        }
                __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);
                __builtin_amdgcn_wave_barrier();
                constexpr int RPI = 64 / CH;  // d rows per pass
                const int c = lane % CH;
                const int64_t m = m0 + wt * 16 * TT + 8 * c;
                const uint32_t b = (uint32_t)min(m, M - 1) / Su, s = (uint32_t)min(m, M - 1) % Su;
#pragma unroll 4
                for (int p = 0; p < 128 / RPI; p++) {
                    const int d = RPI * p + lane / CH;
                    const u32x4 v = *(const u32x4 *)(stg + d * (16 * TT) + 8 * (c ^ ((d >> 2) % CH)));
                    if (m >= M) continue;
                    uint16_t *dst = ep.vt + (((int64_t)b * H + head_i) * 128 + d) * ep.vt_ld + s;
                    if (s + 7 < Su && m + 7 < M && ((uintptr_t)dst & 15) == 0) {
                        *(u32x4 *)dst = v;
                    } else {
                        for (int e = 0; e < 8 && m + e < M; e++) {
                            const uint32_t me = (uint32_t)(m + e);
                            ep.vt[(((int64_t)(me / Su) * H + head_i) * 128 + d) * ep.vt_ld + me % Su] =
                                (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
                        }
                    }
                }
            }
        }
    };
    const int nhead = head * nt, bx = blockIdx.x;
    if (bx < nhead) {
        tiles(std::integral_constant<int, 4>{}, bx, head, 0);
    } else if constexpr (SMALL) {
        constexpr int BM = Shape<WN, 4>::BM, BS = Shape<WN, 2>::BM;
        const int64_t rest = M - (int64_t)head * BM;
        tiles(std::integral_constant<int, 2>{}, bx - nhead, (int)((rest + BS - 1) / BS), (int64_t)head * BM);
    }
}

// ---- the bf16 rows of a quantized weight (its device layout), 32 values per thread ----
__global__ __launch_bounds__(256) void weight_rows_bf16_kernel(GemmWeight w, uint16_t *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, k32 = w.k / 32;
    if (i >= w.n * k32) return;
    const int64_t n = i / k32;
    const int k = (int)(i % k32) * 32;
    // value = code * sc[half] + off, one rounding to f32; codes of the 32 values in 8 words
    uint32_t c[8];
    float sc[2], off = 0.f;
    int bias = 0;  // subtracted from the code
    if (w.fmt == WF_Q8_0) {
        sc[0] = sc[1] = f16_to_f32(w.scales[n * k32 + k / 32]);
        const u32x4 *q = (const u32x4 *)(w.q + n * w.k + k);
#pragma unroll
        for (int e = 0; e < 8; e++) c[e] = q[e >> 2][e & 3] ^ 0x80808080u;  // code + 128, unsigned
        bias = 128;
    } else if (w.fmt == WF_Q4_K) {
        const uint8_t *b = q4k_block(w.q, n, k / 256, w.k / 256), *p = b + 4;
        const int j = (k & 255) / 32, jl = j & 3;
        const int s = j < 4 ? p[jl] & 63 : (p[8 + jl] & 15) | (p[jl] >> 6 << 4);
        const int mn = j < 4 ? p[4 + jl] & 63 : (p[8 + jl] >> 4) | (p[4 + jl] >> 6 << 4);
        sc[0] = sc[1] = f16_to_f32(*(const uint16_t *)b) * (float)s;
        off = -(f16_to_f32(*(const uint16_t *)(b + 2)) * (float)mn);
        const u32x4 *q = (const u32x4 *)(b + 16 + 32 * (j >> 1));
#pragma unroll
        for (int e = 0; e < 8; e++) c[e] = (q[e >> 2][e & 3] >> (4 * (j & 1))) & 0x0F0F0F0Fu;
    } else {  // WF_Q6_K
        const uint8_t *b = q6k_block(w.q, n, k / 256, w.k / 256);
        const int hh = (k & 255) / 128, r = (k & 127) / 32;
        const float d = f16_to_f32(*(const uint16_t *)(b + 208));
#pragma unroll
        for (int h = 0; h < 2; h++) sc[h] = d * (float)(int8_t)b[192 + 8 * hh + 2 * r + h];
        const u32x4 *ql = (const u32x4 *)(b + 64 * hh + 32 * (r & 1)), *qh = (const u32x4 *)(b + 128 + 32 * hh);
#pragma unroll
        for (int e = 0; e < 8; e++)
            c[e] = ((ql[e >> 2][e & 3] >> (r < 2 ? 0 : 4)) & 0x0F0F0F0Fu) |
                   (((qh[e >> 2][e & 3] >> (2 * r)) & 0x03030303u) << 4);
        bias = 32;
    }
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        uint32_t o[4];
#pragma unroll
        for (int h = 0; h < 4; h++) {
            float v[2];
#pragma unroll
            for (int l = 0; l < 2; l++) {
                const int at = 2 * h + l;  // byte of the word pair
                const int code = (int)((c[e + (at >> 2)] >> (8 * (at & 3))) & 0xffu) - bias;
                v[l] = __builtin_fmaf((float)code, sc[e >> 2], off);
            }
            o[h] = pack_bf16x2(v[0], v[1]);
        }
        *(u32x4 *)(out + n * w.k + k + 4 * e) = u32x4{o[0], o[1], o[2], o[3]};
    }
}

template <int EPI>
hipError_t launch_one(const GemmWeight &w, const uint16_t *a, int64_t m, int64_t lda, const EpiParams &ep, int64_t head,
                      int splits, hipStream_t stream) {
    constexpr int WN = waves_n<EPI>(), BM = Shape<WN, 4>::BM, BS = Shape<WN, 2>::BM;
    const int64_t nt = w.n / (128 * WN), rest = std::max<int64_t>(m - head * BM, 0);
    const int64_t wgs = WN == 4 ? (m + BM - 1) / BM * nt : (head + (rest + BS - 1) / BS) * nt;
    qgemm_bf16_kernel<EPI, WN == 2><<<dim3((unsigned)wgs, (unsigned)splits), dim3(64 * NWAVE), 0, stream>>>(
        a, m, lda, w.bf16, w.n, w.k, ep, (int)(WN == 4 ? (m + BM - 1) / BM : head));
    return hipGetLastError();
}

// Time of a round of tiles of 256 and of 128 tokens over the CUs, in us: per k
// step 1.5 and 0.87 with every CU busy, 1.08 and 0.61 for a few workgroups (the
// clock rises: 4096 x 4096 at 300 tokens 79 / 47 us, at 4096 / 2048 tokens 103 /
// 62 us), and about 6 outside the loop.
double round_us(int64_t steps, bool small, int64_t wgs, int64_t cus) {
    const double f = std::min(1.0, (double)wgs / (double)cus);
    return 6.0 + (double)steps * (small ? 0.61 + 0.26 * f : 1.08 + 0.42 * f);
}

}  // namespace

bool qgemm_bf16_fits(const GemmWeight &w) {
    return w.bf16 && w.n % 256 == 0 && w.k % 128 == 0 && w.k > 0 && w.k <= ((int64_t)1 << 21);
}

// Which tiles: the rows as `head` tiles of 256 tokens, dispatched first, and
// the rest in tiles of 128, mixed so that the last round over the CUs is as full
// as it can be (3072 x 12288 x 4096: 277 us in 256-token tiles alone, 287 in
// 128-token tiles, 250 mixed 10 + 4); or, where the 128-token tiles leave CUs
// without one, those tiles split over K (shares of at least 8 steps, at most one
// workgroup per CU, so the partial sums stay within 32 MiB), summed in share
// order by the reduction that applies the epilogue (3 us, and the sums written
// and read once at 8 TB/s, mostly out of the MALL: 4096 x 12288 at 300 tokens, 5
// shares: 41.7 us and 5.3).
Bf16Plan qgemm_bf16_plan(const GemmWeight &w, int64_t m, bool may_split) {
    const int64_t cus = std::max(device_cu_count(), 1), nt = w.n / 256, steps = w.k / BK, full = (m + 255) / 256;
    // the time at which the last of n1 tiles of 256 tokens, then n2 of 128, ends
    auto span = [&](int64_t n1, int64_t n2) {
        const double c1 = round_us(steps, false, n1 + n2, cus), c2 = round_us(steps, true, n1 + n2, cus);
        const int64_t late = n1 % cus, early = cus - late;  // CUs that run one large tile more, the others
        const double t0 = (double)(n1 / cus) * c1, t1 = t0 + c1;
        // small tiles per early (x) and per late CU (y), each round where it ends first:
        // the early ones take c1 / c2 rounds ahead, then the two in turn, late first
        int64_t x = (n2 + early - 1) / early, y = 0;
        const int64_t lead = late ? (int64_t)(c1 / c2) + 1 : x;
        if (x > lead) {
            const int64_t rest = n2 - lead * early, q = rest / cus, r = rest % cus;
            y = q + (r > 0);
            x = lead + q + (r > late);
        }
        return std::max(late ? t1 + (double)y * c2 : t0, t0 + (double)x * c2);
    };
    // the rows themselves, 2 N K bytes at 4 TB/s, whatever the tiles
    const double rows_us = 6.0 + (double)w.n * (double)w.k * 2.0 / 4e6;
    Bf16Plan best{full, 1, span(full * nt, 0)};
    for (int64_t h = 0; h < full; h++) {
        const double t = span(h * nt, (m - 256 * h + 127) / 128 * nt);
        if (t < best.us * 0.995) best = Bf16Plan{h, 1, t};
    }
    best.us = std::max(best.us, rows_us);
    const int64_t tiles = (m + 127) / 128 * nt;
    for (int s = 2; may_split && s <= 16 && tiles * s <= cus && steps / s >= 8 && m * w.n < ((int64_t)1 << 31); s++) {
        const double t = std::max(rows_us, round_us((steps + s - 1) / s, true, tiles * s, cus)) + 3.0 +
                         8.0 * s * (double)m * (double)w.n / 8e6;
        if (t < best.us) best = Bf16Plan{0, s, t};
    }
    return best;
}

// The SwiGLU form that rounds whole Q8_K blocks: tiles of 512 weight rows x 128 tokens.
double qgemm_bf16_q8k_us(const GemmWeight &w, int64_t m) {
    const int64_t cus = std::max(device_cu_count(), 1), tiles = (m + 127) / 128 * (w.n / 512);
    return (double)((tiles + cus - 1) / cus) * (round_us(w.k / BK, false, tiles, cus) + 2.0);
}

hipError_t launch_weight_rows_bf16(const GemmWeight &w, uint16_t *out, hipStream_t stream) {
    if (w.fmt == WF_BF16 || w.k % 32) return hipErrorInvalidValue;
    const int64_t n = w.n * (w.k / 32);
    weight_rows_bf16_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream>>>(w, out);
    return hipGetLastError();
}

hipError_t launch_qgemm_bf16(const GemmWeight &w, const uint16_t *a, int64_t m, int64_t lda, int epi, const EpiParams &ep,
                             const Bf16Plan &plan, hipStream_t stream) {
    if (plan.splits > 1) {
        // partial sums [splits][m][n] after the counter area
        float *part = (float *)((char *)ep.part_ws + STREAM_COUNTER_BYTES);
        EpiParams pe{};
        pe.out = part;
        pe.ldo = w.n;
        const hipError_t e = launch_one<EPI_F32>(w, a, m, lda, pe, 0, plan.splits, stream);
        return e == hipSuccess ? launch_split_epilogue(part, plan.splits, m, w.n, epi, ep, stream) : e;
    }
    switch (epi) {
    case EPI_F32: return launch_one<EPI_F32>(w, a, m, lda, ep, plan.head, 1, stream);
    case EPI_BF16: return launch_one<EPI_BF16>(w, a, m, lda, ep, plan.head, 1, stream);
    case EPI_QKV: return launch_one<EPI_QKV>(w, a, m, lda, ep, plan.head, 1, stream);
    case EPI_RESID: return launch_one<EPI_RESID>(w, a, m, lda, ep, plan.head, 1, stream);
    case EPI_SWIGLU:
        if (ep.hmid_q8k) {
            if (w.n % 512 || !ep.hmid) return hipErrorInvalidValue;
            return launch_one<EPI_SWIGLU_Q8K>(w, a, m, lda, ep, 0, 1, stream);
        }
        return launch_one<EPI_SWIGLU>(w, a, m, lda, ep, plan.head, 1, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace qimm
