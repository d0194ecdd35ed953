// Large-M dequant-GEMM for gfx950 (M >= 512 token rows): C = A (bf16) x W^T.
// Weights with bf16 rows (bf16-stored ones among them; K % 128 == 0) take the
// kernel of qgemm_bf16.hip, other quantized ones with K % 256 == 0 the
// eight-wave kernel of qgemm_wide.hip; this one serves what is left: Q8_0 with
// K % 256 != 0 and bf16-stored weights with K % 128 != 0 or of short K, in plain
// products, in a block's down projection (whose K is the MLP width; the K of its
// other products is the hidden size, a multiple of 256) and in the gate_up of
// bf16-stored weights at hidden 256. q/k/v never comes here (qgemm_route).
//
// Replaces candle's QMatMul::forward (src/quantized_transformer.rs:19-33) on
// the block's token-parallel projections (call sites 133-135, 151, 196, 202).
//
// Tile 256x256x64, 256 threads = 4 waves in a 2x2 grid, each wave 128x128 as
// 4x4 v_mfma_f32_32x32x16_bf16 tiles (accumulators live in AGPRs), one
// workgroup per CU. Per 16-wide k slice a wave reads 8 KB of operands from LDS
// for 16 MFMAs, half the LDS traffic per flop of a 64x64 wave tile. LDS rows
// are dense 128 B with the 16 B chunk index XOR-swizzled by (row & 7), so both
// the staging writes and the MFMA operand reads are bank-conflict free.
// The A tile goes global->LDS directly (no registers); the raw weights are
// loaded two steps ahead and those of step k+1 are dequantized into the other
// LDS stage between the MFMAs of step k. One barrier per 64-wide k step; the
// operand fragments of the next 16-wide slice are read while the current
// slice's MFMAs run. The epilogues work on the accumulators in place.
// Tiles are ordered XCD-aware: each XCD gets a contiguous range of tiles,
// grouped 4 M-tiles at a time so concurrently resident tiles share A rows and
// W columns in that XCD's L2.
#include <type_traits>

#include "device_common.h"
#include "kernels.h"

namespace qimm {
namespace {

constexpr int BM = 256, BN = 256, BK = 64;
constexpr int ROWB = 128;                      // bytes per LDS row: 64 bf16
constexpr int STAGE = 2 * 256 * ROWB;          // A rows then B rows: 64 KB
constexpr int LDS_BYTES = 2 * STAGE;
constexpr int GROUP_M = 4;

// A word whose value the optimizer must not look through (keeps nibble masks as
// whole-word ops so the byte converts below stay v_cvt_f32_ubyte{0..3}).
__device__ __forceinline__ uint32_t opaque(uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
}

// 8 unsigned byte codes (two words) -> 8 bf16 of code*ds + off (exact f32 value,
// rounded to nearest even).
__device__ __forceinline__ u32x4 cvt8(uint32_t x0, uint32_t x1, float ds, float off) {
    auto f = [&](uint32_t x, int i) { return __builtin_fmaf((float)((x >> (8 * i)) & 0xffu), ds, off); };
    return u32x4{pack_bf16x2(f(x0, 0), f(x0, 1)), pack_bf16x2(f(x0, 2), f(x0, 3)),
                 pack_bf16x2(f(x1, 0), f(x1, 1)), pack_bf16x2(f(x1, 2), f(x1, 3))};
}

__device__ __forceinline__ uint32_t word(const u32x4 *v, int byte_off) {
    return v[byte_off >> 4][(byte_off >> 2) & 3];
}

// Raw bytes of one weight row for one 64-wide k step.
struct WRaw {
    u32x4 v[8];
    uint32_t s;
};

template <int FMT>
__device__ __forceinline__ void load_w(const GemmWeight &w, int64_t n, int64_t k0, WRaw &r) {
    const int64_t K = w.k;
    if constexpr (FMT == WF_Q8_0) {
        const uint8_t *p = w.q + n * K + k0;
#pragma unroll
        for (int i = 0; i < 4; i++) r.v[i] = *(const u32x4 *)(p + 16 * i);
        r.s = *(const uint32_t *)(w.scales + n * (K / 32) + k0 / 32);
    } else {
        const uint8_t *p = w.q + (n * K + k0) * 2;
#pragma unroll
        for (int i = 0; i < 8; i++) r.v[i] = *(const u32x4 *)(p + 16 * i);
    }
}

// Per-step dequant constants of one row.
struct WScale {
    float a0, b0, a1, b1;
};

template <int FMT>
__device__ __forceinline__ WScale w_scales(const WRaw &r) {
    WScale s{};
    if constexpr (FMT == WF_Q8_0) {
        const float d0 = f16_bits_to_f32(r.s & 0xffffu), d1 = f16_bits_to_f32(r.s >> 16);
        s.a0 = d0;  // codes biased to unsigned: (q+128)*d - 128*d, exact
        s.b0 = -128.f * d0;
        s.a1 = d1;
        s.b1 = -128.f * d1;
    }
    return s;
}

// bf16 values k in [8j, 8j+8) of the step.
template <int FMT>
__device__ __forceinline__ u32x4 w_chunk(const WRaw &r, const WScale &s, int j) {
    if constexpr (FMT == WF_Q8_0) {
        const uint32_t x0 = opaque(word(r.v, 8 * j) ^ 0x80808080u), x1 = opaque(word(r.v, 8 * j + 4) ^ 0x80808080u);
        return j < 4 ? cvt8(x0, x1, s.a0, s.b0) : cvt8(x0, x1, s.a1, s.b1);
    } else {
        return r.v[j];
    }
}

__device__ __forceinline__ float silu(float g) { return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)); }

template <int FMT, int EPI>
__global__ __launch_bounds__(256, 1) void qgemm_large_kernel(const uint16_t *__restrict__ A, int64_t M,
                                                             int64_t lda, GemmWeight w, EpiParams ep,
                                                             int mt, int nt) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS_BYTES];
    // the wave index as a scalar: the LDS destinations of the direct loads are
    // then scalar values set into M0 without a lane read per load
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, l32 = lane & 31, g = lane >> 5;

    // XCD-aware, M-grouped tile order
    const int total = mt * nt;
    int L = blockIdx.x;
    if ((total & 7) == 0) L = (L & 7) * (total >> 3) + (L >> 3);
    const int per_group = GROUP_M * nt;
    const int grp = L / per_group;
    const int first_m = grp * GROUP_M;
    const int gm = min(mt - first_m, GROUP_M);
    const int mtile = first_m + (L % per_group) % gm;
    const int ntile = (L % per_group) / gm;
    const int64_t m0 = (int64_t)mtile * BM, n0 = (int64_t)ntile * BN;
    const int64_t K = w.k;
    const int KT = (int)(K / BK);

    // A staging by direct global->LDS loads (16 B per lane, lane l lands at
    // base + 16 l): instruction i of wave w fills LDS rows 8(8w+i) .. +8, lane l
    // row 8(8w+i) + l/8 at slot l%8, which must hold logical chunk
    // (l%8) ^ swz_key(row). Rows past M are clamped to row M-1: they only feed
    // output rows the epilogue never writes.
    const uint16_t *asrc[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int row = 8 * (8 * wave + i) + (lane >> 3);
        const int c = (lane & 7) ^ swz_key(row);
        asrc[i] = A + min(m0 + row, M - 1) * lda + 8 * c;
    }
    auto dma_a = [&](int stage, int64_t k0) {
        uint8_t *base = lds + stage * STAGE;
#pragma unroll
        for (int i = 0; i < 8; i++)
            __builtin_amdgcn_global_load_lds((const void *)(asrc[i] + k0), (lds_ptr_t)(base + (8 * wave + i) * 8 * ROWB),
                                             16, 0, 0);
    };
    // bf16 weights (a dequantized copy, [N][K]) take the A path: direct
    // global->LDS loads into the B rows of the stage, same swizzle
    const uint16_t *bsrc[8];
    if constexpr (FMT == WF_BF16) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int row = 8 * (8 * wave + i) + (lane >> 3);
            const int c = (lane & 7) ^ swz_key(row);
            bsrc[i] = (const uint16_t *)w.q + (n0 + row) * K + 8 * c;
        }
    }
    auto dma_b = [&](int stage, int64_t k0) {
        uint8_t *base = lds + stage * STAGE + 256 * ROWB;
#pragma unroll
        for (int i = 0; i < 8; i++)
            __builtin_amdgcn_global_load_lds((const void *)(bsrc[i] + k0), (lds_ptr_t)(base + (8 * wave + i) * 8 * ROWB),
                                             16, 0, 0);
    };
    // W staging (quantized): row n0 + tid, all 8 chunks, through registers
    // (dequantized); raw weights double-buffered two steps ahead
    const int64_t wrow = n0 + tid;
    WRaw rw[2];

    f32x16 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    // operand fragments of one 16-wide k slice, double-buffered across slices
    // (buffer and slice indices are compile-time after unrolling)
    bf16x8 fa[2][4], fb[2][4];
    auto rd = [&](int buf, int stage, int kk) __attribute__((always_inline)) {
        const uint8_t *as = lds + stage * STAGE;
        const uint8_t *bs = as + 256 * ROWB;
#pragma unroll
        for (int i = 0; i < 4; i++) fa[buf][i] = *(const bf16x8 *)(as + swz(wm * 128 + i * 32 + l32, 2 * kk + g));
#pragma unroll
        for (int j = 0; j < 4; j++) fb[buf][j] = *(const bf16x8 *)(bs + swz(wn * 128 + j * 32 + l32, 2 * kk + g));
        // bf16 weights: the reads stay ahead of the MFMAs that follow (those
        // use the other buffer); left alone, the scheduler sinks each read to
        // just before its first use and waits out the LDS latency there (q/k/v
        // shape 441-458 -> 416-424 us). The dequantizing form keeps the
        // scheduler's order: its decode VALU already fills that latency.
        if constexpr (FMT == WF_BF16) __builtin_amdgcn_sched_barrier(0);
    };
    auto mm = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int i = q >> 2, j = q & 3;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[buf][i], fb[buf][j], acc[i][j], 0, 0, 0);
        }
    };

    if constexpr (FMT == WF_BF16) {
        // both operands of steps 0 and 1 in flight, then the same one-barrier
        // step as below without the dequantization
        dma_a(0, 0);
        dma_b(0, 0);
        dma_a(1, (int64_t)min(1, KT - 1) * BK);
        dma_b(1, (int64_t)min(1, KT - 1) * BK);
        __builtin_amdgcn_s_waitcnt(WAIT_VM0_LGKM0);  // vmcnt(0) lgkmcnt(0)
        __syncthreads();
        rd(0, 0, 0);
        auto step_b = [&](int kt, auto sc_) __attribute__((always_inline)) {
            constexpr int s = decltype(sc_)::value, t = s ^ 1;
            rd(1, s, 1);
            mm(0);
            rd(0, s, 2);
            mm(1);
            rd(1, s, 3);
            mm(0);
            __builtin_amdgcn_s_waitcnt(WAIT_VM0_LGKM0);  // stage t's loads (issued a step ago) landed
            __syncthreads();
            dma_a(s, (int64_t)min(kt + 2, KT - 1) * BK);
            dma_b(s, (int64_t)min(kt + 2, KT - 1) * BK);
            rd(0, t, 0);
            mm(1);
        };
        int kt = 0;
        for (; kt + 1 < KT; kt += 2) {
            step_b(kt, std::integral_constant<int, 0>{});
            step_b(kt + 1, std::integral_constant<int, 1>{});
        }
        if (kt < KT) step_b(kt, std::integral_constant<int, 0>{});
    } else {
    // prologue: step 0 staged in stage 0; raw weights of steps 1 and 2 and the
    // A tile of step 1 loaded (step indices clamped to the last step: redundant
    // loads, no branches)
    load_w<FMT>(w, wrow, 0, rw[0]);
    dma_a(0, 0);
    __builtin_amdgcn_s_waitcnt(WAIT_VM0);  // vmcnt(0)
    {
        const WScale sc = w_scales<FMT>(rw[0]);
        uint8_t *bn = lds + 256 * ROWB;
#pragma unroll
        for (int j = 0; j < 8; j++) *(u32x4 *)(bn + swz(tid, j)) = w_chunk<FMT>(rw[0], sc, j);
    }
    load_w<FMT>(w, wrow, (int64_t)min(1, KT - 1) * BK, rw[1]);
    dma_a(1, (int64_t)min(1, KT - 1) * BK);
    load_w<FMT>(w, wrow, (int64_t)min(2, KT - 1) * BK, rw[0]);
    __builtin_amdgcn_s_waitcnt(WAIT_VM0_LGKM0);  // vmcnt(0) lgkmcnt(0)
    __syncthreads();
    rd(0, 0, 0);

    // Step kt, stage s = kt & 1, t = s ^ 1. On entry fa/fb[0] hold slice 0 of
    // step kt, rw[t] holds the raw weights of step kt+1, rw[s] those of step
    // kt+2 and stage t holds the A tile of step kt+1. Slices 0-2 dequantize step
    // kt+1 into stage t while their MFMAs run; then ONE barrier per step: stage t
    // is complete, and every wave is done reading stage s (its last slice sits
    // in registers). After it, stage s receives the A tile of step kt+2 and
    // rw[t] the raw weights of step kt+3 while slice 3 computes and slice 0 of
    // step kt+1 is read. The vmcnt(0) before the barrier covers loads issued a
    // whole step earlier.
    auto step = [&](int kt, auto sc_) __attribute__((always_inline)) {
        constexpr int s = decltype(sc_)::value, t = s ^ 1;
        uint8_t *bn = lds + t * STAGE + 256 * ROWB;
        const WScale sc = w_scales<FMT>(rw[t]);
        rd(1, s, 1);
        mm(0);
#pragma unroll
        for (int c = 0; c < 3; c++) *(u32x4 *)(bn + swz(tid, c)) = w_chunk<FMT>(rw[t], sc, c);
        rd(0, s, 2);
        mm(1);
#pragma unroll
        for (int c = 3; c < 6; c++) *(u32x4 *)(bn + swz(tid, c)) = w_chunk<FMT>(rw[t], sc, c);
        rd(1, s, 3);
        mm(0);
#pragma unroll
        for (int c = 6; c < 8; c++) *(u32x4 *)(bn + swz(tid, c)) = w_chunk<FMT>(rw[t], sc, c);
        __builtin_amdgcn_s_waitcnt(WAIT_VM0_LGKM0);  // vmcnt(0) lgkmcnt(0)
        __syncthreads();
        dma_a(s, (int64_t)min(kt + 2, KT - 1) * BK);
        load_w<FMT>(w, wrow, (int64_t)min(kt + 3, KT - 1) * BK, rw[t]);
        rd(0, t, 0);
        mm(1);
    };
    int kt = 0;
    for (; kt + 1 < KT; kt += 2) {
        step(kt, std::integral_constant<int, 0>{});
        step(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < KT) step(kt, std::integral_constant<int, 0>{});
    }
    __builtin_amdgcn_s_waitcnt(WAIT_VM0);  // vmcnt(0): no load into LDS still in flight

    // ---- epilogue, straight from the accumulators ----
    // acc[i][j][r] holds row wm*128 + 32i + 8(r/4) + 4g + (r%4) and column
    // wn*128 + 32j + l32 of the tile: each lane owns one column of 16 rows per
    // (i, j), 32 lanes cover 32 consecutive columns.
    const int64_t N = w.n;
    const int64_t nw = n0 + wn * 128;  // first global column of this wave
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t mi = m0 + wm * 128 + i * 32 + 4 * g;
        if constexpr (EPI == EPI_F32 || EPI == EPI_BF16) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int64_t m = mi + 8 * (r >> 2) + (r & 3);
                if (m >= M) continue;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int64_t n = nw + j * 32 + l32;
                    const float v = acc[i][j][r];
                    if constexpr (EPI == EPI_F32) {
                        ((float *)ep.out)[m * ep.ldo + n] = v;
                    } else {
                        ((uint16_t *)ep.out)[m * ep.ldo + n] = (uint16_t)(pack_bf16x2(v, 0.f) & 0xffffu);
                    }
                }
            }
        } else if constexpr (EPI == EPI_RESID) {
            // Every load of the 16 rows x 4 columns first (rows past M clamped
            // to M-1), then the stores: one memory round trip per 32 rows
            // instead of one per row. x_out may alias x_in: each element is read
            // and written by the same lane, loads before stores.
            float xv[16][4], gv[16][4];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int64_t m = min(mi + 8 * (r >> 2) + (r & 3), M - 1);
                const float *grow = ep.gvec + (int64_t)((int)m / (int)ep.g_rows_per) * ep.g_stride;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int64_t n = nw + j * 32 + l32;
                    xv[r][j] = ep.x_in[m * N + n];
                    gv[r][j] = grow[n];
                }
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int64_t m = mi + 8 * (r >> 2) + (r & 3);
                if (m >= M) continue;
#pragma unroll
                for (int j = 0; j < 4; j++) ep.x_out[m * N + nw + j * 32 + l32] = xv[r][j] + gv[r][j] * acc[i][j][r];
            }
        } else if constexpr (EPI == EPI_SWIGLU) {
            // columns 32j + l32 (j < 2) are gate, 64 + 32j + l32 the matching up
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int64_t m = mi + 8 * (r >> 2) + (r & 3);
                if (m >= M) continue;
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const float h = silu(acc[i][j][r]) * acc[i][j + 2][r];
                    const int64_t o = m * ep.ldh + nw / 2 + j * 32 + l32;
                    if (ep.hmid_f32)
                        ep.hmid_f32[o] = h;
                    else
                        ep.hmid[o] = (uint16_t)(pack_bf16x2(h, 0.f) & 0xffffu);
                }
            }
        }
    }
}

template <int FMT>
hipError_t launch_fmt(const GemmWeight &w, const uint16_t *a, int64_t m, int64_t lda, int epi,
                      const EpiParams &ep, hipStream_t stream) {
    const int mt = (int)((m + BM - 1) / BM), nt = (int)(w.n / BN);
    dim3 grid((unsigned)(mt * nt)), block(256);
    switch (epi) {
    case EPI_F32: qgemm_large_kernel<FMT, EPI_F32><<<grid, block, 0, stream>>>(a, m, lda, w, ep, mt, nt); break;
    case EPI_BF16: qgemm_large_kernel<FMT, EPI_BF16><<<grid, block, 0, stream>>>(a, m, lda, w, ep, mt, nt); break;
    case EPI_RESID: qgemm_large_kernel<FMT, EPI_RESID><<<grid, block, 0, stream>>>(a, m, lda, w, ep, mt, nt); break;
    case EPI_SWIGLU:
        if constexpr (FMT == WF_BF16) {
            qgemm_large_kernel<FMT, EPI_SWIGLU><<<grid, block, 0, stream>>>(a, m, lda, w, ep, mt, nt);
            break;
        }
        return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

// The 128x128 kernel (split over K where its tiles are still too few) is
// faster whenever its whole grid runs as one wave of its two resident
// workgroups per CU; beyond that its second, partial wave costs more than the
// 256x256 kernel's idle CUs. Measured: Q4_K 4096 x 4096 at 1024 tokens 109 ->
// 66 us and Q6_K 4096 x 12288 352 -> 215 us (256 tiles of 128x128), at 2048
// tokens 2-4% faster (512 tiles); the block step at 1024 image tokens 0.90 ->
// 0.71 ms. At 2304 tokens (576 tiles), 3072, and gate_up at 512 the 256x256
// kernel is faster.
bool qgemm_large_fits(const GemmWeight &w, int64_t m) {
    if (m < 512 || w.n % BN || w.k % BK) return false;
    const int64_t mid_tiles = ((m + 127) / 128) * (w.n / 128);
    return mid_tiles > 2 * (int64_t)device_cu_count();
}

hipError_t launch_qgemm_large(const GemmWeight &w, const uint16_t *a, int64_t m, int64_t lda, int epi,
                              const EpiParams &ep, hipStream_t stream) {
    if (qgemm_wide_fits(w))
        return launch_qgemm_wide(w, a, m, lda, epi, ep, stream);
    switch (w.fmt) {
    case WF_Q8_0: return launch_fmt<WF_Q8_0>(w, a, m, lda, epi, ep, stream);
    case WF_BF16: return launch_fmt<WF_BF16>(w, a, m, lda, epi, ep, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace qimm
