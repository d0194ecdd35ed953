// Joint attention for gfx950: image-token queries over [cached prefix K/V ;
// own K/V], non-causal, head_dim 128, bf16 MFMA with f32 online softmax.
//
// Replaces the unmasked cached-step call of chunked_attention /
// flash_attention (src/transformer.rs:246-296) made from Attention::forward
// (src/quantized_transformer.rs:143-148). The two key segments are read in
// place (no concatenation copy, src/quantized_transformer.rs:143-146).
//
// Common formulation: each wave computes S^T = K_blk Q^T for 32 queries with
// v_mfma_f32_32x32x16_bf16, so every lane owns one query column and the row
// max / row sum need only the lane and its partner lane^32. The probabilities
// stay in registers and are the B operand of O^T += V^T P^T.
//
// attn_fast_kernel: 8 (or 4) waves x 32 queries per workgroup; 64-key K and V^T
// tiles copied HBM -> LDS with global_load_lds (no staging registers) into
// XOR-swizzled, conflict-free layouts, double-buffered; the K rows of a 32-key
// half are read in a bit-swapped order so that each lane's P^T registers hold 8
// consecutive keys and every V^T fragment is one 16 B LDS read; the running
// maximum is folded into the S accumulator start (C = -m) and only moves when it
// grew by more than 2^8, so the common path is p = exp2(s) (q pre-scaled by
// scale*log2 e) and the rescale of O is a rare wave-uniform branch; row sums use
// v_dot2_f32_bf16 over the packed bf16 probabilities, the same values the PV
// product uses. The exact form (SMODE 3) follows every growth of the maximum and
// sums the f32 probabilities instead; exact_softmax() says which calls take it.
// With MASKED it also applies the key mask of build_block_causal_mask (image
// ids) and key validity, per 64-key window and wave: a window whose keys all lie
// before the wave's first query, or all share the queries' image block, runs
// unmasked; one with no visible key is skipped; the others test each score. A
// workgroup stops at the last key any of its queries may see (key_limit_kernel).
// Any segment length: the last window of a segment clamps its K rows and V^T
// chunks to the segment and clears the V^T columns past its end. V^T rows of 16 B
// aligned stride (KeySeg::ld) are copied straight into LDS; rows of any other
// stride go through registers (RV).
// Against a register-staged kernel of 4 waves with per-element bounds, which took
// every length that was no multiple of 8 before (kernel times): 6889 queries over
// 131 + 6889 keys, 32 heads 3.04 -> 0.95 ms, 4299 tokens under the block-causal
// mask 2.27 -> 0.66 ms, without the key split below.
#include <algorithm>
#include <type_traits>

#include "device_common.h"
#include "kernels.h"

namespace qimm {
namespace {

using Seg = KeySeg;

// Key mask of build_block_causal_mask (src/attention_mask.rs:18-66): query i
// sees key j when key_valid[b][j] and (i >= j or i and j lie in the same
// image block, img >= 0). img indexes the one sequence that queries and keys
// share (no prefix); key_valid indexes the concatenated [prefix ; own] keys.
struct KeyMask {
    const int32_t *img;     // [Sq] image block id, -1 for text; null: no block-causal term
    const uint8_t *kvalid;  // [B][kv_len]; null: every key valid
    int64_t kv_len;
};

// A bound on every score (log2 units): q_norm >= max ||q|| (as the kernel
// sees q, scale folded in), k_own >= max ||k|| of the own keys, *k_prefix >= max
// ||k|| of the prefix keys (null: no prefix). When q_norm * max(k_own,
// *k_prefix) <= STATIC_MAX every |score| <= STATIC_MAX (Cauchy-Schwarz), and
// the kernel takes p = exp2(score) against the fixed reference 0: no running
// maximum, no rescaling. exp2 of at most 2^STATIC_MAX summed over any key count
// stays far below f32 overflow, and floating-point sums keep their relative
// precision at any scale, so the result is the softmax's. q_norm = 0 disables.
struct ScoreBound {
    const float *k_prefix;
    float q_norm, k_own;
};
constexpr float RESCALE_TH = 8.0f;  // log2 units
constexpr float STATIC_MAX = 64.0f;

// The last, partial round of query tiles over the CUs, split over the keys: tiles
// `full` .. in dispatch order are `parts` workgroups each. Part `slot` (counted
// from `full`) leaves its unnormalized output o[slot][256][128] and, per query,
// its reference point and row sum ml[slot][256][2].
struct KeySplit {
    int64_t full;
    int parts;
    float *o, *ml;
};

// v_permlane32_swap exchanges the upper 32 lanes of its first operand with
// the lower 32 lanes of its second; with both operands holding x, each lane
// ends up with x and x of lane ^ 32 in the pair. Inline asm because the
// compiler folds a max or sum over the builtin's two results when both
// inputs are the same value.
__device__ __forceinline__ void swap32(float &a, float &b) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ float xmax32(float x) {
    float a = x, b = x;
    swap32(a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float xsum32(float x) {
    float a = x, b = x;
    swap32(a, b);
    return a + b;
}
// acc + lo + hi of a packed bf16 pair
__device__ __forceinline__ float dot2_ones(uint32_t pair, float acc) {
    const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), one, acc, false);
}

// Under the block-causal mask query q sees key k when q >= k or both lie in
// the same image block, so the last key it may see is
// lim[q] - 1 = max(q, last index of its image id). One workgroup: the last
// index of every id in LDS (ids outside [0, S) see every key), then lim.
constexpr int LIMIT_MAX_S = 16384;

__global__ __launch_bounds__(1024) void key_limit_kernel(const int32_t *__restrict__ img, int S,
                                                         int32_t *__restrict__ lim) {
    __shared__ int32_t last[LIMIT_MAX_S];
    for (int i = threadIdx.x; i < S; i += 1024) last[i] = -1;
    __syncthreads();
    for (int k = threadIdx.x; k < S; k += 1024) {
        const int id = img[k];
        if (id >= 0 && id < S) atomicMax(&last[id], k);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < S; q += 1024) {
        const int id = img[q];
        lim[q] = (id >= S ? S - 1 : id >= 0 ? max(q, last[id]) : q) + 1;
    }
}

__device__ __forceinline__ int wave_max_i(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ int wave_min_i(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o));
    return v;
}

// f32 output of a wave's 32 queries x 128 d (O^T accumulators: lane l32 owns
// query q0 + l32, o[dt][4 rq + e] is d = 32 dt + 8 rq + 4 g + e), in two
// 64-wide passes through the wave's f32 staging rows (pitch PITCH floats) so
// that every store covers 256 B of a row. All waves of the workgroup call it.
template <int PITCH>
__device__ __forceinline__ void store_out_f32(float *osf, const f32x16 (&o)[4], float inv, int lane,
                                              float *__restrict__ outf, int64_t bb, int64_t Sq, int64_t row_len,
                                              int64_t col0, int64_t q0) {
    const int g = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int hf = 0; hf < 2; hf++) {
        __syncthreads();
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
#pragma unroll
            for (int rq = 0; rq < 4; rq++) {
                const int t = 2 * hf + dt, d = dt * 32 + 8 * rq + 4 * g;
                *(f32x4 *)(osf + l32 * PITCH + d) = f32x4{o[t][4 * rq] * inv, o[t][4 * rq + 1] * inv,
                                                          o[t][4 * rq + 2] * inv, o[t][4 * rq + 3] * inv};
            }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int r = i * 4 + (lane >> 4), c = (lane & 15) * 4;
            const int64_t qi = q0 + r;
            if (qi < Sq) *(f32x4 *)(outf + (bb * Sq + qi) * row_len + col0 + 64 * hf + c) = *(const f32x4 *)(osf + r * PITCH + c);
        }
    }
}

// bf16 output of a wave's 32 queries x 128 d (the same accumulator layout)
// into its staging rows (pitch PITCH bf16). With q8 every 32-d slice dt of a
// query, 16 values in this lane and 16 in its partner half (lane ^ 32), is
// first rounded as candle's Q8_0 activation block (quant_act4<32>'s
// arithmetic): the to_out projection's input when its weight is Q8_0.
template <int PITCH>
__device__ __forceinline__ void stage_out_bf16(uint16_t *os, const f32x16 (&o)[4], float inv, int lane, bool q8) {
    const int g = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int dt = 0; dt < 4; dt++) {
        float v[16];
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = o[dt][r] * inv;
        if (q8) {
            float a = 0.f;
#pragma unroll
            for (int r = 0; r < 16; r++) a = fmaxf(a, fabsf(v[r]));
            float sc, dq;
            q8_0_scales(xmax32(a), sc, dq);
#pragma unroll
            for (int rq = 0; rq < 4; rq++)
                *(u32x2 *)(os + l32 * PITCH + dt * 32 + 8 * rq + 4 * g) =
                    q8_0_values4(f32x4{v[4 * rq], v[4 * rq + 1], v[4 * rq + 2], v[4 * rq + 3]}, sc, dq);
        } else {
#pragma unroll
            for (int rq = 0; rq < 4; rq++)
                *(u32x2 *)(os + l32 * PITCH + dt * 32 + 8 * rq + 4 * g) =
                    u32x2{pack_bf16x2(v[4 * rq], v[4 * rq + 1]), pack_bf16x2(v[4 * rq + 2], v[4 * rq + 3])};
        }
    }
}

// Candle's Q8_K rounding of the output across a head pair (256 values of a
// query = two heads): this head's part of a query's largest magnitude and the
// first column holding it, as (column << 1 | sign), column col0 + d (col0 =
// 128 for the pair's second head); lane and partner half (lane ^ 32) agree.
__device__ __forceinline__ void q8k_query_max(const f32x16 (&o)[4], float inv, int g, int col0, float &amax,
                                              int &first) {
    float a = 0.f;
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) a = fmaxf(a, fabsf(o[dt][r] * inv));
    a = xmax32(a);
    int f = 0x7fffffff;
#pragma unroll
    for (int dt = 3; dt >= 0; dt--)
#pragma unroll
        for (int r = 15; r >= 0; r--) {
            const float v = o[dt][r] * inv;
            const int code = ((col0 + 32 * dt + 8 * (r >> 2) + 4 * (g) + (r & 3)) << 1) | (v < 0.f ? 1 : 0);
            f = fabsf(v) == a ? code : f;
        }
    float lo = __int_as_float(f), hi = lo;
    swap32(lo, hi);
    amax = a;
    first = min(__float_as_int(lo), __float_as_int(hi));
}

// The f32 output of a wave's 32 queries x 128 d that store_out_f32 wrote, read
// back into the accumulator layout (v[dt][r] = d 32 dt + 8 (r / 4) + 4 g + r % 4)
// through the same staging rows: whole 256 B row pieces from memory, then each
// lane its own values. Rows past Sq are not read (their values are not used).
template <int PITCH>
__device__ __forceinline__ void load_back_f32(float *osf, float (&v)[4][16], int lane, const float *__restrict__ outf,
                                              int64_t bb, int64_t Sq, int64_t row_len, int64_t col0, int64_t q0) {
    const int g = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int hf = 0; hf < 2; hf++) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int r = i * 4 + (lane >> 4), c = (lane & 15) * 4;
            const int64_t qi = q0 + r;
            if (qi < Sq) *(f32x4 *)(osf + r * PITCH + c) = *(const f32x4 *)(outf + (bb * Sq + qi) * row_len + col0 + 64 * hf + c);
        }
        __syncthreads();
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
#pragma unroll
            for (int rq = 0; rq < 4; rq++) {
                const f32x4 x = *(const f32x4 *)(osf + l32 * PITCH + dt * 32 + 8 * rq + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; e++) v[2 * hf + dt][4 * rq + e] = x[e];
            }
    }
}

namespace fast {

// A workgroup of NW waves (8, or 4 where 8-wave workgroups leave CUs idle)
// takes 32 NW queries of one head; each wave owns 32 of them.
constexpr int KB = 64;           // keys per block
constexpr int HD = 128;
constexpr int TILE = KB * HD * 2;     // 16 KB: K (64 rows x 256 B) or V^T (128 rows x 128 B)
constexpr int STAGE = 2 * TILE;       // K tile then V^T tile
constexpr int OP = 136;               // bf16 pitch of the output staging rows
constexpr int OPF = 68;               // f32 pitch of the f32 output staging rows (64 d per pass)
constexpr int lds_bytes(int nw) { return 2 * STAGE > nw * 32 * OP * 2 ? 2 * STAGE : nw * 32 * OP * 2; }

// K tile: key row r holds 16 B chunk c at slot c ^ (r % 16); V^T tile: d row
// holds 8-key chunk c at slot c ^ ((d / 2) % 8). A 16-lane phase of b128 reads
// (16 rows, one chunk) then covers all 64 banks once.
// Two waves per SIMD either way: one 8-wave or two 4-wave workgroups per CU.
// SMODE: 0 = the softmax reference is chosen in the kernel from the score
// bound (the prefix keys' norm is a device value); 1 = fixed reference, 2 =
// running maximum, both decided on the host; 3 = exact (!PRE: sl2 is 1 where q
// carries the scale). A kernel with one form has only that loop's registers to
// allocate.
// RV: V^T rows whose stride is not a multiple of 16 B (a caller's dense V^T of
// an odd length) cannot be copied 16 B at a time into LDS: their chunks are
// loaded unaligned into registers one block ahead and written to the same slots.
// SPLIT: the workgroups from KeySplit::full on are parts of tiles: each takes a
// share of its tile's key blocks and leaves its sums (KeySplit) for attn_merge_kernel.
template <int NW, bool PRE, bool MASKED, int SMODE, bool PAIR, bool RV, bool SPLIT>
__global__ __launch_bounds__(64 * NW, 8 / NW) void attn_fast_kernel(const uint16_t *__restrict__ q, Seg s0, Seg s1,
                                                                    int64_t H, int64_t Sq, int64_t nq, int64_t B,
                                                                    float sl2, uint16_t *__restrict__ out,
                                                                    float *__restrict__ outf, KeyMask km,
                                                                    const int32_t *__restrict__ lim,
                                                                    ScoreBound sb, int q8, KeySplit sp) {
    constexpr bool EXACT = SMODE == 3;
    static_assert(!SPLIT || (NW == 8 && (PRE || EXACT) && !PAIR && !RV), "the split form is the block's 8-wave one");
    static_assert(!EXACT || !PRE, "the exact form scales its scores itself");
    static_assert(!RV || EXACT, "lengths of such rows take the exact form");
    static_assert(NW == 4 || NW == 8, "4 or 8 waves");
    static_assert(!PAIR || (!MASKED && !EXACT), "the paired form is the cached step's");
    constexpr int QB = 32 * NW;  // queries per workgroup
    constexpr int DI = 16 / NW;  // DMA instructions per wave per 16 KB tile
    // operand stages / output staging; in the paired form then each query's
    // first-head maximum and its first dimension (2 words per query)
    __shared__ __attribute__((aligned(16))) uint8_t lds[lds_bytes(NW) + (PAIR ? QB * 8 : 0)];
    __shared__ int wlim[NW];
    // the wave index as a scalar (the DMA destinations then go to M0 without a lane read)
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // XCD-aware order: workgroups are dealt round-robin over 8 XCDs; each XCD
    // gets a contiguous range of (batch, head, query tile) so the query tiles
    // of one head share that XCD's L2 copy of its K/V.
    // Under a key limit later query tiles see more keys: they are dispatched
    // first (query tile major in block order, from the last), so that the short
    // tiles fill the tail; workgroup b takes (batch, head) b % (B H), which
    // keeps a head on one XCD when B H is a multiple of 8.
    // The paired form takes heads 2 hp and 2 hp + 1 in turn (H / 2 head pairs).
    const int64_t HP = PAIR ? H / 2 : H;
    const int64_t total = nq * HP * B;
    int64_t L = blockIdx.x;
    int part = 0, parts = 1;
    int64_t slot = 0;  // of the part's sums
    if constexpr (SPLIT)
        if (L >= sp.full) {
            slot = L - sp.full;
            L = sp.full + slot / sp.parts;
            part = (int)(slot % sp.parts);
            parts = sp.parts;
        }
    int64_t qt, bhp;
    if (MASKED && lim) {
        qt = nq - 1 - L / (HP * B);
        bhp = L % (HP * B);
    } else {
        if ((total & 7) == 0) L = (L & 7) * (total >> 3) + (L >> 3);
        qt = L % nq;
        bhp = L / nq;
    }
    const int64_t bb = bhp / HP;
    const int64_t q0 = qt * QB + wave * 32;

    // one head (t: its index in the pair)
    auto head = [&](auto t_) __attribute__((always_inline)) {
        constexpr int t = decltype(t_)::value;
        const int64_t hh = PAIR ? 2 * (bhp % HP) + t : bhp % HP, bh = bb * H + hh;
        // in the paired form every lane-dependent value of a head derives from this
        // copy of the thread index, which the compiler cannot see through (nothing
        // of the second head is computed early and kept live across the first
        // head's loop); the mask keeps the lane's range known
        int lane = tid;
        if constexpr (PAIR) asm volatile("" : "+v"(lane));
        lane &= 63;
        const int g = lane >> 5, l32 = lane & 31;

        // Q^T fragments (B operand): lane holds query q0+l32, d = 16kk + 8g .. +8
        bf16x8 qf[8];
        {
            const int64_t qi = q0 + l32;
            const uint16_t *qr = q + (bh * Sq + (qi < Sq ? qi : 0)) * HD;
#pragma unroll
            for (int kk = 0; kk < 8; kk++) {
                u32x4 v = *(const u32x4 *)(qr + kk * 16 + g * 8);
                if (qi >= Sq) v = u32x4{0u, 0u, 0u, 0u};
                qf[kk] = __builtin_bit_cast(bf16x8, v);
            }
        }

        const int len0 = (int)s0.len, len1 = (int)s1.len, ld0 = (int)s0.ld, ld1 = (int)s1.ld;
        const int nb0 = (len0 + KB - 1) / KB, nb1 = (len1 + KB - 1) / KB;
        int nblk = nb0 + nb1;

        // Mask state of the wave: its queries [q_lo, q_hi], the lane's query qi
        // and image id, the id range of the wave's queries; with a key limit the
        // workgroup's loop ends at the last key any of its queries may see (the
        // block-causal form has no prefix, so keys are the queries' sequence).
        int q_lo = 0, q_hi = 0, qid_min = -1, qid_max = -1;
        if constexpr (MASKED) {
            const int qi = (int)min(q0 + l32, Sq - 1);
            q_lo = (int)min(q0, Sq - 1);
            q_hi = (int)min(q0 + 31, Sq - 1);
            if (km.img) {
                const int idq = km.img[qi];
                qid_min = __builtin_amdgcn_readfirstlane(wave_min_i(idq));
                qid_max = __builtin_amdgcn_readfirstlane(wave_max_i(idq));
            }
            if (lim) {
                const int wl = __builtin_amdgcn_readfirstlane(wave_max_i(lim[qi]));
                if (lane == 0) wlim[wave] = wl;
                __syncthreads();
                int kmax = wlim[0];
#pragma unroll
                for (int i = 1; i < NW; i++) kmax = max(kmax, wlim[i]);
                nblk = min(nblk, (kmax + KB - 1) / KB);
            }
        }
        int j0 = 0;  // the first key block; the last is nblk - 1
        if constexpr (SPLIT) {
            j0 = nblk * part / parts;
            nblk = nblk * (part + 1) / parts;
        }
        const char *kb0 = (const char *)(s0.k + bh * (int64_t)len0 * HD);
        const char *kb1 = (const char *)(s1.k + bh * (int64_t)len1 * HD);
        const char *vb0 = (const char *)(s0.vt + bh * (int64_t)HD * ld0);
        const char *vb1 = (const char *)(s1.vt + bh * (int64_t)HD * ld1);

        // DMA roles: instruction t = wave + NW i fills K rows 4t .. 4t+3 (lane at
        // row 4t + lane/16, slot lane%16) and V^T rows 8t .. 8t+7 (lane at row
        // 8t + lane/8, slot lane%8); lane l lands at LDS base + 16 l.
        uint32_t koff[DI], vrow[DI], vcol[DI];
#pragma unroll
        for (int i = 0; i < DI; i++) {
            const int r = 4 * (wave + NW * i) + (lane >> 4);
            koff[i] = (uint32_t)(r * 256 + (((lane & 15) ^ (r & 15)) << 4));
            const int d = 8 * (wave + NW * i) + (lane >> 3);
            vrow[i] = (uint32_t)d;
            vcol[i] = (uint32_t)(((lane & 7) ^ ((d >> 1) & 7)) << 4);
        }
        // Block j covers keys [kv0, kv0 + 64) of its segment, of which the first hi
        // exist. A short last block clamps its K rows and V^T chunks to the
        // segment (scores from hi on are masked); every load stays inside it.
        struct Blk {
            const char *kb, *vb;
            int len, ld, kv0, hi, kbase;  // kbase: index of the segment's first key in [s0 ; s1]
        };
        auto blk_of = [&](int j) __attribute__((always_inline)) {
            Blk b;
            const bool first = j < nb0;
            b.kbase = first ? 0 : len0;
            b.len = first ? len0 : len1;
            b.ld = first ? ld0 : ld1;
            b.kb = first ? kb0 : kb1;
            b.vb = first ? vb0 : vb1;
            b.kv0 = (first ? j : j - nb0) * KB;
            b.hi = min(KB, b.len - b.kv0);
            return b;
        };
        u32x4 vreg[DI];  // RV: the next block's V^T chunks of this lane
        auto load_v = [&](const Blk &b) __attribute__((always_inline)) {
            const char *vg = b.vb + (int64_t)b.kv0 * 2;
#pragma unroll
            for (int i = 0; i < DI; i++) {
                const char *row = vg + vrow[i] * (uint32_t)(2 * b.ld);
                if (b.hi == KB) {
                    __builtin_memcpy(&vreg[i], row + vcol[i], 16);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int c = (int)(vcol[i] >> 1) + 2 * e;
                        const uint32_t lo = c < b.hi ? ((const uint16_t *)row)[c] : 0u;
                        const uint32_t hi = c + 1 < b.hi ? ((const uint16_t *)row)[c + 1] : 0u;
                        vreg[i][e] = lo | (hi << 16);
                    }
                }
            }
        };
        auto dma = [&](const Blk &b, int stage) __attribute__((always_inline)) {
            uint8_t *base = lds + stage * STAGE;
            const char *kg = b.kb + (int64_t)b.kv0 * 256;
            const char *vg = b.vb + (int64_t)b.kv0 * 2;
            if (b.hi == KB) {
#pragma unroll
                for (int i = 0; i < DI; i++)
                    __builtin_amdgcn_global_load_lds((const void *)(kg + koff[i]),
                                                     (lds_ptr_t)(base + (wave + NW * i) * 1024), 16, 0, 0);
                if constexpr (!RV) {
#pragma unroll
                    for (int i = 0; i < DI; i++)
                        __builtin_amdgcn_global_load_lds((const void *)(vg + (vrow[i] * (uint32_t)(2 * b.ld) + vcol[i])),
                                                         (lds_ptr_t)(base + TILE + (wave + NW * i) * 1024), 16, 0, 0);
                }
            } else {
#pragma unroll
                for (int i = 0; i < DI; i++) {
                    const int r = 4 * (wave + NW * i) + (lane >> 4);
                    const int gr = min(r, b.hi - 1);
                    __builtin_amdgcn_global_load_lds((const void *)(kg + (koff[i] - r * 256) + gr * 256),
                                                     (lds_ptr_t)(base + (wave + NW * i) * 1024), 16, 0, 0);
                }
                if constexpr (!RV) {
#pragma unroll
                    for (int i = 0; i < DI; i++) {
                        const int gc = min((int)vcol[i] >> 1, ((b.hi + 7) & ~7) - 8);
                        __builtin_amdgcn_global_load_lds((const void *)(vg + vrow[i] * (uint32_t)(2 * b.ld) + 2 * gc),
                                                         (lds_ptr_t)(base + TILE + (wave + NW * i) * 1024), 16, 0, 0);
                    }
                    // an end inside a chunk: the lane's own V^T chunks are cleared from the
                    // end on (a masked key's probability is 0, and the row padding may hold
                    // anything: 0 x NaN must not arise). Waiting for them here, once per
                    // segment, keeps the test out of the other blocks' path (1.2% there).
                    if (b.hi & 7) {
                        __builtin_amdgcn_s_waitcnt(WAIT_VM0);
#pragma unroll 1
                        for (int i = 0; i < DI; i++) {
                            u32x4 *p = (u32x4 *)(base + TILE + (wave + NW * i) * 1024 + 16 * lane);
                            const int left = b.hi - (((lane & 7) ^ (((8 * (wave + NW * i) + (lane >> 3)) >> 1) & 7)) << 3);
                            u32x4 v = *p;
#pragma unroll
                            for (int e = 0; e < 4; e++) v[e] &= left > 2 * e + 1 ? 0xffffffffu : left > 2 * e ? 0xffffu : 0u;
                            *p = v;
                        }
                    }
                }
            }
            if constexpr (RV && !MASKED) load_v(b);
        };
        // RV: the next block's chunks go to LDS at the end of a step, before the
        // barrier that publishes them; the masked form has no registers to hold
        // them over a step (132 spilled) and loads them here too.
        auto seal = [&](const Blk &b, int stage) __attribute__((always_inline)) {
            if constexpr (RV && MASKED) load_v(b);
            uint8_t *base = lds + stage * STAGE + TILE;
#pragma unroll
            for (int i = 0; i < DI; i++) *(u32x4 *)(base + (wave + NW * i) * 1024 + 16 * lane) = vreg[i];
        };

        // S^T row m of a 32-key half is key pi(m) = m with bits 2 and 3 swapped,
        // so accumulator register r of lane (l32, g) is key 16 (r / 8) + 8 g + r % 8
        // and P^T register pairs map to consecutive keys. LDS read offsets are per
        // lane; stage, half and d-tile parts are immediates.
        const int krow = (l32 & ~12) | ((l32 & 4) << 1) | ((l32 & 8) >> 1);
        uint32_t kaddr[8], vaddr[2][2];
#pragma unroll
        for (int kk = 0; kk < 8; kk++) kaddr[kk] = (uint32_t)(krow * 256 + (((2 * kk + g) ^ (krow & 15)) << 4));
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int kk = 0; kk < 2; kk++)
                vaddr[h][kk] = (uint32_t)(TILE + l32 * 128 + (((4 * h + 2 * kk + g) ^ ((l32 >> 1) & 7)) << 4));

        f32x16 o[4];
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[dt][r] = 0.f;
        // scores are kept relative to m_run (score units): the S accumulation
        // starts at -m_run
        float m_run = EXACT ? -INFINITY : 0.f, l_run = 0.f;
        f32x16 negm;
#pragma unroll
        for (int r = 0; r < 16; r++) negm[r] = 0.f;
        bool first_half = true;
        bool fresh = true;  // MASKED: this lane's query has seen no visible key yet

        // -inf for the scores of half h of a window that its query does not see.
        // kmask: visible keys of the window (bit kv), kid: lane kv holds the image
        // id of window key kv, kb0: index of the window's first key, partial: test
        // each score (MASKED only)
        auto hide = [&](f32x16 st, int h, int hi, uint64_t kmask, int kid, int kb0,
                        bool partial) __attribute__((always_inline)) {
            if (hi < h * 32 + 32) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int kv = h * 32 + 16 * (r >> 3) + 8 * g + (r & 7);
                    if (kv >= hi) st[r] = -INFINITY;
                }
            }
            if constexpr (MASKED) {
                if (partial) {
                    // branch-free per-score test (bitwise, no short circuit): the
                    // key's validity bit and, with image ids, causal or same block.
                    // The lane's query and its image id are fetched here: only
                    // windows tested score by score need them.
                    const uint32_t kmw = h ? (uint32_t)(kmask >> 32) : (uint32_t)kmask;
                    if (km.img) {
                        const int qi = (int)min(q0 + l32, Sq - 1);
                        const int idq = km.img[qi];
                        const int qrel = qi - kb0 - h * 32;  // keys of this half at or before the query
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            const int kvh = 16 * (r >> 3) + 8 * g + (r & 7);
                            const int idk = __shfl(kid, h * 32 + kvh);
                            const int ok = (int)((kmw >> kvh) & 1u) & ((int)(qrel >= kvh) | ((int)(idq >= 0) & (int)(idk == idq)));
                            st[r] = ok ? st[r] : -INFINITY;
                        }
                    } else {
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            const int kvh = 16 * (r >> 3) + 8 * g + (r & 7);
                            st[r] = ((kmw >> kvh) & 1u) ? st[r] : -INFINITY;
                        }
                    }
                }
            }
            return st;
        };

        auto half_step = [&](const uint8_t *stg, int h, int hi, uint64_t kmask, int kid, int kb0,
                             bool partial, auto stat) __attribute__((always_inline)) {
            constexpr bool STATIC = decltype(stat)::value;
            f32x16 st;
            if constexpr (STATIC) {
#pragma unroll
                for (int r = 0; r < 16; r++) st[r] = 0.f;
            } else {
                st = negm;
            }
#pragma unroll
            for (int kk = 0; kk < 8; kk++) {
                const bf16x8 a = *(const bf16x8 *)(stg + h * 32 * 256 + kaddr[kk]);
                st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qf[kk], st, 0, 0, 0);
            }
            st = hide(st, h, hi, kmask, kid, kb0, partial);
            if constexpr (!STATIC) {
            float m0 = st[0], m1 = st[1];
#pragma unroll
            for (int r = 2; r < 16; r += 2) {
                m0 = fmaxf(m0, st[r]);
                m1 = fmaxf(m1, st[r + 1]);
            }
            float mx = xmax32(fmaxf(m0, m1));
            if (!PRE) mx *= sl2;  // log2 units
            bool rescale;
            if constexpr (MASKED) {
                // a lane's first visible key sets its reference point; a row with
                // none yet keeps 0 (its probabilities are exp2(-inf) = 0)
                const bool has = mx > -INFINITY;
                rescale = __builtin_amdgcn_ballot_w64(fresh ? has : mx > RESCALE_TH) != 0;
            } else {
                rescale = first_half || __builtin_amdgcn_ballot_w64(mx > RESCALE_TH);
            }
            if (rescale) {
                // move the reference point up by d (log2 units); the first half of
                // a row has at least one unmasked key, so d is finite there
                float d, alpha;
                if constexpr (MASKED) {
                    const bool has = mx > -INFINITY;
                    d = fresh ? (has ? mx : 0.f) : fmaxf(mx, 0.f);
                    alpha = fresh ? 0.f : __builtin_amdgcn_exp2f(-d);
                    fresh = fresh && !has;
                } else {
                    d = first_half ? mx : fmaxf(mx, 0.f);
                    alpha = first_half ? 0.f : __builtin_amdgcn_exp2f(-d);
                }
                first_half = false;
                l_run *= alpha;
#pragma unroll
                for (int dt = 0; dt < 4; dt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
                const float draw = PRE ? d : d / sl2;
                m_run += draw;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    st[r] -= draw;
                    negm[r] = -m_run;
                }
            }
            }  // !STATIC
            uint32_t pk[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float a = PRE ? st[2 * i] : st[2 * i] * sl2;
                const float b = PRE ? st[2 * i + 1] : st[2 * i + 1] * sl2;
                pk[i] = pack_bf16x2(__builtin_amdgcn_exp2f(a), __builtin_amdgcn_exp2f(b));
                l_run = dot2_ones(pk[i], l_run);
            }
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const bf16x8 pf = __builtin_bit_cast(bf16x8, u32x4{pk[4 * kk], pk[4 * kk + 1], pk[4 * kk + 2], pk[4 * kk + 3]});
#pragma unroll
                for (int dt = 0; dt < 4; dt++) {
                    const bf16x8 a = *(const bf16x8 *)(stg + dt * 32 * 128 + vaddr[h][kk]);
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pf, o[dt], 0, 0, 0);
                }
            }
        };

        // The fixed-reference form without a mask, split so that both halves'
        // scores come first: the exponentials of half 0 then issue while half 1's
        // QK MFMAs are still in the matrix pipe, and those of half 1 while half 0's
        // PV MFMAs run.
        auto qk_static = [&](const uint8_t *stg, int h) __attribute__((always_inline)) {
            f32x16 st;
#pragma unroll
            for (int r = 0; r < 16; r++) st[r] = 0.f;
#pragma unroll
            for (int kk = 0; kk < 8; kk++) {
                const bf16x8 a = *(const bf16x8 *)(stg + h * 32 * 256 + kaddr[kk]);
                st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qf[kk], st, 0, 0, 0);
            }
            return st;
        };
        auto pv_static = [&](const uint8_t *stg, int h, f32x16 st, int hi) __attribute__((always_inline)) {
            if (hi < h * 32 + 32) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int kv = h * 32 + 16 * (r >> 3) + 8 * g + (r & 7);
                    if (kv >= hi) st[r] = -INFINITY;
                }
            }
            uint32_t pk[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float a = PRE ? st[2 * i] : st[2 * i] * sl2;
                const float b = PRE ? st[2 * i + 1] : st[2 * i + 1] * sl2;
                pk[i] = pack_bf16x2(__builtin_amdgcn_exp2f(a), __builtin_amdgcn_exp2f(b));
                l_run = dot2_ones(pk[i], l_run);
            }
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const bf16x8 pf = __builtin_bit_cast(bf16x8, u32x4{pk[4 * kk], pk[4 * kk + 1], pk[4 * kk + 2], pk[4 * kk + 3]});
#pragma unroll
                for (int dt = 0; dt < 4; dt++) {
                    const bf16x8 a = *(const bf16x8 *)(stg + dt * 32 * 128 + vaddr[h][kk]);
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pf, o[dt], 0, 0, 0);
                }
            }
        };

        // The exact form: the maximum over the window's 64 keys, the reference point
        // always at the running maximum (the largest probability is 1, with no
        // rounding), f32 row sums. A row with no visible key yet has the reference
        // point 0 (its probabilities are exp2(-inf) = 0).
        float m_ref = 0.f;
        auto pv_exact = [&](const uint8_t *stg, int h, const f32x16 &st) __attribute__((always_inline)) {
            uint32_t pk[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float a = __builtin_amdgcn_exp2f(__builtin_fmaf(st[2 * i], sl2, -m_ref));
                const float b = __builtin_amdgcn_exp2f(__builtin_fmaf(st[2 * i + 1], sl2, -m_ref));
                pk[i] = pack_bf16x2(a, b);
                l_run += a;
                l_run += b;
            }
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const bf16x8 pf = __builtin_bit_cast(bf16x8, u32x4{pk[4 * kk], pk[4 * kk + 1], pk[4 * kk + 2], pk[4 * kk + 3]});
#pragma unroll
                for (int dt = 0; dt < 4; dt++) {
                    const bf16x8 a = *(const bf16x8 *)(stg + dt * 32 * 128 + vaddr[h][kk]);
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pf, o[dt], 0, 0, 0);
                }
            }
        };
        auto exact_step = [&](const uint8_t *stg, int hi, uint64_t kmask, int kid, int kb0,
                              bool partial) __attribute__((always_inline)) {
            f32x16 s0 = qk_static(stg, 0), s1 = qk_static(stg, 1);
            s0 = hide(s0, 0, hi, kmask, kid, kb0, partial);
            s1 = hide(s1, 1, hi, kmask, kid, kb0, partial);
            float m0 = s0[0], m1 = s1[0];
#pragma unroll
            for (int r = 1; r < 16; r++) {
                m0 = fmaxf(m0, s0[r]);
                m1 = fmaxf(m1, s1[r]);
            }
            const float m_new = fmaxf(m_run, xmax32(fmaxf(m0, m1)) * sl2);
            if (__builtin_amdgcn_ballot_w64(m_new > m_run)) {
                m_ref = m_new == -INFINITY ? 0.f : m_new;
                const float alpha = __builtin_amdgcn_exp2f(m_run - m_ref);
                m_run = m_new;
                l_run *= alpha;
#pragma unroll
                for (int dt = 0; dt < 4; dt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
            }
            pv_exact(stg, 0, s0);
            pv_exact(stg, 1, s1);
        };

        // MASKED: lane kv loads the image id of window key kv (0 without ids), or
        // KEY_OFF for a padded key, one block ahead; waited for with the tiles.
        constexpr int KEY_OFF = -0x7fffffff - 1;
        int mk = 0;
        auto mask_load = [&](const Blk &b) __attribute__((always_inline)) {
            const int kv = min(lane, b.hi - 1);
            const int64_t key = (int64_t)b.kbase + b.kv0 + kv;
            const bool valid = km.kvalid ? km.kvalid[bb * km.kv_len + key] != 0 : true;
            const int id = km.img ? km.img[key] : 0;
            mk = valid ? id : KEY_OFF;
        };

        // block j computes from stage cur while block j+1 streams into the other
        auto step = [&](int j, int cur, auto stat) __attribute__((always_inline)) {
            const Blk b = blk_of(j);
            int kid = 0, kb0 = 0;
            uint64_t kmask = 0;
            bool skip = false, partial = false;
            if constexpr (MASKED) {
                // classify the window for this wave's queries (wave-uniform)
                kid = mk;
                kb0 = b.kbase + b.kv0;
                const bool in = lane < b.hi;
                const uint64_t inm = __builtin_amdgcn_ballot_w64(in);
                kmask = __builtin_amdgcn_ballot_w64(in && mk != KEY_OFF);
                const int k_lo = kb0, k_hi = kb0 + b.hi - 1;
                bool full = kmask == inm, empty = kmask == 0;
                if (km.img) {
                    const uint64_t same = __builtin_amdgcn_ballot_w64(in && mk == qid_min);
                    const bool one_block = qid_min == qid_max && qid_min >= 0;
                    full = full && (k_hi <= q_lo || (one_block && same == inm));
                    empty = empty || (k_lo > q_hi && (qid_max < 0 || (qid_min == qid_max && same == 0)));
                }
                skip = empty;
                partial = !full && !empty;
                if (j + 1 < nblk) mask_load(blk_of(j + 1));
            }
            if (j + 1 < nblk) dma(blk_of(j + 1), cur ^ 1);
            const uint8_t *stg = lds + cur * STAGE;
            if constexpr (EXACT) {
                if (!skip) exact_step(stg, b.hi, kmask, kid, kb0, partial);
            } else if constexpr (decltype(stat)::value && !MASKED) {
                const f32x16 s0 = qk_static(stg, 0), s1 = qk_static(stg, 1);
                pv_static(stg, 0, s0, b.hi);
                pv_static(stg, 1, s1, b.hi);
            } else if (!skip) {
                half_step(stg, 0, b.hi, kmask, kid, kb0, partial, stat);
                half_step(stg, 1, b.hi, kmask, kid, kb0, partial, stat);
            }
            __builtin_amdgcn_s_waitcnt(WAIT_VM0);  // vmcnt(0): block j+1 landed
            if constexpr (RV)
                if (j + 1 < nblk) seal(blk_of(j + 1), cur ^ 1);
            __syncthreads();
        };

        if (nblk > j0) {
            if constexpr (MASKED) mask_load(blk_of(j0));
            dma(blk_of(j0), 0);
        }
        __builtin_amdgcn_s_waitcnt(WAIT_VM0);
        if constexpr (RV)
            if (nblk > j0) seal(blk_of(j0), 0);
        __syncthreads();
        // the fixed-reference form when the score bound allows it (wave-uniform)
        bool stat_ok = false;
        if (!EXACT && sb.q_norm > 0.f) {
            const float kn = sb.k_prefix ? fmaxf(sb.k_own, *sb.k_prefix) : sb.k_own;
            stat_ok = sb.q_norm * kn <= STATIC_MAX;
        }
        auto run = [&](auto stat) __attribute__((always_inline)) {
            int j = j0;
            for (; j + 1 < nblk; j += 2) {
                step(j, 0, stat);
                step(j + 1, 1, stat);
            }
            if (j < nblk) step(j, 0, stat);
        };
        if constexpr (SMODE == 1) {
            run(std::true_type{});
        } else if constexpr (SMODE == 2 || EXACT) {
            run(std::false_type{});
        } else {
            if (stat_ok)
                run(std::true_type{});
            else
                run(std::false_type{});
        }

        // normalize and stage O [32 q x 128 d] per wave through LDS for row stores
        const float l_tot = xsum32(l_run);
        if constexpr (SPLIT)
            if (parts > 1) {
                if (g == 0) {
                    float *ml = sp.ml + (slot * QB + wave * 32 + l32) * 2;
                    ml[0] = m_run;
                    ml[1] = l_tot;
                }
                store_out_f32<OPF>((float *)lds + wave * 32 * OPF, o, 1.0f, lane, sp.o + slot * QB * HD, 0, QB, HD, 0,
                                   wave * 32);
                return;
            }
        const float inv = 1.0f / l_tot;
        const int64_t HDt = H * HD;
        uint16_t *os = (uint16_t *)lds + wave * 32 * OP;
        // the wave's staged bf16 rows to out at columns col0 ..
        auto store_rows = [&](int64_t col0) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int r = i * 4 + (lane >> 4);
                const int c = (lane & 15) * 8;
                const int64_t qi = q0 + r;
                if (qi < Sq)
                    *(u32x4 *)(out + (bb * Sq + qi) * HDt + col0 + c) = *(const u32x4 *)(os + r * OP + c);
            }
        };
        if constexpr (PAIR) {
            // Q8_K rounding over the head pair: the first head leaves its f32
            // output in outf (scratch) and each query's largest magnitude and
            // first column in LDS; the second combines them (the first head's
            // columns come first: it wins ties), reads the first head's values
            // back and stores both heads rounded (quant_act4<256>'s arithmetic)
            float a;
            int f;
            q8k_query_max(o, inv, g, 128 * t, a, f);
            float *pmax = (float *)(lds + lds_bytes(NW));
            int *pfirst = (int *)(pmax + QB);
            const int qslot = wave * 32 + l32;
            if constexpr (t == 0) {
                if (g == 0) {
                    pmax[qslot] = a;
                    pfirst[qslot] = f;
                }
                store_out_f32<OPF>((float *)lds + wave * 32 * OPF, o, inv, lane, outf, bb, Sq, HDt, hh * HD, q0);
                __syncthreads();  // staging reads done before the second head's stages land
            } else {
                if (!(a > pmax[qslot])) {
                    a = pmax[qslot];
                    f = pfirst[qslot];
                }
                float sc, dq;
                q8k_scales(a, (f & 1) ? -a : a, sc, dq);
                float va[4][16];
                load_back_f32<OPF>((float *)lds + wave * 32 * OPF, va, lane, outf, bb, Sq, HDt, (hh - 1) * HD, q0);
#pragma unroll
                for (int hd = 0; hd < 2; hd++) {
                    __syncthreads();
#pragma unroll
                    for (int dt = 0; dt < 4; dt++)
#pragma unroll
                        for (int rq = 0; rq < 4; rq++) {
                            f32x4 x;
#pragma unroll
                            for (int e = 0; e < 4; e++) x[e] = hd == 0 ? va[dt][4 * rq + e] : o[dt][4 * rq + e] * inv;
                            *(u32x2 *)(os + l32 * OP + dt * 32 + 8 * rq + 4 * g) = q8k_values4(x, sc, dq);
                        }
                    __syncthreads();
                    store_rows((hh - 1 + hd) * HD);
                }
            }
            return;
        }
        if (outf) {
            store_out_f32<OPF>((float *)lds + wave * 32 * OPF, o, inv, lane, outf, bb, Sq, HDt, hh * HD, q0);
            return;
        }
        stage_out_bf16<OP>(os, o, inv, lane, q8 != 0);
        __syncthreads();
        store_rows(hh * HD);
    };
    head(std::integral_constant<int, 0>{});
    if constexpr (PAIR) head(std::integral_constant<int, 1>{});
}

// Sums the parts of split tile blockIdx.x / 32 (in part order; relative to the
// largest reference point), normalizes and stores as attn_fast_kernel does: one
// query per 32 lanes, 4 d per lane, eight queries per workgroup.
__global__ __launch_bounds__(256) void attn_merge_kernel(KeySplit sp, int64_t nq, int64_t H, int64_t B, int64_t Sq,
                                                         int by_limit, uint16_t *__restrict__ out,
                                                         float *__restrict__ outf, int q8) {
    const int64_t r = blockIdx.x >> 5, total = nq * H * B;
    const int ql = (int)(blockIdx.x & 31) * 8 + (threadIdx.x >> 5), d = (threadIdx.x & 31) * 4;
    int64_t L = sp.full + r, qt, bh;  // the tile, as attn_fast_kernel maps it
    if (by_limit) {
        qt = nq - 1 - L / (H * B);
        bh = L % (H * B);
    } else {
        if ((total & 7) == 0) L = (L & 7) * (total >> 3) + (L >> 3);
        qt = L % nq;
        bh = L / nq;
    }
    const int64_t qi = qt * 256 + ql;
    if (qi >= Sq) return;
    const float *ml = sp.ml + (r * sp.parts * 256 + ql) * 2, *o = sp.o + (r * sp.parts * 256 + ql) * HD + d;
    float m = -INFINITY;
    for (int p = 0; p < sp.parts; p++)  // a part without a visible key has no reference point
        if (ml[p * 512 + 1] > 0.f) m = fmaxf(m, ml[p * 512]);
    f32x4 acc{0.f, 0.f, 0.f, 0.f};
    float l = 0.f;
    for (int p = 0; p < sp.parts; p++) {
        const float lp = ml[p * 512 + 1], a = lp > 0.f ? __builtin_amdgcn_exp2f(ml[p * 512] - m) : lp;
        l += a * lp;
        const f32x4 v = *(const f32x4 *)(o + (int64_t)p * 256 * HD);
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] += a * v[e];
    }
    const float inv = 1.0f / l;
#pragma unroll
    for (int e = 0; e < 4; e++) acc[e] *= inv;
    const int64_t at = ((bh / H) * Sq + qi) * (H * HD) + (bh % H) * HD + d;
    if (outf)
        *(f32x4 *)(outf + at) = acc;
    else if (q8)
        *(u32x2 *)(out + at) = quant_act4<32>(acc);
    else
        *(u32x2 *)(out + at) = u32x2{pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3])};
}

}  // namespace fast

template <int NW, bool PRE, bool MASKED, int SMODE = 0, bool PAIR = false, bool RV = false, bool SPLIT = false>
void launch_fast(const uint16_t *q, Seg s0, Seg s1, int64_t h, int64_t sq, int64_t b, float sl2, uint16_t *out,
                 float *outf, const KeyMask &km, const int32_t *lim, const ScoreBound &sb, int q8,
                 hipStream_t stream, KeySplit sp = KeySplit{0, 1, nullptr, nullptr}) {
    if constexpr (!SPLIT && NW == 8 && (PRE || SMODE == 3) && !PAIR && !RV)
        if (sp.parts > 1)
            return launch_fast<NW, PRE, MASKED, SMODE, PAIR, RV, true>(q, s0, s1, h, sq, b, sl2, out, outf, km, lim, sb, q8,
                                                                       stream, sp);
    const int64_t nq = (sq + 32 * NW - 1) / (32 * NW);
    const int64_t tiles = nq * (PAIR ? h / 2 : h) * b, rest = SPLIT ? tiles - sp.full : 0;
    fast::attn_fast_kernel<NW, PRE, MASKED, SMODE, PAIR, RV, SPLIT>
        <<<dim3((unsigned)(tiles + rest * (sp.parts - 1))), dim3(64 * NW), 0, stream>>>(q, s0, s1, h, sq, nq, b, sl2, out,
                                                                                        outf, km, lim, sb, q8, sp);
    if constexpr (SPLIT)
        fast::attn_merge_kernel<<<dim3((unsigned)(rest * 32)), dim3(256), 0, stream>>>(sp, nq, h, b, sq, MASKED && lim ? 1 : 0,
                                                                                      out, outf, q8);
}

// The masked kernel with the softmax form decided on the host where the score
// bound needs no device value (no prefix keys).
template <bool PRE>
void launch_masked(const uint16_t *q, Seg s0, Seg s1, int64_t h, int64_t sq, int64_t b, float sl2, uint16_t *out,
                   float *outf, const KeyMask &km, const int32_t *lim, const ScoreBound &sb, int q8,
                   hipStream_t stream, const KeySplit &sp) {
    if (sb.q_norm <= 0.f)
        launch_fast<8, PRE, true, 2>(q, s0, s1, h, sq, b, sl2, out, outf, km, lim, sb, q8, stream, sp);
    else if (sb.k_prefix)
        launch_fast<8, PRE, true, 0>(q, s0, s1, h, sq, b, sl2, out, outf, km, lim, sb, q8, stream, sp);
    else if (sb.q_norm * sb.k_own <= STATIC_MAX)
        launch_fast<8, PRE, true, 1>(q, s0, s1, h, sq, b, sl2, out, outf, km, lim, sb, q8, stream, sp);
    else
        launch_fast<8, PRE, true, 2>(q, s0, s1, h, sq, b, sl2, out, outf, km, lim, sb, q8, stream, sp);
}

// Waves per workgroup of the unmasked fast kernel, from the rounds each form
// takes. An 8-wave workgroup holds a CU alone; a round of them costs 1. Two
// 4-wave workgroups share a CU and do the same work in 1.05 (one wave per
// SIMD each, twice the K/V tile traffic per query); a round with at most one
// 4-wave workgroup per CU, half the work, takes 0.84. Measured at 32 heads,
// 256 prefix keys on 256 CUs: 1024 queries 42.3 -> 35.7 us and 2304 queries
// 150 -> 133 us with 4 waves, 4096 queries 268 us with 8 against 282 with 4.
int fast_waves(int64_t bh, int64_t sq) {
    const int64_t cus = device_cu_count();
    if (cus <= 0) return 8;
    const int64_t n8 = (sq + 255) / 256 * bh, n4 = (sq + 127) / 128 * bh;
    const int64_t c8 = 100 * ((n8 + cus - 1) / cus);
    const int64_t r4 = n4 % (2 * cus);
    const int64_t c4 = 105 * (n4 / (2 * cus)) + (r4 == 0 ? 0 : r4 <= cus ? 84 : 105);
    return c4 < c8 ? 4 : 8;
}

// Parts per tile of the last, partial round of 8-wave tiles (the others run
// whole), 1 = not split, by an estimate in us: a tile takes 2.15 us per key block
// (2.7 masked) and about 8 beside them, a part its share and the 8; the parts'
// sums are written and read once (131 KB each at 4 TB/s) by one launch more.
// Never more than two parts per CU: 68 MB of sums. `now` is the estimate without it.
// Under the block-causal mask the last tiles are the first queries', priced as if
// they saw every key: so do those of an image block near the start (an edit's), while
// a long prompt's see a few hundred, and the split then only costs its launch and sums
// (about 20 us); the ids are on the device, so the host cannot tell.
// Measured at 32 heads, kernel and merge: 4299 masked tokens (544 tiles for 256
// CUs, the last 32 in 8 parts) 661 -> 385 us, 6889 queries over 7020 keys (864
// tiles, the last 96 in 2) 953 -> 793, 3072 over 3289 (384, the last 128 in 2;
// 4-wave tiles before) 236 -> 200.
constexpr int MAX_PARTS = 8;
int split_parts(int64_t bh, int64_t sq, int64_t keys, bool masked, double now, double more) {
    const int64_t cus = device_cu_count(), tiles = (sq + 255) / 256 * bh;
    if (cus <= 0 || tiles % cus == 0) return 1;
    const int64_t rest = tiles % cus;
    const double loop = (masked ? 2.7 : 2.15) * (double)((keys + 63) / 64);
    int best = 1;
    double best_us = 0.97 * now;
    for (int s = 2; s <= MAX_PARTS && rest * s <= 2 * cus; s++) {
        const double us = (double)(tiles / cus) * (loop + 8.0) + (double)((rest * s + cus - 1) / cus) * (loop / s + 8.0) + 6.0 +
                          (double)(rest * s) * 0.131 * 2.0 / 4.0 + more;
        if (us < best_us) {
            best_us = us;
            best = s;
        }
    }
    return best;
}
double tile_rounds_us(int64_t bh, int64_t sq, int64_t keys, bool masked, double rounds) {
    return rounds * ((masked ? 2.7 : 2.15) * (double)((keys + 63) / 64) + 8.0);
}
KeySplit key_split(int64_t bh, int64_t sq, int parts, float *scratch) {
    const int64_t cus = device_cu_count(), tiles = (sq + 255) / 256 * bh, rest = tiles % cus;
    return KeySplit{tiles - rest, parts, scratch, scratch + rest * parts * 256 * 128};
}

// sl2 = softmax scale * log2(e) applied to raw scores, or 1 when q already
// carries it (PRE)
// The output rounding of the launchers (out_qblk): 0 none (bf16 to out, or f32
// to outf when it is set); 32 candle's Q8_0 blocks, rounded in the kernels'
// epilogue; 256 Q8_K blocks, which span two heads: the paired kernel rounds
// them where it runs (the cached step's 8-wave form, an even head count),
// else the output goes to outf in f32 and the rows quantizer rounds it. outf
// is the f32 scratch [B, Sq, H * 128] for 256.
bool out_qblk_ok(int out_qblk, const float *outf) {
    return out_qblk == 0 || out_qblk == 32 || (out_qblk == 256 && outf);
}
hipError_t finish_q8k(int out_qblk, bool rounded, const float *outf, int64_t b, int64_t h, int64_t sq,
                      uint16_t *out, hipStream_t stream) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || out_qblk != 256 || rounded) return e;
    return launch_quant_rows(outf, h * 128, b * sq, h * 128, 256, out, h * 128, stream);
}

// [prefix ; own] with an empty prefix dropped; false: not a valid pair
bool segments(KeySeg prefix, KeySeg own, Seg &s0, Seg &s1) {
    if (prefix.len < 0 || own.len < 0 || prefix.len + own.len <= 0) return false;
    if ((prefix.len > 0 && prefix.ld < prefix.len) || (own.len > 0 && own.ld < own.len)) return false;
    s0 = prefix.len > 0 ? prefix : own;
    s1 = prefix.len > 0 ? own : KeySeg{own.k, own.vt, 0, own.ld};
    return true;
}
// V^T rows that start on 16 B (their base does): copied straight into LDS. The
// cache's and the block's own V^T always have such rows; a caller's dense V^T
// has them when its length is a multiple of 8.
bool rows16(const Seg &s) { return s.len == 0 || s.ld % 8 == 0; }

// Which calls take the exact form: those with a segment length that is no multiple
// of 8, and the block-causal mask without key limits. There is no other reason in
// the lengths than that these calls have always had its precision (a register-staged
// kernel of their own served them) and keep it, while the multiples of 8 have always
// had the lagging and fixed references. Relative error against 64 bits: exact /
// fixed, queries like their keys, 77 keys 1.71e-3 / 2.13e-3, 765 keys 1.91e-3 /
// 2.15e-3; exact / lagging, random queries, 2577 keys 2.26e-3 / 2.33e-3. Time:
// as the lagging form's; attention of a block, fixed -> exact: 3072 queries over 217 +
// 3072 keys 201 -> 221 us, 6889 over 131 + 6889 757 -> 845, block-causal 4299 353 -> 409,
// 4096 over 217 + 4096 309 -> 340 with the Q8_K rounding as a pass (the paired kernel
// has no exact form).
bool exact_softmax(const KeySeg &prefix, const KeySeg &own, bool unlimited) {
    return ((prefix.len | own.len) & 7) != 0 || unlimited;
}

template <bool PRE>
hipError_t launch(const uint16_t *q, KeySeg prefix, KeySeg own, int64_t b, int64_t h, int64_t sq, float sl2,
                  uint16_t *out, float *outf, const ScoreBound &sb, int out_qblk, hipStream_t stream,
                  float *scratch = nullptr, bool round_later = false) {
    if (sq <= 0 || b <= 0 || h <= 0) return hipSuccess;
    Seg s0, s1;
    if (!segments(prefix, own, s0, s1) || !out_qblk_ok(out_qblk, outf)) return hipErrorInvalidValue;
    const int q8 = out_qblk == 32 && !round_later;
    float *f32out = q8 ? nullptr : outf;  // f32 output (0 with outf, 256 not paired, or round_later)
    bool rounded = round_later;
    const KeyMask km{nullptr, nullptr, prefix.len + own.len};
    const int nw = fast_waves(b * h, sq);
    const bool exact = exact_softmax(prefix, own, false);
    const bool pair = PRE && !exact && out_qblk == 256 && nw == 8 && h % 2 == 0;
    constexpr int SM = PRE ? 0 : 2;  // without the block's norms no score bound is known
    if constexpr (PRE)
        if (scratch && rows16(s0) && rows16(s1)) {
            const int64_t cus = std::max(device_cu_count(), 1), keys = prefix.len + own.len, n8 = (sq + 255) / 256 * b * h;
            const int64_t n4 = (sq + 127) / 128 * b * h, r4 = n4 % (2 * cus);
            const double rounds = pair ? 2.0 * (double)((n8 / 2 + cus - 1) / cus)
                                  : nw == 8 ? (double)((n8 + cus - 1) / cus)
                                            : 1.05 * (double)(n4 / (2 * cus)) + (r4 == 0 ? 0.0 : r4 <= cus ? 0.84 : 1.05);
            // the paired kernel rounds in its epilogue, the split one in a pass over f32 rows
            const double more = pair ? 5.0 + (double)(b * sq * h) * 128.0 * 6.0 / 4.5e6 : 0.0;
            if (const int parts = split_parts(b * h, sq, keys, false, tile_rounds_us(b * h, sq, keys, false, rounds), more);
                parts > 1) {
                const KeySplit sp = key_split(b * h, sq, parts, scratch);
                if (exact)
                    launch_fast<8, false, false, 3>(q, s0, s1, h, sq, b, sl2, out, f32out, km, nullptr, sb, q8, stream, sp);
                else
                    launch_fast<8, true, false>(q, s0, s1, h, sq, b, sl2, out, f32out, km, nullptr, sb, q8, stream, sp);
                return finish_q8k(out_qblk, rounded, outf, b, h, sq, out, stream);
            }
        }
    if (!rows16(s0) || !rows16(s1)) {
        if (nw == 4)
            launch_fast<4, false, false, 3, false, true>(q, s0, s1, h, sq, b, sl2, out, f32out, km, nullptr, sb, q8, stream);
        else
            launch_fast<8, false, false, 3, false, true>(q, s0, s1, h, sq, b, sl2, out, f32out, km, nullptr, sb, q8, stream);
    } else if (exact && nw == 4) {
        launch_fast<4, false, false, 3>(q, s0, s1, h, sq, b, sl2, out, f32out, km, nullptr, sb, q8, stream);
    } else if (exact) {
        launch_fast<8, false, false, 3>(q, s0, s1, h, sq, b, sl2, out, f32out, km, nullptr, sb, q8, stream);
    } else if (pair && !round_later) {
        launch_fast<8, true, false, 0, true>(q, s0, s1, h, sq, b, sl2, out, outf, km, nullptr, sb, 0, stream);
        rounded = true;
    } else if (nw == 4) {
        launch_fast<4, PRE, false, SM>(q, s0, s1, h, sq, b, sl2, out, f32out, km, nullptr, sb, q8, stream);
    } else {
        launch_fast<8, PRE, false, SM>(q, s0, s1, h, sq, b, sl2, out, f32out, km, nullptr, sb, q8, stream);
    }
    return finish_q8k(out_qblk, rounded, outf, b, h, sq, out, stream);
}

}  // namespace

size_t attention_scratch_bytes(int64_t bh, int64_t sq) {
    // what any split of up to this many tiles can take (MAX_PARTS per tile, two
    // parts per CU): it grows with the tiles, so that scratch reserved for a size
    // serves every smaller one
    const int64_t cus = device_cu_count(), tiles = (sq + 255) / 256 * bh;
    return (size_t)std::min<int64_t>(MAX_PARTS * tiles, 2 * std::max<int64_t>(cus, 0)) * 256 * (128 + 2) * 4;
}

hipError_t launch_attention(const uint16_t *q, KeySeg prefix, KeySeg own, int64_t b, int64_t h, int64_t sq,
                            float scale, uint16_t *out, hipStream_t stream, float *outf) {
    return launch<false>(q, prefix, own, b, h, sq, scale * 1.4426950408889634f, out, outf,
                         ScoreBound{nullptr, 0.f, 0.f}, 0, stream);
}

hipError_t launch_attention_masked(const uint16_t *q, KeySeg prefix, KeySeg own, int64_t b, int64_t h, int64_t sq,
                                   float sl2, const int32_t *img, const uint8_t *kvalid, int32_t *lim_scratch,
                                   uint16_t *out, hipStream_t stream, float *outf, const float *k_prefix_norm,
                                   float q_norm, float k_own_norm, int out_qblk, float *scratch, bool round_later) {
    if (sq <= 0 || b <= 0 || h <= 0) return hipSuccess;
    Seg s0, s1;
    if (!segments(prefix, own, s0, s1) || !out_qblk_ok(out_qblk, outf)) return hipErrorInvalidValue;
    const int out_q8 = out_qblk == 32 && !round_later;
    if (out_q8) outf = nullptr;
    if (img && (prefix.len != 0 || own.len != sq)) return hipErrorInvalidValue;  // block-causal: one shared sequence
    const KeyMask km{img, kvalid, prefix.len + own.len};
    // the last visible key of each query (none known: every window is classified)
    const int32_t *lim = nullptr;
    if (img && lim_scratch && sq <= LIMIT_MAX_S) {
        key_limit_kernel<<<dim3(1), dim3(1024), 0, stream>>>(img, (int)sq, lim_scratch);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        lim = lim_scratch;
    }
    // the bound is on scores in log2 units: q's norm times sl2
    const ScoreBound sb{prefix.len > 0 ? k_prefix_norm : nullptr, q_norm * sl2, k_own_norm};
    const bool exact = exact_softmax(prefix, own, img && !lim);
    if (!rows16(s0) || !rows16(s1))
        launch_fast<8, false, true, 3, false, true>(q, s0, s1, h, sq, b, sl2, out, outf, km, lim, sb, out_q8, stream);
    else if (exact || sl2 == 1.0f) {  // 1: q already carries the scale (the block's q/k/v epilogue)
        KeySplit sp{0, 1, nullptr, nullptr};
        if (scratch) {
            const int64_t cus = std::max(device_cu_count(), 1), n8 = (sq + 255) / 256 * b * h;
            const double now = tile_rounds_us(b * h, sq, km.kv_len, true, (double)((n8 + cus - 1) / cus));
            if (const int parts = split_parts(b * h, sq, km.kv_len, true, now, 0.0); parts > 1)
                sp = key_split(b * h, sq, parts, scratch);
        }
        if (exact)
            launch_fast<8, false, true, 3>(q, s0, s1, h, sq, b, sl2, out, outf, km, lim, sb, out_q8, stream, sp);
        else
            launch_masked<true>(q, s0, s1, h, sq, b, sl2, out, outf, km, lim, sb, out_q8, stream, sp);
    } else
        launch_masked<false>(q, s0, s1, h, sq, b, sl2, out, outf, km, lim, sb, out_q8, stream,
                             KeySplit{0, 1, nullptr, nullptr});
    return finish_q8k(out_qblk, round_later, outf, b, h, sq, out, stream);
}

hipError_t launch_attention_log2(const uint16_t *q, KeySeg prefix, KeySeg own, int64_t b, int64_t h, int64_t sq,
                                 uint16_t *out, hipStream_t stream, float *outf, const float *k_prefix_norm,
                                 float q_norm, float k_own_norm, int out_qblk, float *scratch, bool round_later) {
    return launch<true>(q, prefix, own, b, h, sq, 1.0f, out, outf,
                        ScoreBound{prefix.len > 0 ? k_prefix_norm : nullptr, q_norm, k_own_norm}, out_qblk, stream, scratch, round_later);
}

}  // namespace qimm
