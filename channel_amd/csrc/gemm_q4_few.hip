// Batched contractions over Q4 weights for few tokens (a short message, the
// tail of a prompt): gemm_q4.hip's contractions (shaders/batch_gemm_q4.wgsl,
// shaders/batch_fused_mlp_q4.wgsl) where few_tokens holds.
//
// What bounds them: reading the weights (gate/up at 12B dims: 66 MB against
// 8.5 GFLOP at 24 tokens), then turning them into bf16 (21 VALU operations
// per 8 weights, ~8 us of the chip's VALU for gate/up).  The 64- and 128-token
// tiles of gemm_q4.hip take about as long for 8 tokens as for 128, each walking
// its K behind a barrier per slab.  Here weights go from memory to registers in
// the order an MFMA operand holds them, and activations too, with no LDS and no
// barrier before the end:
//  * v_mfma_f32_16x16x32_bf16 with the weights as A (16 features) and the
//    tokens as B.  Lane (r, g) = (lane & 15, lane >> 4) loads whole 32-weight
//    blocks of row r; word j of the block it holds is its A operand of one
//    MFMA (8 codes), so which K an MFMA step covers is a fixed permutation,
//    and the activations are stored in that order (xb_at in chn_internal.h)
//    by the kernel that makes them.
//  * A step covers 256 K: lane (r, g) takes blocks 2g and 2g + 1, so every
//    weight load of a wave asks for 16 whole 128-byte lines.  (Blocks g and
//    4 + g, half lines per load: 28.0 against 23.5 us for gate/up at 8
//    tokens; non-temporal loads of half lines, each line fetched twice: 31.)
//  * What is left to bound it is instruction issue: a wave issues a VALU
//    operation every 8 cycles at most, two waves of a SIMD one every 4.7, and
//    waves wait to issue 46 % of their time, for memory 19 %.  Loads count
//    too: the scales of a lane's two blocks (Q4R) come in one 4-byte load
//    (two 2-byte loads: gate/up at 24 tokens 27.4 against 25.9 us a call, at
//    64 tokens 43.2 against 40.8; down at 24 tokens 25.8 against 24.9).
//  * The waves of a workgroup share its feature tiles and take every
//    WK-th step, so together they read the rows front to back; their sums
//    meet in LDS in wave order (results do not depend on timing).
//  * Activations are read as operand fragments of one contiguous KB from the
//    cache.  (Row-major activations, 16 rows by 64 bytes per load: 38 against
//    30 us for gate/up at 24 tokens, 33 against 19 us for down.)
// Two feature tiles per matrix and 4 waves where that gives about a workgroup
// per CU, else one tile and 8 waves: gate/up 15360 x 3840 at 24 tokens 26.0
// against 31.1 us with one tile; down 3840 x 15360 17.6 against 24.8 us with
// two.
// Measured at 12B dims, weights from HBM, before (tiles of 128 or 256 tokens
// that took weights through LDS) and now, us, 8 / 32 / 64 tokens: gate/up 111 ->
// 23, 113 -> 26, 118 -> 38; down 55 -> 14, 56 -> 18, 57 -> 26; q/k/v 29 -> 8, 30 ->
// 9, 31 -> 12 (128 tokens 31 -> 20); o_proj 18 -> 6, 19 -> 7, 19 -> 9.
#include "chn_internal.h"

namespace chn {

typedef __bf16 fbf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 fbf16x2 __attribute__((ext_vector_type(2)));
typedef float ff32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t fu32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));

struct FewArgs {
    const __bf16 *X;                   // activations in xb_at order, ntt token tiles
    const unsigned char *W[3], *W1;    // one matrix per segment; W1: the up matrix
    float *Y[3];                       // [n_tok][M[s]]
    __bf16 *Yb;                        // != NULL: the result as bf16 instead of Y[0], in xb_at order for yb_ntt
    uint32_t M[3], g0[3];              // rows and first feature group of each segment
    uint32_t n_tok, K, ntt, ntg, ngrp, yb_ntt; // tokens' tiles, groups of NT of those, feature groups
};

// Eight codes of one nibble word to bf16(scale * (q - 8)): `q` in two's
// complement (q - 8), s16 = 16 * scale; v_cvt_off_f32_i4 gives (q - 8) / 16,
// so the product is exact before its one rounding, as in gemm_q4.hip.
__device__ __forceinline__ fbf16x8 few_dequant(uint32_t q, float s16) {
    uint32_t h = q >> 4;
    __asm__("" : "+v"(h));              // one shift for the four high nibbles, byte selects for the rest
    fu32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const fbf16x2 p = {(__bf16)(__builtin_amdgcn_cvt_off_f32_i4((int)((q >> (8 * j)) & 0xffu)) * s16),
                           (__bf16)(__builtin_amdgcn_cvt_off_f32_i4((int)((h >> (8 * j)) & 0xffu)) * s16)};
        o[j] = __builtin_bit_cast(uint32_t, p);
    }
    return __builtin_bit_cast(fbf16x8, o);
}

template <int NMAT, int FT, int NT, bool REP, int WK>
__global__ __launch_bounds__(64 * WK) void k_q4gemm_few(FewArgs a) {
    constexpr int NF = NMAT * FT;                      // feature tiles of a wave
    __shared__ ff32x4 red[WK][NF * NT][64];

    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t wk = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r = lane & 15, g = lane >> 4;
    // work items: feature groups in runs of 8, the token groups of a run
    // next, so that the token groups of one feature group run on one XCD
    // (workgroup i runs on XCD i % 8) and share its L2's weights
    const uint32_t run = blockIdx.x / (8 * a.ntg), rem = blockIdx.x % (8 * a.ntg);
    uint32_t grp = run * 8 + rem % 8;
    const uint32_t tt0 = rem / 8 * NT;
    if (grp >= a.ngrp) return;                         // uniform, before any barrier
    const int sg = (grp >= a.g0[1] ? 1 : 0) + (grp >= a.g0[2] ? 1 : 0);
    const unsigned char *W0 = sg == 0 ? a.W[0] : (sg == 1 ? a.W[1] : a.W[2]);
    const uint32_t M = sg == 0 ? a.M[0] : (sg == 1 ? a.M[1] : a.M[2]);
    float *Y = sg == 0 ? a.Y[0] : (sg == 1 ? a.Y[1] : a.Y[2]);
    grp -= sg == 0 ? 0u : (sg == 1 ? a.g0[1] : a.g0[2]);
    const uint32_t n0 = grp * (16 * FT);
    const uint32_t nb = a.K / 32, nstep = (nb + 7) / 8;
    // this wave's steps: wk, wk + WK, ...
    const uint32_t cnt = wk < nstep ? (nstep - wk + WK - 1) / WK : 0;
    const uint32_t last = cnt ? wk + (cnt - 1) * WK : 0;

    const unsigned char *wq[NF], *ws[NF];              // this lane's row (clamped: rows past M are not stored)
#pragma unroll
    for (int m = 0; m < NMAT; ++m)
#pragma unroll
        for (int f = 0; f < FT; ++f) {
            const uint32_t n = min(n0 + f * 16 + r, M - 1);
            const unsigned char *W = m == 0 ? W0 : a.W1;
            wq[m * FT + f] = W + (size_t)n * nb * (REP ? 16 : 20);
            ws[m * FT + f] = W + (size_t)M * nb * 16 + (size_t)n * nb * 2;
        }
    const __bf16 *xf = a.X + lane * 8;

    struct Wstep {
        fu32x4 q[NF][2];
        uint32_t s[NF][REP ? 1 : 2];                   // REP: the two blocks' scales in one word
    };
    struct Xhalf {
        fu32x4 x[NT][4];
    };
    // Loads are unconditional: a step past the wave's last reloads that one
    // (from cache), a block past the row's end its last block.
    auto step = [&](uint32_t i) { return min(wk + i * WK, last); };
    auto load_w = [&](uint32_t i, Wstep &w) {
        const uint32_t b0 = 8 * step(i) + 2 * g;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            // the scales of blocks b0 and b0 + 1, or of the row's last two
            // (the word before a row's scales is readable: codes or scales)
            if (REP) w.s[f][0] = *(const u32_a2 *)(ws[f] + (ptrdiff_t)min((int)b0, (int)nb - 2) * 2);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const size_t b = min(b0 + h, nb - 1);
                if (REP) {
                    w.q[f][h] = *(const fu32x4 *)(wq[f] + b * 16);
                } else {
                    const uint32_t *p = (const uint32_t *)(wq[f] + b * 20);
                    const u32x4_a4 v = *(const u32x4_a4 *)(p + 1);
                    w.s[f][h] = p[0];
                    w.q[f][h] = fu32x4{v[0], v[1], v[2], v[3]};
                }
            }
        }
    };
    auto load_x = [&](uint32_t i, int h, Xhalf &x) {
        const __bf16 *p = xf + ((size_t)step(i) * 2 + h) * a.ntt * 2048;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) x.x[t][j] = *(const fu32x4 *)(p + (min(tt0 + t, a.ntt - 1) * 4 + j) * 512);
    };
    ff32x4 acc[NF][NT];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[f][t] = ff32x4{0, 0, 0, 0};
    const bool ragged = (nb & 7) != 0;                 // the last step has blocks past the row's end
    auto compute = [&](uint32_t i, int h, const Wstep &w, Xhalf &x) {
        uint32_t ok = 0xffffffffu, sh = 16 * h;
        if (ragged) {                                  // those contribute exact zeros on both sides
            ok = opaque_mask(8 * step(i) + 2 * g + h < nb);
            if (8 * step(i) + 2 * g + 1 >= nb) sh = 16;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) x.x[t][j] &= ok;
        }
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            const float s16 = 16.0f * f16_lo_to_f32((REP ? w.s[f][0] >> sh : w.s[f][h]) & ok);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const fbf16x8 d = few_dequant(REP ? w.q[f][h][j] : w.q[f][h][j] ^ 0x88888888u, s16);
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[f][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d, __builtin_bit_cast(fbf16x8, x.x[t][j]),
                                                                        acc[f][t], 0, 0, 0);
            }
        }
    };

    if (cnt) {
        Xhalf x0, x1;
        Wstep w;
        load_x(0, 0, x0);
        load_w(0, w);
        load_x(0, 1, x1);
        for (uint32_t i = 0; i < cnt; ++i) {
            compute(i, 0, w, x0);
            load_x(i + 1, 0, x0);
            compute(i, 1, w, x1);
            load_w(i + 1, w);
            load_x(i + 1, 1, x1);
        }
    }
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int t = 0; t < NT; ++t) red[wk][f * NT + t][lane] = acc[f][t];
    __syncthreads();
    // unit (tile ft = f * NT + t, lane l): features n0 + 16 f + 4 (l >> 4) +
    // 0..3 of token 16 (tt0 + t) + (l & 15)
    for (int u = tid; u < FT * NT * 64; u += 64 * WK) {
        const int l = u & 63, ft = u >> 6;
        ff32x4 v = red[0][ft][l];
#pragma unroll
        for (int k = 1; k < WK; ++k) v += red[k][ft][l];
        if (NMAT == 2) {
            ff32x4 up = red[0][(NF - FT) * NT + ft][l];
#pragma unroll
            for (int k = 1; k < WK; ++k) up += red[k][(NF - FT) * NT + ft][l];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = gelu_tanh(v[i]) * up[i];
        }
        const uint32_t t = (tt0 + ft % NT) * 16 + (l & 15), n = n0 + (ft / NT) * 16 + 4 * (l >> 4);
        if (t >= a.n_tok) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n + i < M) {
                if (a.Yb) a.Yb[xb_at(a.yb_ntt, M, t, n + i)] = (__bf16)v[i];
                else Y[(size_t)t * M + n + i] = v[i];
            }
    }
}

// fp32 rows to bf16 (RNE) in xb_at order, four values per thread.
__global__ __launch_bounds__(256) void k_to_bf16_few(const float *__restrict__ x, __bf16 *__restrict__ y,
                                                     uint32_t n_tok, uint32_t K, uint32_t ntt) {
    const uint32_t k = (blockIdx.x * 256 + threadIdx.x) * 4, t = blockIdx.y;
    if (k >= K) return;
    const float4 v = *(const float4 *)(x + (size_t)t * K + k);
    __bf16 *o = y + xb_at(ntt, K, t, k);
    *(fbf16x2 *)o = fbf16x2{(__bf16)v.x, (__bf16)v.y};
    *(fbf16x2 *)(o + 2) = fbf16x2{(__bf16)v.z, (__bf16)v.w};
}

void launch_to_bf16_few(hipStream_t st, const float *X, __bf16 *xb, uint32_t n_tok, uint32_t K) {
    k_to_bf16_few<<<dim3((K / 4 + 255) / 256, n_tok), 256, 0, st>>>(X, xb, n_tok, K, xb_tiles(n_tok));
}

template <int NMAT, int FT, bool REP, int WK>
static void launch_few_nt(hipStream_t st, FewArgs &a) {
    // token groups of at most 4 tiles, evenly filled (5 tiles: 3 + 2)
    a.ntg = (a.ntt + 3) / 4;
    const uint32_t nt = (a.ntt + a.ntg - 1) / a.ntg;
    const unsigned grid = (a.ngrp + 7) / 8 * 8 * a.ntg;
    switch (nt) {
    case 1: k_q4gemm_few<NMAT, FT, 1, REP, WK><<<grid, 64 * WK, 0, st>>>(a); break;
    case 2: k_q4gemm_few<NMAT, FT, 2, REP, WK><<<grid, 64 * WK, 0, st>>>(a); break;
    case 3: k_q4gemm_few<NMAT, FT, 3, REP, WK><<<grid, 64 * WK, 0, st>>>(a); break;
    default: k_q4gemm_few<NMAT, FT, 4, REP, WK><<<grid, 64 * WK, 0, st>>>(a); break;
    }
}

template <int NMAT, bool REP>
static void launch_few_shape(hipStream_t st, FewArgs &a, int nseg) {
    uint32_t rows = 0;
    for (int s = 0; s < nseg; ++s) rows += a.M[s];
    const uint32_t per = few_features(rows);
    uint32_t g = 0;
    for (int s = 0; s < 3; ++s) {
        a.g0[s] = s < nseg ? g : 0xffffffffu;
        if (s < nseg) g += (a.M[s] + per - 1) / per;
    }
    a.ngrp = g;
    if (per == 32) launch_few_nt<NMAT, 2, REP, 4>(st, a);
    else launch_few_nt<NMAT, 1, REP, 8>(st, a);
}

void launch_q4gemm_few(hipStream_t st, int nmat, int nseg, const uint32_t *const *W, const uint32_t *W1,
                       float *const *Y, const uint32_t *M, uint32_t n_tok, uint32_t K, const __bf16 *xb, bool repacked,
                       __bf16 *Yb, uint32_t yb_ntt) {
    FewArgs a{};
    a.X = xb;
    for (int s = 0; s < nseg; ++s) {
        a.W[s] = (const unsigned char *)W[s];
        a.Y[s] = Y[s];
        a.M[s] = M[s];
    }
    a.W1 = (const unsigned char *)W1;
    a.Yb = Yb;
    a.n_tok = n_tok;
    a.K = K;
    a.ntt = xb_tiles(n_tok);
    a.yb_ntt = yb_ntt;
    if (nmat == 2) {
        if (repacked) launch_few_shape<2, true>(st, a, nseg);
        else launch_few_shape<2, false>(st, a, nseg);
    } else {
        if (repacked) launch_few_shape<1, true>(st, a, nseg);
        else launch_few_shape<1, false>(st, a, nseg);
    }
}

}  // namespace chn
