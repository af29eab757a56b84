// Batched prefill contractions over Q4 weights on gfx950 MFMA:
// batch_gemm_q4 (shaders/batch_gemm_q4.wgsl) and batch_fused_mlp_q4
// (shaders/batch_fused_mlp_q4.wgsl), for more tokens than gemm_q4_few.hip
// serves (few_tokens).
//
//   Y[t, n] = sum_k X[t, k] * W[n, k]        (t < n_tok, n < M)
//
// v_mfma_f32_16x16x32_bf16 with the weights as A (16 features) and the
// tokens as B; activations are rounded to bf16 (RNE) once, by their producer
// or a pre-pass, weights to bf16(scale * (q - 8)); fp32 accumulation.
#include "chn_internal.h"

namespace chn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

// Activations to bf16 (RNE).
__global__ __launch_bounds__(256) void k_to_bf16(const float *__restrict__ x, __bf16 *__restrict__ y, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x * 4;
    for (size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4; i < n; i += stride) {
        const float4 v = *(const float4 *)(x + i);     // (K % 32 == 0, so n % 4 == 0)
        *(bf16x4 *)(y + i) = bf16x4{(__bf16)v.x, (__bf16)v.y, (__bf16)v.z, (__bf16)v.w};
    }
}

// y = the sum of np partial outputs p + i * n, in index order.
__global__ __launch_bounds__(256) void k_sum_parts(const float *__restrict__ p, float *__restrict__ y, size_t n,
                                                   uint32_t np) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    if (i + 4 <= n && n % 4 == 0 && ((uintptr_t)y & 15) == 0) {
        f32x4 v = *(const f32x4 *)(p + i);
        for (uint32_t k = 1; k < np; ++k) v += *(const f32x4 *)(p + k * n + i);
        *(f32x4 *)(y + i) = v;
    } else {
        for (size_t j = i; j < n && j < i + 4; ++j) {
            float v = p[j];
            for (uint32_t k = 1; k < np; ++k) v += p[k * n + j];
            y[j] = v;
        }
    }
}

struct GemmArgs {
    const __bf16 *X;                   // [n_tok][K]
    const unsigned char *W[3], *W1;    // Q4 or Q4R, one matrix per segment; W1: the up matrix
    float *Y[3];                       // [n_tok][M[s]]
    __bf16 *Yb;                        // != NULL: the result as bf16 instead of Y[0], in xb_at order for yb_ntt
    uint32_t M[3], c0[3];              // rows and first column tile of each segment
    uint32_t n_tok, K, n_ct, n_tt, yb_ntt;
    // Split K: ksplit workgroups per tile, split p stores its sums to Y + p *
    // ypart; the consumer (or k_sum_parts) adds them.
    uint32_t ksplit;
    size_t ypart;
};

__device__ __attribute__((aligned(16))) const uint32_t g_zero16[4] = {0, 0, 0, 0};

// Barrier of the four waves that share the LDS counter n: the wave's last LDS
// reads and its DMA are done (the caller waited), lane 0 counts it in, and it
// goes on once the count has reached `target`.  The four waves are in one
// workgroup, so all of them run, and each counts itself in before it waits.
// With s_barrier the two groups of a G 2 workgroup wait for each other at
// every slab: q/k/v at 300 tokens 39.1 against 37.2 us, at 512 42.9 against 42.5;
// o_proj at 300 tokens 31.0 against 30.2, at 700 42.7 against 40.8.
__device__ __forceinline__ void group_barrier(uint32_t *n, uint32_t target, int lane) {
    __asm__ volatile("" ::: "memory");
    if (lane == 0) __hip_atomic_fetch_add(n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while ((int32_t)(__builtin_amdgcn_readfirstlane(
                         __hip_atomic_load(n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) -
                     target) < 0) {
    }
    __asm__ volatile("" ::: "memory");
}

// The contraction of one tile: 128 tokens x 64 FT / NMAT features per
// matrix, four waves (times G) of all 128 tokens x FT feature tiles of 16.
//
// K is walked in slabs of 128 (four 32-blocks).  X's slab (32 KB of bf16
// rows, 16-byte chunks XOR-swizzled by row so that fragment reads meet no
// bank conflict) travels by DMA (global_load_lds) into one of two LDS slots,
// one slab ahead.  Weights never touch LDS: lane (r, g) = (lane & 15, lane
// >> 4) loads block g of the slab from row r of each of its tiles, and word j
// of that block, turned into 8 bf16, is its A operand of the MFMAs of K group
// j, so a wave dequantizes exactly what it multiplies; the next word's
// dequantization (21 VALU operations per 8 weights: v_cvt_off_f32_i4 gives
// (q - 8) / 16, times 16 * scale is exact before its one rounding) is spread
// between the current word's MFMAs.  X fragments are read three ahead.  A
// slab has one barrier, passed when its last fragments have been read: from
// then on its slot takes the DMA of the slab after next.
//
// What bounds it: the card's power.  With two workgroups per CU the matrix
// pipe is 65 (FT 2) to 77 % (FT 4) busy while the clock falls from 2.4 to 1.7
// and 2.05 GHz; a large bf16 product of the vendor library, without
// dequantization, reaches 1.14-1.2 PFLOP/s here.  So what counts is bytes
// and operations per MFMA: the kernels this replaces moved each weight
// through LDS as codes and as bf16 (0.66-0.92 PFLOP/s on the same shapes).
// One workgroup per CU leaves the pipe 37-40 % busy (a wave's own VALU and
// LDS waits are not hidden by its MFMAs), so a shape with few tiles takes
// two waves per SIMD another way: G 2 walks two halves of K in eight waves
// whose sums meet in LDS, ksplit does so in separate workgroups.
//
// Calls at 12B dims with their bf16 pass, before and now, us: 512 x 3840 ->
// 15360 89 / 72; q/k/v 300 tokens 64 / 37, 512 tokens 51 / 43; gate/up 256
// tokens 120 / 70, 512 tokens 126 / 124; down 512 tokens 98 / 81, 1024 tokens
// 191 / 144; o_proj 512 tokens 40 / 33, 1024 tokens 74 / 47.
//
// RAG: K % 128 != 0, the last slab's missing blocks contribute exact zeros.
template <int NMAT, int BT, int FT, int G, bool REP, bool RAG>
__device__ __forceinline__ void gemm_tile(const GemmArgs &a) {
    constexpr int NTT = BT / 16, NF = FT / NMAT, BN = 64 * NF, NST = 4 * NTT, NU = FT * 4;
    constexpr int SLOT = BT * 256, RING = 4, LA = RING - 1;
    constexpr bool kAtOnce = NMAT == 2 && FT == 4 && REP;
    __shared__ __attribute__((aligned(16))) unsigned char sm[2 * G * SLOT];
    __shared__ uint32_t arrived[2];                            // G 2: waves of a group that passed a slab, counted up
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;
    const uint32_t grp = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
    const uint32_t r = lane & 15, g = lane >> 4;
    // work items (split, column tile, token tile), token tile fastest, dealt
    // to the XCDs in contiguous runs (workgroup i runs on XCD i % 8), so the
    // token tiles of a feature block share one L2's weights
    const uint32_t nwork = a.n_ct * a.n_tt * a.ksplit, per = (nwork + 7) / 8;
    const uint32_t work = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (work >= nwork) return;                             // uniform, before any barrier
    const uint32_t tt = work % a.n_tt, rest = work / a.n_tt, ks = rest / a.n_ct;
    uint32_t ct = rest % a.n_ct;
    const int sg = (ct >= a.c0[1] ? 1 : 0) + (ct >= a.c0[2] ? 1 : 0);
    const unsigned char *W0 = sg == 0 ? a.W[0] : (sg == 1 ? a.W[1] : a.W[2]);
    const uint32_t M = sg == 0 ? a.M[0] : (sg == 1 ? a.M[1] : a.M[2]);
    float *Y = sg == 0 ? a.Y[0] : (sg == 1 ? a.Y[1] : a.Y[2]);
    ct -= sg == 0 ? 0u : (sg == 1 ? a.c0[1] : a.c0[2]);
    const uint32_t n0 = ct * BN + wave * (16 * NF), t0 = tt * BT;
    const uint32_t K = a.K, nb = K / 32, S = (nb + 3) / 4;
    // this group's slabs [s0, s1) of the workgroup's share of K
    const uint32_t ntot = a.ksplit * G, part = ks * G + grp;
    const uint32_t s0 = part * S / ntot, s1 = (part + 1) * S / ntot;
    unsigned char *xs = sm + grp * 2 * SLOT;

    // X: instruction i of wave w copies rows 16 i + 4 w .. + 3 of the slab, chunk
    // c of row t to position c ^ (t & 15).  Rows past the last token (their
    // columns are not stored) are clamped: the tile's last group of 16 rows with a
    // token in it, group gl, has lane offsets of its own, and the groups after it
    // copy it again.  A group's offset is scalar (64 bits: K may be any width), so
    // the addresses take two registers.  With an offset per group three of the four
    // FT 4 kernels spilled 10 to 16 registers in the K loop, each reload a wait for
    // the DMA issued before it: one matrix 15360 x 3840 at 1024 tokens 133 (Q4R) and
    // 159 us (Q4) against 123 and 129, gate/up on Q4 at 512 tokens 148 against 129.
    const uint32_t xrow = 4 * wave + (lane >> 4), chunk = (lane & 15) ^ (xrow & 15);
    const __bf16 *Xt = a.X + (size_t)t0 * K;
    const uint32_t rlim = a.n_tok - 1 - t0, gl = rlim / 16;
    const uint32_t xo = (xrow * K + chunk * 8) * 2, xol = (min(xrow, rlim - 16 * gl) * K + chunk * 8) * 2;
    auto issue_x = [&](uint32_t s, uint32_t slot) {            // slot: byte offset
        const unsigned char *Xs = (const unsigned char *)(Xt + (size_t)s * 128);
        const bool zero = RAG && s * 128 + chunk * 8 >= K;     // past the row's end (K % 128 != 0)
        uint32_t g1 = gl;
        if (FT == 4) __asm__ volatile("" : "+s"(g1));          // select per slab: hoisted, the offsets would stay live
#pragma unroll
        for (int i = 0; i < NTT; ++i) {
            const unsigned char *Xg = Xs + (size_t)min((uint32_t)i, g1) * 32 * K;
            __builtin_amdgcn_global_load_lds(zero ? (const unsigned char *)g_zero16 : Xg + ((uint32_t)i < g1 ? xo : xol),
                                             (lds_t *)(xs + slot + (wave + 4 * i) * 1024), 16, 0, 0);
        }
    };
    struct Raw {
        u32x4v q[FT];
        uint32_t s[FT];
    };
    // weight rows relative to the wave's first one (their bytes fit 32 bits);
    // rows past M are clamped and not stored
    const unsigned char *Wb[NMAT], *Sb[NMAT];
#pragma unroll
    for (int m = 0; m < NMAT; ++m) {
        const unsigned char *W = m == 0 ? W0 : a.W1;
        const uint32_t nr = min(n0, M - 1);
        Wb[m] = W + (size_t)nr * nb * (REP ? 16 : 20);
        Sb[m] = W + (size_t)M * nb * 16 + (size_t)nr * nb * 2;
    }
    const uint32_t nlim = M - 1 - min(n0, M - 1);
    const uint32_t wgl = __builtin_amdgcn_readfirstlane(nlim / 16), wr = r * nb, wrl = min(r, nlim - 16 * wgl) * nb;
    auto load_raw = [&](uint32_t s, Raw &w, int f) {
        const uint32_t b = RAG ? min(4 * s + g, nb - 1) : 4 * s + g;
        uint32_t o;
        if (NF == 4) {                                         // as X's rows: two lane offsets for the four tiles
            uint32_t g1 = wgl;
            __asm__ volatile("" : "+s"(g1));
            o = min((uint32_t)(f % NF), g1) * 16 * nb + ((uint32_t)(f % NF) < g1 ? wr : wrl) + b;
        } else {
            o = min(f % NF * 16 + r, nlim) * nb + b;
        }
        if (REP) {
            w.q[f] = *(const u32x4v *)(Wb[f / NF] + o * 16);
            w.s[f] = *(const uint16_t *)(Sb[f / NF] + o * 2);
        } else {
            const uint32_t *p = (const uint32_t *)(Wb[f / NF] + o * 20);
            const u32x4_a4 v = *(const u32x4_a4 *)(p + 1);
            w.s[f] = p[0];
            w.q[f] = u32x4v{v[0], v[1], v[2], v[3]};
        }
    };
    float sc[FT];
    uint32_t hi[FT];
    auto unit = [&](const u32x4v &q, int j, int f, int p, u32x4v &d) {   // pair p of word j of tile f
        const uint32_t w = REP ? q[j] : q[j] ^ 0x88888888u;
        if (p == 0) {
            hi[f] = w >> 4;
            __asm__("" : "+v"(hi[f]));
        }
        const bf16x2 v = {(__bf16)(__builtin_amdgcn_cvt_off_f32_i4((int)((w >> (8 * p)) & 0xffu)) * sc[f]),
                          (__bf16)(__builtin_amdgcn_cvt_off_f32_i4((int)((hi[f] >> (8 * p)) & 0xffu)) * sc[f])};
        d[p] = __builtin_bit_cast(uint32_t, v);
    };
    auto scale = [&](uint32_t s, const Raw &w, int f) {
        sc[f] = 16.0f * f16_lo_to_f32(w.s[f]);
        if (RAG) sc[f] = mask_f(sc[f], opaque_mask(4 * s + g < nb));
    };
    const uint32_t smb = lds_addr(xs);
    uint32_t xb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) xb[j] = smb + r * 256 + (((4 * g + j) ^ r) & 15) * 16;

    f32x4 acc[FT][NTT];
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int t = 0; t < NTT; ++t) acc[f][t] = f32x4{0, 0, 0, 0};
    u32x4v A[2][FT];
    bf16x8 xf[RING];
    Raw rc, rn;
    if (G == 2 && tid < 2) arrived[tid] = 0;
    issue_x(min(s0, S - 1), 0);
#pragma unroll
    for (int f = 0; f < FT; ++f) load_raw(min(s0, S - 1), rc, f);
    wait_vm_lgkm0<0>();
    bare_barrier();
    if (s0 + 1 < s1) issue_x(s0 + 1, SLOT);
    static_for<LA>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        xf[i] = lds_read<bf16x8, (i % NTT) * 4096>(xb[i / NTT]);
    });
    lds_wait();                                                // no read in flight into the loop
    static_for<LA>([&](auto i_) { lds_pin(xf[decltype(i_)::value]); });
#pragma unroll
    for (int f = 0; f < FT; ++f) {
        scale(s0, rc, f);
#pragma unroll
        for (int p = 0; p < 4; ++p) unit(rc.q[f], 0, f, p, A[0][f]);
    }
    uint32_t slot = 0;                                         // byte offset of slab s's X
    for (uint32_t s = s0; s < s1; ++s) {
        const uint32_t sn = min(s + 1, S - 1);
        static_for<NST>([&](auto i_) {
            constexpr int i = decltype(i_)::value, j = i / NTT, t = i % NTT;
            if constexpr (i == NST - LA) {                     // slab s's last fragments are read
                wait_vm_lgkm0<0>();                            // ... and slab s + 1's DMA landed
                if constexpr (G == 2) group_barrier(&arrived[grp], 4 * (s - s0 + 1), lane);
                else bare_barrier();                           // ... for every wave of the group
                if (s + 2 < s1) issue_x(s + 2, slot);
                slot ^= SLOT;
#pragma unroll
                for (int k = 0; k < 4; ++k) xb[k] ^= SLOT;
            }
            // the next slab's weights, used from word group 3 on: spread, or at
            // once where the addresses still fit the registers (gate/up 121
            // against 123 us)
            if constexpr (kAtOnce && i == 0) {
#pragma unroll
                for (int f = 0; f < FT; ++f) load_raw(sn, rn, f);
            }
            if constexpr (!kAtOnce && i % 2 == 0 && i / 2 < FT) load_raw(sn, rn, i / 2);
            constexpr int ia = (i + LA) % NST;
            xf[(i + LA) % RING] = lds_read<bf16x8, (ia % NTT) * 4096>(xb[ia / NTT]);
            lds_wait_n<LA>();
            lds_pin(xf[i % RING]);
            static_for<FT>([&](auto f_) {
                constexpr int f = decltype(f_)::value;
                acc[f][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, A[j & 1][f]),
                                                                    xf[i % RING], acc[f][t], 0, 0, 0);
            });
            constexpr int u0 = t * NU / NTT, u1 = (t + 1) * NU / NTT;
            static_for<u1 - u0>([&](auto u_) {
                constexpr int u = u0 + decltype(u_)::value, f = u / 4, p = u % 4;
                if constexpr (j == 3 && p == 0) scale(s + 1, rn, f);
                unit(j < 3 ? rc.q[f] : rn.q[f], (j + 1) & 3, f, p, A[(j + 1) & 1][f]);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
#pragma unroll
        for (int f = 0; f < FT; ++f) rc.q[f] = rn.q[f];
    }
    lds_wait();
#pragma unroll
    for (int i = 0; i < RING; ++i) lds_pin(xf[i]);

    if constexpr (G == 2) {                                    // the two groups' sums meet in LDS
        wait_vm_lgkm0<0>();
        bare_barrier();
        f32x4 *red = (f32x4 *)sm + wave * (FT * NTT * 64) + lane;
        if (grp == 1)
#pragma unroll
            for (int f = 0; f < FT; ++f)
#pragma unroll
                for (int t = 0; t < NTT; ++t) red[(f * NTT + t) * 64] = acc[f][t];
        __syncthreads();
        if (grp == 1) return;
#pragma unroll
        for (int f = 0; f < FT; ++f)
#pragma unroll
            for (int t = 0; t < NTT; ++t) acc[f][t] += red[(f * NTT + t) * 64];
    }
    // epilogue: lane holds features 4g + i of each tile, token r
    float *Yp = Y + ks * a.ypart;
    const bool vec = M % 4 == 0 && ((uintptr_t)a.Yb & 7) == 0;
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int t = 0; t < NTT; ++t) {
            const uint32_t tok = t0 + 16 * t + r, n = n0 + 16 * f + 4 * g;
            f32x4 v = acc[f][t];
            if (NMAT == 2)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = gelu_tanh(v[i]) * acc[(NMAT - 1) * NF + f][t][i];
            if (tok >= a.n_tok || n >= M) continue;
            if (a.Yb) {
                __bf16 *y = a.Yb + xb_at(a.yb_ntt, M, tok, n);     // (four k of a token lie together)
                if (vec) {
                    *(bf16x4 *)y = bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (n + i < M) y[i] = (__bf16)v[i];
                }
                continue;
            }
            float *y = Yp + (size_t)tok * M + n;                   // (4-byte alignment is enough)
            if (n + 4 <= M) {
                *(f32x4_a4 *)y = v;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < M) y[i] = v[i];
            }
        }
}

// Two matrices (gate/up + GELU-tanh * up), 128 features of each per workgroup.
template <bool REP>
__global__ __launch_bounds__(256, 2) void k_q4gemm2d(GemmArgs a) { gemm_tile<2, 128, 4, 1, REP, false>(a); }
// One matrix, 256 features per workgroup.
template <bool REP>
__global__ __launch_bounds__(256, 2) void k_q4gemm2s(GemmArgs a) { gemm_tile<1, 128, 4, 1, REP, false>(a); }
// 128 features (64 of each of two matrices) x BT tokens per workgroup, K
// halves in G groups.
template <int NMAT, int BT, int G, bool REP, bool RAG>
__global__ __launch_bounds__(256 * G, 2) void k_q4gemm_p(GemmArgs a) { gemm_tile<NMAT, BT, 2, G, REP, RAG>(a); }

// Launch shape of one contraction.  T is the number of 128-token x 128-feature
// tiles (64 + 64 for two matrices); two workgroups of one group fit a CU.
//  * FT 4 tiles (half the X reads per MFMA, 3-6 % faster when the chip is
//    full) where T / 2 of them fill the last round of 512 to 7/8: gate/up 512
//    tokens 121 against 128 us, but 700 tokens 197 against 188; K % 128 == 0.
//  * 128-token tiles of one group from T >= 360 (15360 x 3840, 300 tokens: 65
//    us, two groups 73) and for two matrices.
//  * Below, tiles of 64 or 128 tokens, one or two groups of waves and K in up
//    to four parts by shape_us's estimate.
struct GemmShape {
    bool ft4;
    uint32_t bt, groups, ksplit;
};
// The time in us in which the shapes of one matrix differ: rounds of workgroups
// over the CUs, each the start of a tile and its walk over the slabs, a slab in
// the time of a lone wave per SIMD or, where more, that of the waves which share
// it (a CU holds 4 waves per SIMD of 64-token tiles, 2 of 128-token ones); the
// two groups' meeting; the partial outputs, written and read again, and the launch
// that sums them if the caller does not (summed).  The constants are fitted to
// 18000 calls of 1932 sizes (256..24576 rows, K 128..15360, 65..1024 tokens, both
// layouts): 5 % rms, and the shape it picks is 1 % slower than the best one on
// average.  us, by thresholds on T as before and now: 2048 x 1024 1024 tokens
// 25.7 / 15.6, 3840 x 1024 512 tokens 23.1 / 14.3, 3840 x 4096 256 tokens 27.7 /
// 25.9, 8192 x 4096 256 tokens 39.2 / 33.2, q/k/v of 3072 rows x 512 300 tokens
// 12.3 / 10.1; 7 % over a grid of public calls.  It loses up to 6 % at some sizes
// (2048 x 4096 600 tokens 32.0 / 33.8, 2048 x 2048 256 tokens 16.0 / 17.0).
static float shape_us(uint32_t n_tok, uint32_t ct, uint32_t slabs, float outputs, const GemmShape &s, bool summed) {
    // (a few ns per shape: every count is a power of two)
    const bool small = s.bt == 64;
    const float lone = small ? 0.8f : 1.14f, shared = (small ? 0.69f : 0.97f) * s.groups, start = small ? 0.1f : 0.9f;
    const uint32_t g = s.groups >> 1, p = s.ksplit >> 1, cap = (small ? 2u : 1u) - g;     // logarithms
    const uint32_t wgs = (ct * ((n_tok + s.bt - 1) >> (small ? 6 : 7))) << p, room = 8 + cap;
    const uint32_t full = wgs >> room, rest = (wgs - (full << room) + 255) >> 8;
    const float walk = (float)((slabs + (1u << (g + p)) - 1) >> (g + p));
    auto round = [&](uint32_t per_cu) { return start + walk * fmaxf(shared * per_cu, lone); };
    float us = full * round(1u << cap) + (rest ? round(rest) : 0.0f) + (g ? (small ? 0.5f : 1.75f) : 0.0f);
    if (p) us += (summed ? 1.0f : 1.77f) * 1e-6f * outputs * s.ksplit + (summed ? 0.0f : 2.33f);
    return us;
}
static GemmShape gemm_shape(uint32_t nmat, uint32_t n_tok, uint32_t ct, uint32_t K, uint32_t rows, uint32_t max_parts,
                            bool summed) {
    const uint32_t T = ct * ((n_tok + 127) / 128), T4 = T / 2, slabs = (K + 127) / 128;
    if (K % 128 == 0 && T4 >= 448 && (T4 >= 2048 || T4 % 512 >= 448 || T4 % 512 == 0)) return {true, 128, 1, 1};
    GemmShape best{false, 128, 1, 1};
    if (nmat == 2 || T >= 360) return best;
    const float outputs = (float)n_tok * rows;
    float least = 1e30f;
    for (const uint32_t bt : {64u, 128u})
        for (const uint32_t g : {1u, 2u})
            for (uint32_t ks = 1; ks <= max_parts && ks * g <= slabs; ks *= 2) {
                // (the public calls' parts lie in the context's scratch)
                if (ks > 1 && !summed && (double)ks * n_tok * rows * 4 > (double)kGemmScratch) break;
                const GemmShape s{false, bt, g, ks};
                const float us = shape_us(n_tok, ct, slabs, outputs, s, summed);
                if (us < least) {
                    least = us;
                    best = s;
                }
            }
    return best;
}

template <int NMAT, bool REP>
static void launch_gemm(hipStream_t st, GemmArgs &a, int nseg, const GemmShape &sh) {
    const uint32_t bn = (sh.ft4 ? 256 : 128) / NMAT;
    uint32_t c = 0;
    for (int s = 0; s < 3; ++s) {
        a.c0[s] = s < nseg ? c : 0xffffffffu;
        if (s < nseg) c += (a.M[s] + bn - 1) / bn;
    }
    a.n_ct = c;
    a.n_tt = (a.n_tok + sh.bt - 1) / sh.bt;
    a.ksplit = sh.ksplit;
    const unsigned grid = (a.n_ct * a.n_tt * a.ksplit + 7) / 8 * 8;
    const bool rag = a.K % 128 != 0;
    if constexpr (NMAT == 2) {
        if (sh.ft4) k_q4gemm2d<REP><<<grid, 256, 0, st>>>(a);
        else if (rag) k_q4gemm_p<2, 128, 1, REP, true><<<grid, 256, 0, st>>>(a);
        else k_q4gemm_p<2, 128, 1, REP, false><<<grid, 256, 0, st>>>(a);
    } else if (sh.ft4) {
        k_q4gemm2s<REP><<<grid, 256, 0, st>>>(a);
    } else if (sh.bt == 128 && sh.groups == 2) {
        if (rag) k_q4gemm_p<1, 128, 2, REP, true><<<grid, 512, 0, st>>>(a);
        else k_q4gemm_p<1, 128, 2, REP, false><<<grid, 512, 0, st>>>(a);
    } else if (sh.bt == 64 && sh.groups == 2) {
        if (rag) k_q4gemm_p<1, 64, 2, REP, true><<<grid, 512, 0, st>>>(a);
        else k_q4gemm_p<1, 64, 2, REP, false><<<grid, 512, 0, st>>>(a);
    } else if (sh.bt == 64) {
        if (rag) k_q4gemm_p<1, 64, 1, REP, true><<<grid, 256, 0, st>>>(a);
        else k_q4gemm_p<1, 64, 1, REP, false><<<grid, 256, 0, st>>>(a);
    } else {
        if (rag) k_q4gemm_p<1, 128, 1, REP, true><<<grid, 256, 0, st>>>(a);
        else k_q4gemm_p<1, 128, 1, REP, false><<<grid, 256, 0, st>>>(a);
    }
}

static void launch_to_bf16(hipStream_t st, const float *X, __bf16 *xb, size_t n) {
    const size_t g = (n / 4 + 255) / 256;
    k_to_bf16<<<(unsigned)(g > 8192 ? 8192 : g), 256, 0, st>>>(X, xb, n);
}

static uint32_t gemm_cols(int nmat, int nseg, const uint32_t *M) {
    uint32_t ct = 0;
    for (int s = 0; s < nseg; ++s) ct += (M[s] * nmat + 127) / 128;
    return ct;
}

// nseg matrices over the same activations (nmat 1), or gate and up.  A shape
// that splits K writes the parts to scratch (kGemmScratch bytes), from where
// they are summed into Y[0], or to po's buffers (Y[0] and on); with neither it
// is not split.
static int gemm_run(chn_ctx *ctx, int nmat, int nseg, const float *X, const uint32_t *const *W, const uint32_t *W1,
                    float *const *Y, const uint32_t *M, uint32_t n_tok, uint32_t K, __bf16 *xb, bool repacked,
                    __bf16 *Yb, PartialOut *po, float *scratch, uint32_t yb_ntt = 0) {
    hipStream_t st = ctx->stream;
    uint32_t rows = 0;
    for (int s = 0; s < nseg; ++s) rows += M[s];
    if (po) po->parts = 1;
    if (Yb && nmat == 1) return set_err(ctx, CHN_E_UNSUPPORTED, "bf16 output needs the two-matrix contraction");
    if (few_tokens(n_tok, nmat, K, rows, nseg)) {
        if (X) {
            launch_to_bf16_few(st, X, xb, n_tok, K);
            CHN_LAUNCHED(ctx, "k_to_bf16_few");
        }
        launch_q4gemm_few(st, nmat, nseg, W, W1, Y, M, n_tok, K, xb, repacked, Yb, yb_ntt);
        CHN_LAUNCHED(ctx, "k_q4gemm_few");
        return CHN_OK;
    }
    GemmArgs a{};
    a.X = xb;
    for (int s = 0; s < nseg; ++s) {
        a.W[s] = (const unsigned char *)W[s];
        a.Y[s] = Y[s];
        a.M[s] = M[s];
    }
    a.W1 = (const unsigned char *)W1;
    a.Yb = Yb;
    a.yb_ntt = yb_ntt;
    a.n_tok = n_tok;
    a.K = K;
    const uint32_t max_parts = nseg > 1 ? 1 : (scratch ? 4 : (po ? po->max_parts : 1));
    const GemmShape sh = gemm_shape(nmat, n_tok, gemm_cols(nmat, nseg, M), K, rows, max_parts, !scratch);
    if (sh.ksplit > 1 && scratch) {
        a.Y[0] = scratch;
        a.ypart = (size_t)n_tok * M[0];
    } else if (sh.ksplit > 1) {
        a.ypart = po->stride;
        po->parts = sh.ksplit;
    }
    if (X) {
        launch_to_bf16(st, X, xb, (size_t)n_tok * K);
        CHN_LAUNCHED(ctx, "k_to_bf16");
    }
    if (nmat == 2) {
        if (repacked) launch_gemm<2, true>(st, a, nseg, sh);
        else launch_gemm<2, false>(st, a, nseg, sh);
    } else {
        if (repacked) launch_gemm<1, true>(st, a, nseg, sh);
        else launch_gemm<1, false>(st, a, nseg, sh);
    }
    CHN_LAUNCHED(ctx, "k_q4gemm");
    if (sh.ksplit > 1 && scratch) {
        k_sum_parts<<<(unsigned)((a.ypart / 4 + 256) / 256), 256, 0, st>>>(scratch, Y[0], a.ypart, sh.ksplit);
        CHN_LAUNCHED(ctx, "k_sum_parts");
    }
    return CHN_OK;
}

int launch_q4gemm(chn_ctx *ctx, int nmat, const float *X, const uint32_t *W0, const uint32_t *W1, float *Y,
                  uint32_t n_tok, uint32_t M, uint32_t K, __bf16 *xb, bool repacked, __bf16 *Yb, PartialOut *po,
                  uint32_t yb_ntt) {
    return gemm_run(ctx, nmat, 1, X, &W0, W1, &Y, &M, n_tok, K, xb, repacked, Yb, po, nullptr, yb_ntt);
}

// q, k and v of one layer in one launch: three repacked matrices over the
// same activations (one bf16 conversion, none when X is NULL and xb already
// holds them).
int launch_q4gemm_qkv(chn_ctx *ctx, const float *X, const uint32_t *Wq, const uint32_t *Wk, const uint32_t *Wv,
                      float *Yq, float *Yk, float *Yv, uint32_t n_tok, uint32_t Mq, uint32_t Mkv, uint32_t K,
                      __bf16 *xb) {
    const uint32_t *const W[3] = {Wq, Wk, Wv};
    float *const Y[3] = {Yq, Yk, Yv};
    const uint32_t M[3] = {Mq, Mkv, Mkv};
    return gemm_run(ctx, 1, 3, X, W, nullptr, Y, M, n_tok, K, xb, true, nullptr, nullptr, nullptr);
}

// The public calls' buffer for the bf16 activations (kGemmScratch).
static int public_activations(chn_ctx *ctx, uint32_t n_tok, int nmat, uint32_t K, uint32_t rows, int nseg,
                              __bf16 *&xb) {
    if (few_tokens(n_tok, nmat, K, rows, nseg)) {
        xb = (__bf16 *)ctx->gemm_scratch;
        return CHN_OK;
    }
    const int rc = ensure_workspace(ctx, (size_t)n_tok * K * 2);
    xb = (__bf16 *)ctx->ws;
    return rc;
}

static int gemm_common(chn_ctx *ctx, int nmat, const uint32_t *W0, const uint32_t *W1, const float *X, float *Y,
                       uint32_t n_tok, uint32_t M, uint32_t K, bool repacked = false, __bf16 *Yb = nullptr) {
    CHN_REQUIRE(ctx, W0 && X && (Y || Yb) && (nmat == 1 || W1), "NULL argument");
    CHN_REQUIRE(ctx, K > 0 && K % 32 == 0, "K=%u must be a positive multiple of 32", K);
    CHN_REQUIRE(ctx, K % 8 == 0 && aligned(X, 16), "X must be 16-byte aligned");
    CHN_REQUIRE(ctx, aligned(W0, repacked ? 16 : 4) && (!W1 || aligned(W1, repacked ? 16 : 4)),
                "weights must be %d-byte aligned", repacked ? 16 : 4);
    if (!n_tok || !M) return CHN_OK;
    __bf16 *xb = nullptr;
    int rc = public_activations(ctx, n_tok, nmat, K, M, 1, xb);
    if (rc) return rc;
    return gemm_run(ctx, nmat, 1, X, &W0, W1, &Y, &M, n_tok, K, xb, repacked, Yb, nullptr, (float *)ctx->gemm_scratch);
}

}  // namespace chn

using namespace chn;

extern "C" int chn_batch_gemm_q4(chn_ctx *ctx, const uint32_t *W, const float *X, float *Y, uint32_t n_tok,
                                 uint32_t M, uint32_t K) {
    if (!ctx) return CHN_E_INVALID;
    return gemm_common(ctx, 1, W, nullptr, X, Y, n_tok, M, K);
}

extern "C" int chn_batch_fused_mlp_q4(chn_ctx *ctx, const uint32_t *Wg, const uint32_t *Wu, const float *X,
                                      float *Y, uint32_t n_tok, uint32_t M, uint32_t K) {
    if (!ctx) return CHN_E_INVALID;
    return gemm_common(ctx, 2, Wg, Wu, X, Y, n_tok, M, K);
}

// The model's prefill contractions over repacked (Q4R) weights, as
// chn_prefill launches them.
extern "C" int chn_batch_gemm_q4r(chn_ctx *ctx, const void *W, const float *X, float *Y, uint32_t n_tok, uint32_t M,
                                  uint32_t K) {
    if (!ctx) return CHN_E_INVALID;
    return gemm_common(ctx, 1, (const uint32_t *)W, nullptr, X, Y, n_tok, M, K, true);
}

extern "C" int chn_batch_fused_mlp_q4r(chn_ctx *ctx, const void *Wg, const void *Wu, const float *X, float *Y,
                                       uint16_t *Y_bf16, uint32_t n_tok, uint32_t M, uint32_t K) {
    if (!ctx) return CHN_E_INVALID;
    CHN_REQUIRE(ctx, (Y == nullptr) != (Y_bf16 == nullptr), "exactly one of Y and Y_bf16 must be given");
    return gemm_common(ctx, 2, (const uint32_t *)Wg, (const uint32_t *)Wu, X, Y, n_tok, M, K, true,
                       (__bf16 *)Y_bf16);
}

extern "C" int chn_batch_qkv_q4r(chn_ctx *ctx, const void *Wq, const void *Wk, const void *Wv, const float *X,
                                 float *Yq, float *Yk, float *Yv, uint32_t n_tok, uint32_t q_dim, uint32_t kv_dim,
                                 uint32_t K) {
    if (!ctx) return CHN_E_INVALID;
    CHN_REQUIRE(ctx, Wq && Wk && Wv && X && Yq && Yk && Yv, "NULL argument");
    CHN_REQUIRE(ctx, K > 0 && K % 32 == 0, "K=%u must be a positive multiple of 32", K);
    CHN_REQUIRE(ctx, aligned(X, 16) && aligned(Wq, 16) && aligned(Wk, 16) && aligned(Wv, 16), "misaligned argument");
    if (!n_tok || !q_dim || !kv_dim) return CHN_OK;
    __bf16 *xb = nullptr;
    int rc = public_activations(ctx, n_tok, 1, K, q_dim + 2 * kv_dim, 3, xb);
    if (rc) return rc;
    return launch_q4gemm_qkv(ctx, X, (const uint32_t *)Wq, (const uint32_t *)Wk, (const uint32_t *)Wv, Yq, Yk, Yv,
                             n_tok, q_dim, kv_dim, K, xb);
}
