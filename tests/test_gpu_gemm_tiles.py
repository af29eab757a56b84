"""GPU parity of the prefill contractions above the few-token limits at the
edges of their launch shapes: 64- and 128-token tiles, one and two groups of
waves, split K with and without scratch sums, K that ends inside a slab of
128, rows and tokens that end inside a tile.  Bar: 1e-4 against the
bf16-operand model (equal operand roundings, another order of fp32 sums)."""
import numpy as np
import pytest

import channel_amd as ca
from gpu_util import f32_host, q4_host, rel_err, say, synth_normal_dev, synth_q4_dev
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("repacked", [False, True])
@pytest.mark.parametrize("n_tok,M,K", [
    # 64-token tiles, one group of waves
    (129, 130, 32),        # one block of K
    (257, 70, 416),        # a tile of one token
    (300, 7000, 160),
    (129, 2903, 1568),     # K split in two, ragged K, odd row length
    (200, 300, 1056),      # K split in four, ragged K
    # 64-token tiles, two groups
    (513, 200, 672),       # one with a slab less
    (513, 200, 768),
    (129, 2903, 1312),     # K split in two
    (65, 200, 8224),       # K split in four
    # 128-token tiles, one group
    (385, 11520, 96),      # 360 tiles, one ragged slab
    (65, 5000, 3104),      # K split in four
    # 128-token tiles, two groups
    (257, 7001, 1440),     # one with a slab less, odd row length
    (65, 9000, 3936),      # K split in two
    (65, 4500, 5664),      # K split in four
    (130, 57300, 128),     # 256-feature tiles (448 of them), one slab
    (130, 57300, 384),     # an odd and an even number of slabs: both DMA slots, the hand-over of the weights
    (250, 57300, 512),     # (the last group of tokens and of features partly and wholly past the end)
])
def test_gemm_launch_shapes(ctx, n_tok, M, K, repacked):
    W = synth_q4_dev(ctx, M, K, 60 + M)
    Wh = q4_host(ctx, W, M, K)
    if repacked:
        R = ctx.alloc(ca.q4r_bytes(M, K))
        ctx.call("chn_q4_repack", W, M, K, R)
        W = R
    X = synth_normal_dev(ctx, n_tok * K, 61 + K)
    Y = ctx.alloc((n_tok * M + 64) * 4)
    ctx.fill_u32(Y, 0x7FC00000, n_tok * M + 64)
    say(f"gemm n_tok={n_tok} M={M} K={K} repacked={repacked}")
    ctx.call("chn_batch_gemm_q4r" if repacked else "chn_batch_gemm_q4", W, X, Y, n_tok, M, K)
    got = f32_host(ctx, Y, n_tok * M + 64)
    Xh = f32_host(ctx, X, n_tok * K).reshape(n_tok, K)
    assert np.all(np.isnan(got[n_tok * M:]))                       # nothing written past the result
    want = oracle.batch_gemm_q4_bf16(Wh, Xh, n_tok, M, K, oracle.NTHREADS)
    assert rel_err(got[: n_tok * M].reshape(n_tok, M), want) < 1e-4


@pytest.mark.parametrize("repacked", [False, True])
@pytest.mark.parametrize("n_tok,M,K", [(65, 200, 352), (130, 28610, 128), (130, 28610, 384), (245, 28610, 256)])
def test_gate_up_launch_shapes(ctx, n_tok, M, K, repacked):
    """64 and (448 tiles, K % 128 == 0) 128 features of each matrix per workgroup."""
    W, Wh = [], []
    for i in range(2):
        w = synth_q4_dev(ctx, M, K, 65 + i)
        Wh.append(q4_host(ctx, w, M, K))
        if repacked:
            r = ctx.alloc(ca.q4r_bytes(M, K))
            ctx.call("chn_q4_repack", w, M, K, r)
            w = r
        W.append(w)
    X = synth_normal_dev(ctx, n_tok * K, 67)
    Y = ctx.alloc(n_tok * M * 4)
    say(f"gate/up n_tok={n_tok} M={M} K={K} repacked={repacked}")
    if repacked:
        ctx.call("chn_batch_fused_mlp_q4r", *W, X, Y, None, n_tok, M, K)
    else:
        ctx.call("chn_batch_fused_mlp_q4", *W, X, Y, n_tok, M, K)
    Xh = f32_host(ctx, X, n_tok * K).reshape(n_tok, K)
    g, u = (oracle.batch_gemm_q4_bf16(w, Xh, n_tok, M, K, oracle.NTHREADS) for w in Wh)
    want = oracle.gelu_tanh(g.ravel()).reshape(n_tok, M) * u
    assert rel_err(f32_host(ctx, Y, n_tok * M).reshape(n_tok, M), want) < 1e-4


def test_qkv_wide_tiles(ctx):
    """Three segments on 256-feature tiles (512 of them), several slabs."""
    n_tok, K, rows = 1020, 384, (8190, 4095, 4095)
    X = synth_normal_dev(ctx, n_tok * K, 69)
    Xh = f32_host(ctx, X, n_tok * K).reshape(n_tok, K)
    R, Wh, Y = [], [], [ctx.alloc(n_tok * M * 4) for M in rows]
    for i, M in enumerate(rows):
        w = synth_q4_dev(ctx, M, K, 70 + i)
        Wh.append(q4_host(ctx, w, M, K))
        R.append(ctx.alloc(ca.q4r_bytes(M, K)))
        ctx.call("chn_q4_repack", w, M, K, R[-1])
    say(f"qkv n_tok={n_tok} rows={rows} K={K}")
    ctx.call("chn_batch_qkv_q4r", *R, X, *Y, n_tok, rows[0], rows[1], K)
    for w, y, M in zip(Wh, Y, rows):
        want = oracle.batch_gemm_q4_bf16(w, Xh, n_tok, M, K, oracle.NTHREADS)
        assert rel_err(f32_host(ctx, y, n_tok * M).reshape(n_tok, M), want) < 1e-4


def test_nonfinite_activations_stay_in_their_row(ctx):
    """Padding (K past a slab's end, tokens past a tile's) contributes exact
    zeros next to infinities and NaN: only the rows that hold them change."""
    n_tok, M, K = 150, 100, 1056
    W = synth_q4_dev(ctx, M, K, 68)
    rng = np.random.default_rng(5)
    Xh = rng.standard_normal((n_tok, K)).astype(np.float32)
    bad = Xh.copy()
    bad[3, K - 1], bad[149, 0] = np.inf, np.nan
    out = []
    for x in (Xh, bad):
        Y = ctx.alloc(n_tok * M * 4)
        for n in (n_tok, 100):                                     # both kernels
            ctx.call("chn_batch_gemm_q4", W, ctx.upload(x), Y, n, M, K)
            out.append(f32_host(ctx, Y, n * M).reshape(n, M))
    for clean, got in ((out[0], out[2]), (out[1], out[3])):
        rows = [r for r in range(clean.shape[0]) if r not in (3, 149)]
        assert np.array_equal(clean[rows], got[rows]) and np.all(np.isfinite(clean))
        assert not np.any(np.isfinite(got[3]))
