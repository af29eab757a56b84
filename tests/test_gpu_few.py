"""GPU parity of the few-token contractions (few_tokens, k_q4gemm_few) at
the edges of their tiles: 16-token tiles and groups of 1..4 of them, 16- and
32-feature workgroups, K steps of 256 that end inside a step, a half or a
block, and the sizes above 128 tokens that they take.  Bar as for the other MFMA contractions: 1e-4 against the
bf16-operand model (the same operand roundings, so only the order of the
fp32 sums differs: K * 2^-24 <= 1e-3 of the terms' magnitudes at worst,
~sqrt(K) * 2^-24 ~ 1e-5 in practice)."""
import numpy as np
import pytest

import channel_amd as ca
from channel_amd.model import Model
from gpu_util import assert_topk_valid, f32_host, q4_host, rel_err, say, synth_normal_dev, synth_q4_dev
import oracle
from oracle import model as OM

pytestmark = pytest.mark.gpu


def _matrix(ctx, rows, K, seed, repacked):
    W = synth_q4_dev(ctx, rows, K, seed)
    Wh = q4_host(ctx, W, rows, K)
    if repacked:
        R = ctx.alloc(ca.q4r_bytes(rows, K))
        ctx.call("chn_q4_repack", W, rows, K, R)
        return R, Wh
    return W, Wh


@pytest.mark.parametrize("repacked", [False, True])
@pytest.mark.parametrize("n_tok,M,K", [
    (1, 16, 32),         # one block, fewer steps than waves
    (16, 17, 224),       # a full token tile, one feature past a tile, a step short of a block
    (17, 500, 288),      # a second tile of one token, one block into a second step
    (33, 7681, 384),     # 32-feature workgroups, one row past the last, half a step at the end
    (65, 48, 2304),      # five tiles in groups of three and two; nine steps over eight waves
    (128, 100, 4128),    # eight tiles, two groups of four
    (129, 300, 512),     # nine tiles in three groups, the shortest K above 128 tokens
    (512, 1024, 1024),   # eight groups of four, the most workgroups and the longest K there
    (401, 1000, 992),    # 26 tiles in seven groups, ragged K
])
def test_few_gemm_parity(ctx, n_tok, M, K, repacked):
    W, Wh = _matrix(ctx, M, K, 70 + M, repacked)
    X = synth_normal_dev(ctx, n_tok * K, 71 + K)
    Y = ctx.alloc((n_tok * M + 64) * 4)
    ctx.fill_u32(Y, 0x7FC00000, n_tok * M + 64)
    say(f"few-token gemm n_tok={n_tok} M={M} K={K} repacked={repacked}")
    ctx.call("chn_batch_gemm_q4r" if repacked else "chn_batch_gemm_q4", W, X, Y, n_tok, M, K)
    got = f32_host(ctx, Y, n_tok * M + 64)
    Xh = f32_host(ctx, X, n_tok * K).reshape(n_tok, K)
    want = oracle.batch_gemm_q4_bf16(Wh, Xh, n_tok, M, K, oracle.NTHREADS)
    assert np.all(np.isnan(got[n_tok * M:]))                       # nothing written past the result
    assert rel_err(got[: n_tok * M].reshape(n_tok, M), want) < 1e-4


@pytest.mark.parametrize("n_tok,M,K,bf16_out", [(24, 7680, 256, True), (24, 7680, 256, False), (100, 90, 352, True)])
def test_few_fused_mlp_parity(ctx, n_tok, M, K, bf16_out):
    """Both workgroup widths of the two-matrix form; the public bf16 result is row-major."""
    Wg, Wgh = _matrix(ctx, M, K, 80, True)
    Wu, Wuh = _matrix(ctx, M, K, 81, True)
    X = synth_normal_dev(ctx, n_tok * K, 82)
    Y = ctx.alloc(n_tok * M * 4)
    say(f"few-token fused mlp n_tok={n_tok} M={M} K={K} bf16={bf16_out}")
    ctx.call("chn_batch_fused_mlp_q4r", Wg, Wu, X, None if bf16_out else Y, Y if bf16_out else None, n_tok, M, K)
    if bf16_out:
        got = (ctx.download(Y, np.uint16, n_tok * M).astype(np.uint32) << 16).view(np.float32)
    else:
        got = f32_host(ctx, Y, n_tok * M)
    Xh = f32_host(ctx, X, n_tok * K).reshape(n_tok, K)
    g16 = oracle.batch_gemm_q4_bf16(Wgh, Xh, n_tok, M, K, oracle.NTHREADS)
    u16 = oracle.batch_gemm_q4_bf16(Wuh, Xh, n_tok, M, K, oracle.NTHREADS)
    want = oracle.gelu_tanh(g16.ravel()).reshape(n_tok, M) * u16
    # a bf16 result is within 2^-8 of the value it rounds
    assert rel_err(got.reshape(n_tok, M), want) < (2.0 ** -8 if bf16_out else 1e-4)


@pytest.mark.parametrize("qd,kvd", [(50, 30), (5000, 1500)])
def test_few_qkv_segments(ctx, qd, kvd):
    """Three matrices in one launch, none ending on a workgroup's edge."""
    n_tok, K = 40, 320
    mats = [_matrix(ctx, m, K, 90 + i, True) for i, m in enumerate((qd, kvd, kvd))]
    X = synth_normal_dev(ctx, n_tok * K, 93)
    Y = [ctx.alloc(n_tok * m * 4) for m in (qd, kvd, kvd)]
    say(f"few-token qkv {qd} | {kvd} | {kvd}")
    ctx.call("chn_batch_qkv_q4r", *[m[0] for m in mats], X, *Y, n_tok, qd, kvd, K)
    Xh = f32_host(ctx, X, n_tok * K).reshape(n_tok, K)
    for (_, Wh), y, M in zip(mats, Y, (qd, kvd, kvd)):
        want = oracle.batch_gemm_q4_bf16(Wh, Xh, n_tok, M, K, oracle.NTHREADS)
        assert rel_err(f32_host(ctx, y, n_tok * M).reshape(n_tok, M), want) < 1e-4


@pytest.mark.parametrize("max_tok,n", [(1, 1), (128, 21), (160, 128), (160, 129)])
def test_prefill_across_the_token_limit(ctx, max_tok, n):
    """Whole prefills whose widths end inside a K step (hidden 384, FFN 640),
    with 256- and 512-wide heads, on both sides of the limit: every producer
    of bf16 activations writes the order its contraction reads."""
    cfg = OM.default_config(hidden_size=384, intermediate_size=640, vocab_size=512, num_layers=2, num_heads=2,
                            num_kv_heads=1, head_dim=256, rotary_dim=256, global_head_dim=512, layer_full=[0, 1],
                            max_prefill_tokens=max_tok, sliding_window=64)
    layers, embed, final = OM.random_model(cfg, 5)
    W = OM.Weights(cfg, layers, embed, final)
    say(f"prefill of {n} tokens, at most {max_tok}")
    toks = [int(t) for t in np.random.default_rng(n).integers(0, 512, n)]
    with Model.create(ctx, cfg, layers, embed, final) as m:
        lg, ids, vals = m.prefill_batch(toks, np.arange(n), 0, 0)
        kv = [m.kv_read(i, 0, n) for i in range(2)]
    kc, vc = OM.new_caches(cfg, 4096)
    _, _, lg_o, _, _ = OM.prefill(W, kc, vc, toks, np.arange(n), 0, 0, bf16_gemm=True, window=1024)
    assert rel_err(lg, lg_o) < 1e-2
    assert_topk_valid(ids, vals, lg_o, 1e-2, f"prefill {n}")
    for i, (k, v) in enumerate(kv):
        kvd = k.shape[1]
        assert rel_err(k, kc[i][: n * kvd].reshape(n, kvd)) < 1e-2
        assert rel_err(v, vc[i][: n * kvd].reshape(n, kvd)) < 1e-2
