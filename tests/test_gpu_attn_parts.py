"""Prefill attention with 256-wide heads where the key list is cut into fewer,
longer parts than four chunks (pa_part_chunks): one round of workgroups, lists
whose parts end off the window's edge, and a list so long that every length
gives the most parts.  The first, middle and last tokens against the oracle.
Bar as for the other shapes of this kernel: scores drop the product of the two
low halves, 2^-16 of |q| |k| per term (1e-3 after the softmax at most here; a
lost or repeated chunk of a part is a per cent or more)."""
import numpy as np
import pytest

from gpu_util import f32_host, rel_err, say, synth_normal_dev
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,gqa,n,prev,window", [
    (16, 2, 704, 40, 0),          # 11 tiles of 64 tokens, 4 to 24 chunks each
    (16, 8, 1000, 0, 0),          # 16-token tiles, one to 32 chunks
    (16, 2, 1024, 1500, 1024),    # 35 chunks per tile in two parts
    (8, 1, 500, 601, 333),        # window start and list end off the chunk grid
    (16, 2, 1024, 3000, 0),       # up to 126 chunks in four parts
])
def test_parts(ctx, nq, gqa, n, prev, window):
    D, nkv = 256, nq // gqa
    kvd, S = nkv * D, prev + n
    Kc = synth_normal_dev(ctx, S * kvd, 50 + n)
    Vc = synth_normal_dev(ctx, S * kvd, 51 + n)
    Q = synth_normal_dev(ctx, n * nq * D, 52 + n, 0.1)
    slots = np.random.default_rng(n + prev).permutation(S).astype(np.uint32)
    out = ctx.alloc(n * nq * D * 4)
    say(f"attention parts nq={nq} gqa={gqa} n={n} prev={prev} window={window}")
    ctx.call("chn_batch_causal_attn", Q, Kc, Vc, ctx.upload(slots), n, prev, nq, D, kvd, gqa, 1.0, window, out)
    got = f32_host(ctx, out, n * nq * D).reshape(n, -1)
    assert np.all(np.isfinite(got))
    Qh, Kh, Vh = f32_host(ctx, Q, n * nq * D).reshape(n, -1), f32_host(ctx, Kc, S * kvd), f32_host(ctx, Vc, S * kvd)
    for t in (0, n // 2, n - 3):
        want = oracle.batch_causal_attn(np.ascontiguousarray(Qh[t: t + 3]), Kh, Vh, slots[: prev + t + 3], 3, prev + t,
                                        nq, D, kvd, gqa, 1.0, window)
        assert rel_err(got[t: t + 3], want.reshape(3, -1)) < 1e-3


@pytest.mark.parametrize("step", [-2.0, 0.0, 2.0, 4.0, 9.0])
def test_rising_scores(ctx, step):
    """Scores that rise (or fall) by up to `step` times 16 per 32-key chunk,
    differently for the queries of a wave: the sums are rescaled in every chunk,
    in some, or only in the first."""
    nq, gqa, D, n, prev = 4, 2, 256, 70, 470
    nkv, S = nq // gqa, prev + n
    rng = np.random.default_rng(3)
    u = rng.choice([-1.0, 1.0], D) / 16
    K = (0.02 * rng.standard_normal((S, nkv, D)) + (step * np.arange(S) / 32)[:, None, None] * u).astype(np.float32)
    V = rng.standard_normal((S, nkv * D)).astype(np.float32)
    Q = (rng.standard_normal((n, nq, D)) + u * rng.uniform(0, 1, (n, nq, 1)) * 16 ** 0.5 * 4).astype(np.float32) / 4
    slots = np.arange(S, dtype=np.uint32)
    out = ctx.alloc(n * nq * D * 4)
    say(f"attention with scores rising by {step} per chunk")
    ctx.call("chn_batch_causal_attn", ctx.upload(Q), ctx.upload(K), ctx.upload(V), ctx.upload(slots), n, prev, nq, D,
             nkv * D, gqa, 4.0, 0, out)
    want = oracle.batch_causal_attn(Q.reshape(n, -1), K.ravel(), V.ravel(), slots, n, prev, nq, D, nkv * D, gqa, 4.0, 0)
    assert rel_err(f32_host(ctx, out, n * nq * D), want.ravel()) < 1e-3
