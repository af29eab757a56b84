"""q/k norm + RoPE + K/V write (k_qkv_rope) at the edges of its split: one row
per wave below 8192 rows and two from there on, row counts that leave waves
with one row or none, head sizes that are no multiple of 64, no rotation, no
KV heads, K as V, operands aligned to 4 bytes only.

Bars: the batch of n tokens equals n single-token calls bit for bit (the same
operations per row in every split), and the first and last tokens agree with
the oracle to 1e-4 (fp32 sums of at most 512 terms and angles of clock * freq
rounded to fp32: |angle| * 2^-24 <= 1e-4 at clock 1500)."""
import numpy as np
import pytest

from gpu_util import f32_host, rel_err, say
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,nkv,D,rot,keqv,n", [
    (16, 8, 256, 256, 0, 255),   # 8160 rows: the last size with one row per wave
    (16, 8, 256, 256, 0, 256),   # 8192: the first with two
    (7, 0, 64, 64, 0, 1171),     # 7 rows per token: a wave with one row, no KV head
    (6, 3, 100, 36, 0, 700),     # 12 rows: a wave with none; head size and suffix no multiple of 64
    (5, 2, 200, 0, 1, 920),      # no rotation, V from the raw K
    (3, 1, 500, 250, 0, 30),     # the wide form
    (1, 1, 2, 2, 0, 3),
])
def test_rows(ctx, nq, nkv, D, rot, keqv, n):
    qd, kvd, clock = nq * D, nkv * D, 1500 - n
    rng = np.random.default_rng(D + n)
    q, k, v = (rng.standard_normal(n * w + 1).astype(np.float32) for w in (qd, kvd, kvd))
    qn, kn = ((1 + 0.1 * rng.standard_normal(D)).astype(np.float32) for _ in range(2))
    slots = rng.permutation(n + 9).astype(np.uint32)[: n + 2]
    step = ctx.upload(np.stack([clock + np.arange(n), slots[2:]], 1).astype(np.uint32))
    dq, dk, dv, dqn, dkn, ds = (ctx.upload(a) for a in (q, k, v, qn, kn, slots))
    fill = np.full((n + 9) * max(kvd, 1) + 1, 7.0, np.float32)
    outs = []
    for batch in (True, False):
        qo, kc, vc = ctx.alloc(n * qd * 4 + 4), ctx.upload(fill), ctx.upload(fill)
        say(f"qkv_rope rows nq={nq} nkv={nkv} D={D} n={n} batch={batch}")
        # 4 bytes past each buffer's start
        if batch:
            ctx.call("chn_batch_qkv_rope", dq.ptr + 4, dk.ptr + 4, dv.ptr + 4, dqn, dkn, qo.ptr + 4, kc.ptr + 4,
                     vc.ptr + 4, ds, 2, clock, n, nq, nkv, D, rot, keqv, 1e4, 1e-6)
        else:
            for t in range(n):
                ctx.call("chn_qkv_rope", dq.ptr + 4 + 4 * t * qd, dk.ptr + 4 + 4 * t * kvd, dv.ptr + 4 + 4 * t * kvd,
                         dqn, dkn, qo.ptr + 4 + 4 * t * qd, kc.ptr + 4, vc.ptr + 4, step.ptr + 8 * t, nq, nkv, D, rot,
                         keqv, 1e4, 1e-6)
        outs.append([ctx.download(qo, np.float32, n * qd, 4), f32_host(ctx, kc, fill.size), f32_host(ctx, vc, fill.size)])
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
    qo, kc, vc = outs[0]
    assert kc[0] == 7.0 and vc[0] == 7.0
    kc, vc = kc[1:].reshape(n + 9, -1), vc[1:].reshape(n + 9, -1)
    unused = np.setdiff1d(np.arange(n + 9), slots[2:])
    assert np.all(kc[unused] == 7.0) and np.all(vc[unused] == 7.0)
    for t in (0, n - 1):
        kc_o, vc_o = np.zeros(max(kvd, 1), np.float32), np.zeros(max(kvd, 1), np.float32)
        row = slice(t * kvd + 1, (t + 1) * kvd + 1)
        qo_o = oracle.qkv_rope(q[1 + t * qd: 1 + (t + 1) * qd], k[row], v[row], qn, kn, kc_o, vc_o, nq, nkv, D, rot,
                               keqv, 1e4, 1e-6, clock + t, 0)
        assert rel_err(qo[t * qd: (t + 1) * qd], qo_o) < 1e-4
        if nkv:
            assert rel_err(kc[slots[2 + t]], kc_o) < 1e-4
            assert rel_err(vc[slots[2 + t]], vc_o) < 1e-4
