"""GPU parity of prefill attention with 512-wide heads (k_prefill_attn_d512)
at the edges of its tiles: 16-row query tiles that end inside, key steps of
16, lists cut into parts, windows that start inside a step.  Operands and
sums are fp32, as in the oracle; the bar is the fp32 one (1e-3; about 1e-6
is expected from the order of the sums)."""
import numpy as np
import pytest

from gpu_util import f32_host, rel_err, say, synth_normal_dev
import oracle

pytestmark = pytest.mark.gpu


def _run(ctx, nq, gqa, n, prev, window, kc, vc, slots):
    D, kvd = 512, nq // gqa * 512
    Q = synth_normal_dev(ctx, n * nq * D, 42 + n, 0.1)
    Kc, Vc, ds = ctx.upload(kc), ctx.upload(vc), ctx.upload(slots)
    out = ctx.alloc(n * nq * D * 4)
    say(f"batch_causal_attn D=512 nq={nq} gqa={gqa} n={n} prev={prev} window={window}")
    ctx.call("chn_batch_causal_attn", Q, Kc, Vc, ds, n, prev, nq, D, kvd, gqa, 1.0, window, out)
    return f32_host(ctx, Q, n * nq * D), f32_host(ctx, out, n * nq * D)


def _cache(nslot, kvd, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal(nslot * kvd, dtype=np.float32), rng.standard_normal(nslot * kvd, dtype=np.float32),
            rng.permutation(nslot).astype(np.uint32))


@pytest.mark.parametrize("nq,gqa,n,prev,window", [
    (1, 1, 1, 0, 0),           # one query, one key
    (4, 4, 5, 15, 0),          # a tile and a quarter; the list ends on a step's edge
    (8, 2, 9, 120, 33),        # a window that starts inside a step, two tiles
    (2, 1, 40, 1000, 0),       # parts of a long list
    (8, 4, 3, 2200, 0),        # more than 2048 keys: four parts
    (4, 4, 9, 5200, 0),        # parts of more than 1024 keys
    (16, 2, 260, 0, 0),        # enough workgroups for one part
    (4, 4, 70, 300, 100),      # parts whose first chunks a late query does not see
])
def test_prefill_attn_512(ctx, nq, gqa, n, prev, window):
    kvd = nq // gqa * 512
    kc, vc, perm = _cache(max(2304, prev + n), kvd, n + prev)
    slots = perm[: prev + n]
    q, got = _run(ctx, nq, gqa, n, prev, window, kc, vc, slots)
    want = oracle.batch_causal_attn(q, kc, vc, slots, n, prev, nq, 512, kvd, gqa, 1.0, window, oracle.NTHREADS)
    e = rel_err(got, want)
    say(f"  {e:.2e}")
    assert e < 1e-5


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_prefill_attn_512_nonfinite_keys(ctx, bad):
    """A non-finite V row reaches the queries that see it and no other of its
    tile, ahead of it (causality) or behind it (window); a non-finite K row
    that no query sees changes nothing."""
    nq, gqa, n, prev, window = 4, 4, 24, 40, 20
    kvd = 512
    kc, vc, perm = _cache(128, kvd, 3)
    slots = perm[: prev + n]
    key = prev + 10                      # seen by tokens 10 .. 29 within the window
    clean_q, clean = _run(ctx, nq, gqa, n, prev, window, kc, vc, slots)
    vc2, kc2 = vc.copy().reshape(-1, kvd), kc.copy().reshape(-1, kvd)
    vc2[slots[key]] = bad
    vc2[perm[prev + n:]] = bad           # rows that are not listed
    kc2[slots[5]] = np.nan               # before every window
    _, got = _run(ctx, nq, gqa, n, prev, window, kc2.ravel(), vc2.ravel(), slots)
    got, clean = got.reshape(n, -1), clean.reshape(n, -1)
    sees = np.array([prev + t + 1 - window <= key <= prev + t for t in range(n)])
    assert np.all(np.isfinite(got[~sees])) and not np.any(np.isfinite(got[sees]))
    # the products are the same ones in another grouping: K * 2^-24 of the terms
    assert np.max(np.abs(got[~sees] - clean[~sees])) < 1e-5
