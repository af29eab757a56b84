"""Performance cases of the Q4 inference backend, through its public entry points.

A case is a dict of plain values whose "kind" names the path:

  gemv          one Q4 matvec on the reference's block layout (chn_gemv_q4),
                the call a host makes that keeps the reference's weights
  ffn_decode    the MLP half of a decode step over several layers: norms +
                gate/up + GELU (chn_ffn_gate_up_q4r), then the down projection
                on the planes it wrote (chn_gemv_q4r_xp)
  attn_decode   the attention half of a decode step over several layers: q/k
                norm + RoPE + K/V write (chn_qkv_rope), then attention over
                the active slots of a ring (chn_decode_attn)
  logits        the end of a decode step: Q8 logits over the tied embedding
                (chn_gemv_q8r) and the softcapped top-64 (chn_topk64)
  gemm_prefill  one batched contraction on the reference's layout
                (chn_batch_gemm_q4)
  mlp_prefill   the MLP of one prefill layer: pre-FFN norm, gate/up + GELU,
                down (chn_batch_add_rmsnorm, chn_batch_fused_mlp_q4r,
                chn_batch_gemm_q4r)
  qkv_prefill   the front of one prefill layer: input norm, q/k/v, q/k norm +
                RoPE + K/V write (chn_batch_rmsnorm, chn_batch_qkv_q4r,
                chn_batch_qkv_rope)
  attn_prefill  causal attention of a prompt chunk over earlier and new keys
                (chn_batch_causal_attn)
  prefill       a whole Model.prefill_batch call: a chunk of a prompt through
                the first layers of a model, logits back on the host
  decode        a whole Model.decode_greedy call of several tokens, then the
                last step's logits read back (Model.read_logits)

Sizes: the 12B-class model of bench.py (hidden 3840, FFN 15360, 16 query / 8
KV heads of 256, vocabulary 262144), the reference's prefill chunk (at most
1024 tokens) and ring (4096 slots), and generic smaller models.
"""
import math

import numpy as np
import torch

import channel_amd as ca
from channel_amd.model import Model, ModelConfig

EPS = 1e-6
RING = 4096           # slots of the KV ring
WINDOW_SLOTS = 3968   # its FIFO part, the rest holds recalled entries
THETA, THETA_FULL = 1e4, 1e6


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the single matvec that bench.py calls gemv: the smallest call, bound by its launch
        dict(name="gemv_8192x2048", kind="gemv", M=8192, K=2048),
        # six layers, so that the weights come from HBM as they do in a 48-layer step
        dict(name="ffn_decode_12b", kind="ffn_decode", layers=6, H=3840, I=15360),
        # a conversation that has filled the ring: a global layer's list
        dict(name="attn_decode_ring", kind="attn_decode", layers=4, S=4096, D=256, nq=16, nkv=8, clock=9000),
        # the whole vocabulary of the 12B model
        dict(name="logits_12b", kind="logits", V=262144, K=3840),
        # a prompt of 512 tokens on the reference's layout (bench.py's prefill)
        dict(name="gemm_prefill_512", kind="gemm_prefill", n=512, M=15360, K=3840),
        # a short chat message
        dict(name="mlp_prefill_24", kind="mlp_prefill", n=24, H=3840, I=15360),
        # the largest chunk the reference's server sends
        dict(name="mlp_prefill_1024", kind="mlp_prefill", n=1024, H=3840, I=15360),
        # an ordinary message that fills no tile
        dict(name="qkv_prefill_300", kind="qkv_prefill", n=300, H=3840, D=256, nq=16, nkv=8, rot=256, clock=700),
        # a full chunk in the middle of a document, as a sliding layer sees it
        dict(name="attn_prefill_1024", kind="attn_prefill", n=1024, prev=1500, D=256, nq=16, nkv=8, window=1024),
        # a message in a conversation, as a full layer with 512-wide heads sees it
        dict(name="attn_prefill_d512", kind="attn_prefill", n=200, prev=411, D=512, nq=16, nkv=4, window=0),
        # a 512-token prompt (six layers: rounding in 16 bits travels from layer to layer)
        dict(name="prefill_512", kind="prefill", layers=6, n=512, H=3840, I=15360, D=256, gD=0, nq=16, nkv=8,
             gnkv=0, V=262144),
        # bench.py's workload: tokens of the 48-layer model after a prompt
        dict(name="decode_12b", kind="decode", layers=48, tokens=8, clock=600, H=3840, I=15360, D=256, gD=0, nq=16,
             nkv=8, gnkv=0, V=262144),
    ]


def _log_int(rng, lo, hi, step=1):
    """An integer between lo and hi, even over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def _heads(rng):
    """(D, nq, nkv): the head shapes the attention takes."""
    D = rng.choice([256, 256, 512])
    nkv = rng.choice([1, 2, 4, 8])
    return D, nkv * rng.choice([1, 2, 4]), nkv


def draw(rng):
    kind = rng.choice(["gemv", "ffn_decode", "attn_decode", "logits", "gemm_prefill", "mlp_prefill", "qkv_prefill",
                       "attn_prefill", "prefill", "decode"])
    if kind == "gemv":
        return dict(kind=kind, M=_log_int(rng, 1024, 20000), K=_log_int(rng, 256, 8192, 32))
    if kind == "ffn_decode":
        return dict(kind=kind, layers=rng.randint(2, 6), H=_log_int(rng, 512, 4096, 128),
                    I=_log_int(rng, 1024, 15360, 128))
    if kind == "attn_decode":
        D, nq, nkv = _heads(rng)
        S = _log_int(rng, 1, RING)
        return dict(kind=kind, layers=rng.randint(2, 4), S=S, D=D, nq=nq, nkv=nkv, clock=S + rng.randint(0, 20000))
    if kind == "logits":
        return dict(kind=kind, V=_log_int(rng, 8192, 262144), K=_log_int(rng, 512, 3840, 128))
    if kind == "gemm_prefill":
        return dict(kind=kind, n=_log_int(rng, 1, 1024), M=_log_int(rng, 512, 8192), K=_log_int(rng, 256, 8192, 32))
    if kind == "mlp_prefill":
        return dict(kind=kind, n=_log_int(rng, 1, 1024), H=_log_int(rng, 512, 3840, 64),
                    I=_log_int(rng, 1024, 15360, 64))
    if kind == "qkv_prefill":
        D, nq, nkv = _heads(rng)
        return dict(kind=kind, n=_log_int(rng, 1, 1024), H=_log_int(rng, 512, 3840, 32), D=D, nq=nq, nkv=nkv,
                    rot=rng.choice([D, D, D // 2]), clock=rng.randint(0, 3000))
    if kind == "attn_prefill":
        D, nq, nkv = _heads(rng)
        n = _log_int(rng, 1, 1024)
        return dict(kind=kind, n=n, prev=rng.randint(0, 1500 if D == 256 else 600), D=D, nq=nq, nkv=nkv,
                    window=rng.choice([0, 1024, 512]) if D == 256 else 0)
    H, I = _log_int(rng, 512, 3840, 128), _log_int(rng, 1024, 15360, 128)
    _, nq, nkv = _heads(rng)
    wide = rng.random() < 0.3     # full layers with 512-wide heads
    model = dict(layers=rng.randint(5, 6) if kind == "prefill" else rng.randint(5, 24), H=H, I=I, D=256,
                 gD=512 if wide else 0, nq=nq, nkv=nkv, gnkv=0, V=_log_int(rng, 8192, 262144))
    if kind == "prefill":
        return dict(kind=kind, n=_log_int(rng, 1, 512), **model)
    return dict(kind=kind, tokens=rng.randint(1, 8), clock=_log_int(rng, 16, 2000), **model)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed, k=0):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + k) % (1 << 62))


def _randn(shape, g, std=1.0):
    return torch.randn(shape, generator=g, device="cuda") * std


def _weight_q4(rows, K, g):
    """Gaussian weights in the reference's Q4 blocks: int32 [rows][K/32][5], word 0 = f16 scale | f16 min << 16,
    words 1..4 = 32 codes of 4 bits."""
    w = _randn((rows, K // 32, 32), g, 0.02)
    d = w.abs().amax(2, keepdim=True) / 8
    q = (w / d + 8.5).floor_().clamp_(0, 15).to(torch.int32)
    half = lambda v: v.to(torch.float16).view(torch.int16).to(torch.int32) & 0xFFFF  # noqa: E731
    out = torch.empty((rows, K // 32, 5), dtype=torch.int32, device="cuda")
    out[:, :, 0] = half(d[:, :, 0]) | (half(-8 * d[:, :, 0]) << 16)
    q = q.view(rows, K // 32, 4, 8)
    word = q[..., 0].clone()
    for i in range(1, 8):
        word |= q[..., i] << (4 * i)
    out[:, :, 1:] = word
    return out


def _dequant_q4(W):
    """float64 [rows][K] of the blocks."""
    s = (W[:, :, 0] & 0xFFFF).to(torch.int16).view(torch.float16).double()
    q = torch.stack([(W[:, :, 1:] >> (4 * i)) & 15 for i in range(8)], 3)
    return ((q.double() - 8) * s[:, :, None, None]).flatten(1)


def _rows_like_activations(n, K, g):
    """Normed rows: unit variance, with a few channels that are larger throughout, as trained models have them."""
    x = _randn((n, K), g)
    hot = torch.randperm(K, generator=g, device="cuda")[: max(1, K // 256)]
    x[:, hot] *= 6.0
    return x


def _norm_weight(n, g, base=1.0):
    return (1.0 + _randn((n,), g, 0.1)) * base


def _inputs(case, seed):
    """The tensors of a kernel-level case; exact() makes the same ones again."""
    g, t, kind = _gen(seed), {}, case["kind"]
    if kind == "gemv":
        t["W"] = [_weight_q4(case["M"], case["K"], g)]
        t["x"] = _rows_like_activations(1, case["K"], g)[0].contiguous()
    elif kind == "ffn_decode":
        H, I = case["H"], case["I"]
        t["x"], t["r"] = _randn((H,), g, 3.0), _randn((case["layers"], H), g)
        t["post"], t["pre"] = ([_norm_weight(H, g) for _ in range(case["layers"])] for _ in range(2))
    elif kind == "attn_decode":
        D, nq, nkv, L = case["D"], case["nq"], case["nkv"], case["layers"]
        t["q"], t["k"], t["v"] = (_randn((L, h * D), g) for h in (nq, nkv, nkv))
        # q/k norms a quarter of one keep unit-scale scores O(1), as trained ones do
        t["qw"], t["kw"] = _norm_weight(D, g, 0.25), _norm_weight(D, g, 0.25)
        t["kc"] = [_randn((RING, nkv * D), g, 0.25) for _ in range(L)]
        t["vc"] = [_randn((RING, nkv * D), g) for _ in range(L)]
    elif kind == "logits":
        V, K = case["V"], case["K"]
        w = _randn((V, K // 32, 32), g, 0.02)
        d = w.abs().amax(2, keepdim=True) / 127
        t["codes"] = (w / d).round_().to(torch.int8)
        t["scale"] = d[:, :, 0].contiguous()
        t["x"] = _randn((K,), g)
    elif kind in ("gemm_prefill", "mlp_prefill", "qkv_prefill"):
        width = case["K"] if kind == "gemm_prefill" else case["H"]
        t["X"] = _rows_like_activations(case["n"], width, g)
        if kind == "mlp_prefill":
            t["R"] = _randn((case["n"], width), g)
        t["nw"] = _norm_weight(width, g)
        if kind == "qkv_prefill":
            t["qw"], t["kw"] = _norm_weight(case["D"], g, 0.25), _norm_weight(case["D"], g, 0.25)
    else:
        n, keys, D, nq, nkv = case["n"], case["prev"] + case["n"], case["D"], case["nq"], case["nkv"]
        t["q"] = _randn((n, nq * D), g, 0.25)
        t["kc"] = _randn((RING, nkv * D), g, 0.25)
        t["vc"] = _randn((RING, nkv * D), g)
        # the chunk's keys end somewhere in the ring, in clock order
        first = int(torch.randint(0, WINDOW_SLOTS, (1,), generator=g, device="cuda"))
        t["slots"] = ((torch.arange(keys, device="cuda") + first) % WINDOW_SLOTS).to(torch.int32)
    return t


def _weights(case, seed, layer=0):
    """The Q4 matrices of one layer of a kernel-level case."""
    g, kind = _gen(seed, 17 + layer), case["kind"]
    if kind in ("ffn_decode", "mlp_prefill"):
        shapes = [(case["I"], case["H"]), (case["I"], case["H"]), (case["H"], case["I"])]
    elif kind == "qkv_prefill":
        shapes = [(h * case["D"], case["H"]) for h in (case["nq"], case["nkv"], case["nkv"])]
    else:
        shapes = [(case["M"], case["K"])]
    return [_weight_q4(r, K, g) for r, K in shapes]


def _slot_of(case):
    """The ring slot of the newest token of attn_decode, and its list in clock order."""
    S, newest = case["S"], case["clock"] % RING
    return newest, (torch.arange(S, device="cuda") + newest + 1 - S) % RING


def _model_config(case):
    return ModelConfig.from_dict(dict(
        hidden_size=case["H"], intermediate_size=case["I"], vocab_size=case["V"], num_layers=case["layers"],
        num_heads=case["nq"], num_kv_heads=case["nkv"], head_dim=case["D"], rotary_dim=case["D"],
        global_head_dim=case["gD"], num_global_kv_heads=case["gnkv"], rms_norm_eps=EPS, rope_theta=THETA,
        rope_theta_full=THETA_FULL, sliding_window=512, k_eq_v=0, max_prefill_tokens=1024,
        layer_full=[1 if (i + 1) % 5 == 0 else 0 for i in range(case["layers"])]))


def _model_inputs(case, seed):
    """(weight seed, token ids, per-layer K rows, V rows) of a whole call."""
    g = _gen(seed, 5)
    if case["kind"] == "prefill":
        return int(seed) * 7919 + 1, torch.randint(0, case["V"], (case["n"],), generator=g, device="cuda"), None, None
    kv = [case["nkv"] * (case["gD"] if (i + 1) % 5 == 0 and case["gD"] else case["D"]) for i in range(case["layers"])]
    tok = torch.randint(0, case["V"], (1,), generator=g, device="cuda")
    k = [_randn((case["clock"], d), g, 0.25) for d in kv]
    v = [_randn((case["clock"], d), g) for d in kv]
    return int(seed) * 7919 + 1, tok, k, v


# ---------------------------------------------------------------------------
# the program
# ---------------------------------------------------------------------------
_CTX = []


def _ctx():
    """The program's one context."""
    if not _CTX:
        _CTX.append(ca.Context(0))
    return _CTX[0]


class State:
    """What a program holds: bound calls, the tensors they use, what they give."""

    def __init__(self):
        self.calls, self.keep, self.out, self.model, self.whole = [], [], None, None, None

    def call(self, fn, *args):
        self.keep.extend(a for a in args if isinstance(a, torch.Tensor))
        self.calls.append(_ctx().bind(fn, *[a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args]))

    def __del__(self):
        if self.model is not None:
            self.model.close()


def _buf(*shape):
    return torch.empty(shape, dtype=torch.float32, device="cuda")


def _repacked(W):
    """The matrix as the model holds it (Q4R)."""
    rows, nb = W.shape[0], W.shape[1]
    out = torch.empty(ca.q4r_bytes(rows, nb * 32), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    _ctx().call("chn_q4_repack", W.data_ptr(), rows, nb * 32, out.data_ptr())
    _ctx().sync()
    return out


def prepare(case, seed):
    s, kind = State(), case["kind"]
    if kind in ("prefill", "decode"):
        return _prepare_model(case, seed, s)
    t = _inputs(case, seed)
    if kind == "gemv":
        y = _buf(case["M"])
        s.call("chn_gemv_q4", t["W"][0], t["x"], y, case["M"], case["K"])
        s.out = y
    elif kind == "ffn_decode":
        H, I = case["H"], case["I"]
        x, outs = t["x"], []
        for i in range(case["layers"]):
            Wg, Wu, Wd = (_repacked(w) for w in _weights(case, seed, i))
            r = t["r"][i].contiguous()
            x2, normed, act, y = _buf(H), _buf(H), _buf(I), _buf(H)
            planes = torch.empty(ca.xplanes_bytes(I), dtype=torch.uint8, device="cuda")
            s.call("chn_ffn_gate_up_q4r", Wg, Wu, x, r, t["post"][i], t["pre"][i], x2, normed, act, planes, I, H, EPS)
            s.call("chn_gemv_q4r_xp", Wd, planes, y, H, I)
            outs += [x2, act, y]
            x = x2
        s.out = outs
    elif kind == "attn_decode":
        D, nq, nkv = case["D"], case["nq"], case["nkv"]
        slot, lst = _slot_of(case)
        slots = torch.zeros(RING, dtype=torch.int32, device="cuda")
        slots[: case["S"]] = lst.to(torch.int32)
        step = torch.tensor([case["clock"], slot], dtype=torch.int32, device="cuda")
        count = torch.tensor([case["S"]], dtype=torch.int32, device="cuda")
        outs = []
        for i in range(case["layers"]):
            q, k, v = (t[n][i].contiguous() for n in "qkv")
            qo, o, kc, vc = _buf(nq * D), _buf(nq * D), t["kc"][i], t["vc"][i]
            s.call("chn_qkv_rope", q, k, v, t["qw"], t["kw"], qo, kc, vc, step, nq, nkv, D, D, 0, THETA_FULL, EPS)
            s.call("chn_decode_attn", qo, kc, vc, slots, count, RING, nq, D, nkv * D, nq // nkv, 1.0, o)
            outs += [o, kc, vc]
        s.out = outs
    elif kind == "logits":
        V, K = case["V"], case["K"]
        w = torch.empty((V, K // 32, 36), dtype=torch.uint8, device="cuda")
        w[:, :, :4] = t["scale"].view(V, K // 32, 1).view(torch.uint8)
        w[:, :, 4:] = t["codes"].view(torch.uint8)
        r = torch.empty(V * (K // 32) * 36, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        _ctx().call("chn_q8_repack", w.data_ptr(), V, K, r.data_ptr())
        _ctx().sync()
        y, ids, vals = _buf(V), torch.zeros(64, dtype=torch.int32, device="cuda"), _buf(64)
        s.call("chn_gemv_q8r", r, t["x"], y, V, K)
        s.call("chn_topk64", y, V, ids, vals)
        s.out = [y, vals]
    elif kind == "gemm_prefill":
        n, M, K = case["n"], case["M"], case["K"]
        y = _buf(n, M)
        s.call("chn_batch_gemm_q4", _weights(case, seed)[0], t["X"], y, n, M, K)
        s.out = y
    elif kind == "mlp_prefill":
        n, H, I = case["n"], case["H"], case["I"]
        Wg, Wu, Wd = (_repacked(w) for w in _weights(case, seed))
        x, xn, act, y = _buf(n, H), _buf(n, H), _buf(n, I), _buf(n, H)
        # the call updates the stream in place: it is put back from X first, as a new chunk's would be
        s.call("chn_copy", x, t["X"], n * H * 4)
        s.call("chn_batch_add_rmsnorm", x, t["R"], t["nw"], xn, n, H, EPS, 1.0)
        s.call("chn_batch_fused_mlp_q4r", Wg, Wu, xn, act, None, n, I, H)
        s.call("chn_batch_gemm_q4r", Wd, act, y, n, H, I)
        s.out = [x, act, y]
    elif kind == "qkv_prefill":
        n, H, D, nq, nkv = case["n"], case["H"], case["D"], case["nq"], case["nkv"]
        Wq, Wk, Wv = (_repacked(w) for w in _weights(case, seed))
        xn, q, k, v, qo = _buf(n, H), _buf(n, nq * D), _buf(n, nkv * D), _buf(n, nkv * D), _buf(n, nq * D)
        slots = ((torch.arange(n, device="cuda") + case["clock"]) % WINDOW_SLOTS).to(torch.int32)
        kc, vc = torch.zeros((2, RING, nkv * D), device="cuda")
        s.call("chn_batch_rmsnorm", t["X"], t["nw"], xn, n, H, EPS)
        s.call("chn_batch_qkv_q4r", Wq, Wk, Wv, xn, q, k, v, n, nq * D, nkv * D, H)
        s.call("chn_batch_qkv_rope", q, k, v, t["qw"], t["kw"], qo, kc, vc, slots, 0, case["clock"], n, nq, nkv, D,
               case["rot"], 0, THETA, EPS)
        s.out = [qo, kc, vc]
    else:
        n, D, nq, nkv = case["n"], case["D"], case["nq"], case["nkv"]
        o = _buf(n, nq * D)
        s.call("chn_batch_causal_attn", t["q"], t["kc"], t["vc"], t["slots"], n, case["prev"], nq, D, nkv * D,
               nq // nkv, 1.0, case["window"], o)
        s.out = o
    s.keep.append(t)
    return s


def _prepare_model(case, seed, s):
    wseed, tok, k, v = _model_inputs(case, seed)
    torch.cuda.synchronize()
    m = s.model = Model.synthetic(_ctx(), _model_config(case), wseed)
    tok = tok.cpu().numpy().astype(np.uint32)
    if case["kind"] == "prefill":
        slots = np.arange(case["n"], dtype=np.uint32)

        def whole():
            logits, _, vals = m.prefill_batch(tok, slots, 0, 0)
            return [logits, vals]
    else:
        for i in range(case["layers"]):
            m.kv_write(i, 0, k[i].cpu().numpy(), v[i].cpu().numpy())

        def whole():
            ids = m.decode_greedy(int(tok[0]), case["clock"], case["tokens"])
            return [ids.astype(np.int64), m.read_logits()]
    s.whole = whole
    return s


def run(state):
    if state.whole is not None:
        return state.whole()
    for call in state.calls:
        call()
    return state.out


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how close results have to be
# ---------------------------------------------------------------------------
def _q4r(rows, K):
    return rows * (K // 32) * 18


def _pairs(n, prev, window):
    """Query-key pairs of a causal chunk."""
    return sum(min(prev + t + 1, window or (1 << 30)) for t in range(n))


def _model_work(case):
    """(bytes of the layers' weights and logits table, parameters, per layer (KV width, q width, full))."""
    H, I, layers, wb, par = case["H"], case["I"], [], 0, 0
    for i in range(case["layers"]):
        full = (i + 1) % 5 == 0
        D = case["gD"] if full and case["gD"] else case["D"]
        qd, kvd = case["nq"] * D, case["nkv"] * D
        layers.append((kvd, qd, full))
        for r, K in ((qd + 2 * kvd, H), (H, qd), (2 * I, H), (H, I)):
            wb += _q4r(r, K)
            par += r * K
    return wb, par, layers


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        M, K = case["M"], case["K"]
        return {"bytes": M * (K // 32) * 20 + 4 * (M + K), "flops": 2 * M * K}
    if kind == "ffn_decode":
        H, I = case["H"], case["I"]
        one = 3 * _q4r(I, H) + 4 * (5 * H + I) + ca.xplanes_bytes(I) + 4 * H
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 6 * H * I}
    if kind == "attn_decode":
        qd, kvd, S = case["nq"] * case["D"], case["nkv"] * case["D"], case["S"]
        return {"bytes": case["layers"] * 4 * (2 * S * kvd + 4 * kvd + 3 * qd + S),
                "flops": case["layers"] * 4 * S * qd}
    if kind == "logits":
        V, K = case["V"], case["K"]
        return {"bytes": V * (K // 32) * 36 + 4 * (V + K), "flops": 2 * V * K}
    if kind == "gemm_prefill":
        n, M, K = case["n"], case["M"], case["K"]
        return {"bytes": M * (K // 32) * 20 + 4 * n * (M + K), "flops": 2 * n * M * K}
    if kind == "mlp_prefill":
        n, H, I = case["n"], case["H"], case["I"]
        return {"bytes": 3 * _q4r(I, H) + 4 * n * (4 * H + I), "flops": 6 * n * H * I}
    if kind == "qkv_prefill":
        n, H, out = case["n"], case["H"], (case["nq"] + 2 * case["nkv"]) * case["D"]
        return {"bytes": _q4r(out, H) + 4 * n * (H + out), "flops": 2 * n * H * out}
    if kind == "attn_prefill":
        n, qd, kvd = case["n"], case["nq"] * case["D"], case["nkv"] * case["D"]
        keys = min(case["prev"] + n, (case["window"] or (1 << 30)) + n)
        return {"bytes": 4 * (2 * n * qd + 2 * keys * kvd), "flops": 4 * _pairs(n, case["prev"], case["window"]) * qd}
    wb, par, layers = _model_work(case)
    V, H = case["V"], case["H"]
    head = V * (H // 32) * 36 + 4 * V
    if kind == "prefill":
        n = case["n"]
        att = sum(4 * _pairs(n, 0, 0 if full else 1024) * qd for _, qd, full in layers)
        return {"bytes": wb + head + n * (4 * H + 8 * sum(k for k, _, _ in layers)),
                "flops": 2 * n * par + att + 2 * V * H}
    b = f = 0
    for i in range(case["tokens"]):
        c = case["clock"] + i + 1
        kv = sum(8 * (c if full else min(c, 512)) * k for k, _, full in layers)
        at = sum(4 * (c if full else min(c, 512)) * q for _, q, full in layers)
        b, f = b + wb + head + kv, f + 2 * par + 2 * V * H + at
    return {"bytes": b, "flops": f}


def tolerance(case):
    return TOLERANCE[case["kind"]]


# About four times the error measured against exact() (see the kinds above):
# 18-bit block fixed point and fp32 sums in the decode matvecs, 22 bits in the
# logits, fp32 attention (its softmax multiplies the error of the scores by
# their size), bf16 operands in the prefill contractions.
TOLERANCE = {
    "gemv": {"rel": 2e-5},            # measured 4e-6
    "ffn_decode": {"rel": 4e-5},      # 9e-6
    "attn_decode": {"rel": 4e-4},     # 9e-5: the fp32 rotation angle
    "logits": {"rel": 2e-6},          # 3e-7
    "gemm_prefill": {"rel": 1e-2},    # 2.4e-3
    "mlp_prefill": {"rel": 1.6e-2},   # 4.1e-3
    "qkv_prefill": {"rel": 1e-2},     # 2.4e-3
    "attn_prefill": {"rel": 2.4e-5},  # 6e-6: keys, values and probabilities in two bf16 parts
    "prefill": {"rel": 1.2e-2},       # 2.7e-3
    "decode": {"rel": 1.6e-3},        # 4e-4
}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _rms(x, w=None):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _rope(x, clocks, rot, theta):
    """Pairs (d, d + rot/2) of [tokens][heads][D] turned by the tokens' clocks."""
    half = rot // 2
    ang = clocks.double()[:, None, None] * theta ** (-2.0 * torch.arange(half, device="cuda").double() / rot)
    c, s, a, b = ang.cos(), ang.sin(), x[..., :half], x[..., half:rot]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., rot:]], -1)


def _attend(q, k, v, prev, window):
    """Causal attention of [n][nq][D] over [prev + n][nkv][D]."""
    n, nq, _ = q.shape
    gqa, at = nq // k.shape[1], torch.arange(k.shape[0], device="cuda")
    S = prev + 1 + torch.arange(n, device="cuda")
    seen = at[None, :] < S[:, None]
    if window:
        seen &= at[None, :] >= S[:, None] - window
    out = torch.empty_like(q)
    for h in range(nq):
        p = (q[:, h] @ k[:, h // gqa].T).masked_fill_(~seen, -math.inf).softmax(1)
        out[:, h] = p @ v[:, h // gqa]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        return _exact_model(case, seed)
    t = _inputs(case, seed)
    t = {n: v.double() if isinstance(v, torch.Tensor) and v.is_floating_point() else v for n, v in t.items()}
    if kind == "gemv":
        return _dequant_q4(t["W"][0]) @ t["x"]
    if kind == "ffn_decode":
        x, outs = t["x"], []
        for i in range(case["layers"]):
            W = _weights(case, seed, i)
            x = x + _rms(t["r"][i], t["post"][i].double())
            y = _rms(x, t["pre"][i].double())
            act = _gelu(_dequant_q4(W[0]) @ y) * (_dequant_q4(W[1]) @ y)
            outs += [x, act, _dequant_q4(W[2]) @ act]
        return outs
    if kind == "attn_decode":
        D, nq, nkv = case["D"], case["nq"], case["nkv"]
        slot, lst = _slot_of(case)
        clock, outs = torch.tensor([case["clock"]], device="cuda"), []
        for i in range(case["layers"]):
            head = lambda n, h: t[n][i].view(1, h, D)  # noqa: B023,E731
            kc, vc = t["kc"][i].double(), t["vc"][i].double()
            q = _rope(_rms(head("q", nq), t["qw"]), clock, D, THETA_FULL)
            kc[slot] = _rope(_rms(head("k", nkv), t["kw"]), clock, D, THETA_FULL).flatten()
            vc[slot] = _rms(head("v", nkv)).flatten()
            o = _attend(q, kc[lst].view(-1, nkv, D), vc[lst].view(-1, nkv, D), case["S"] - 1, 0)
            outs += [o.flatten(), kc, vc]
        return outs
    if kind == "logits":
        V, K = case["V"], case["K"]
        y = torch.cat([((c.double() * s[:, :, None]).flatten(1)) @ t["x"]
                       for c, s in zip(t["codes"].split(16384), t["scale"].split(16384))])
        return [y, (30 * torch.tanh(y / 30)).topk(64).values]
    if kind == "gemm_prefill":
        return t["X"] @ _dequant_q4(_weights(case, seed)[0]).T
    if kind == "mlp_prefill":
        W = _weights(case, seed)
        x = t["X"] + t["R"]
        y = _rms(x, t["nw"])
        act = _gelu(y @ _dequant_q4(W[0]).T) * (y @ _dequant_q4(W[1]).T)
        return [x, act, act @ _dequant_q4(W[2]).T]
    if kind == "qkv_prefill":
        n, D, nq, nkv = case["n"], case["D"], case["nq"], case["nkv"]
        y = _rms(t["X"], t["nw"])
        q, k, v = ((y @ _dequant_q4(W).T).view(n, -1, D) for W in _weights(case, seed))
        clocks = torch.arange(n, device="cuda") + case["clock"]
        kc, vc = torch.zeros((2, RING, nkv * D), dtype=torch.float64, device="cuda")
        at = clocks % WINDOW_SLOTS
        kc[at] = _rope(_rms(k, t["kw"]), clocks, case["rot"], THETA).flatten(1)
        vc[at] = _rms(v).flatten(1)
        return [_rope(_rms(q, t["qw"]), clocks, case["rot"], THETA).flatten(1), kc, vc]
    n, D, nq, nkv = case["n"], case["D"], case["nq"], case["nkv"]
    at = t["slots"].long()
    return _attend(t["q"].view(n, nq, D), t["kc"][at].view(-1, nkv, D), t["vc"][at].view(-1, nkv, D), case["prev"],
                   case["window"]).flatten(1)


# The synthetic model's generators, restated: splitmix64's output function
# over a counter (64-bit arithmetic wraps).
def _signed(v):
    return v - (1 << 64) if v >> 63 else v


def _mix64(seed, idx):
    def shr(z, k):
        return (z >> k) & ((1 << (64 - k)) - 1)
    z = (idx + 1) * _signed(0x9E3779B97F4A7C15) + _signed(seed & ((1 << 64) - 1))
    z = (z ^ shr(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ shr(z, 27)) * _signed(0x94D049BB133111EB)
    return z ^ shr(z, 31)


def _synth_q4(rows, K, seed):
    """float64 [rows][K]: uniform codes, f16 scales U(0.005, 0.02)."""
    blk = torch.arange(rows * (K // 32), device="cuda") * 3
    u = ((_mix64(seed, blk) >> 40) & 0xFFFFFF).double() / 16777216
    # one float32 fma: exact in 64 bits, then rounded
    scale = (u * float(np.float32(0.02) - np.float32(0.005)) + float(np.float32(0.005))).float().half().double()
    h = torch.stack([_mix64(seed, blk + 1), _mix64(seed, blk + 2)], 1)
    q = torch.stack([(h >> (4 * i)) & 15 for i in range(16)], 2).flatten(1)
    return ((q.double() - 8) * scale[:, None]).view(rows, K)


def _synth_embed(idx, seed):
    """bf16 N(0, 0.02) at the flat positions, as float32."""
    h = _mix64(seed, idx)
    u1 = (((h >> 40) & 0xFFFFFF).double() + 1) / 16777216
    u2 = ((h >> 16) & 0xFFFFFF).double() / 16777216
    z = (-2 * u1.log()).sqrt() * (6.283185307179586 * u2).cos()
    return (z * float(np.float32(0.02))).float().bfloat16().float()


def _exact_model(case, seed):
    wseed, tok, kp, vp = _model_inputs(case, seed)
    if case["kind"] == "decode" and case["tokens"] * case["layers"] > 480:
        return None
    H, I, V, nq = case["H"], case["I"], case["V"], case["nq"]
    cols = torch.arange(H, device="cuda")
    rows_of = lambda ids: _synth_embed(ids[:, None] * H + cols, wseed + 7)  # noqa: E731
    prefill = case["kind"] == "prefill"
    kc, vc = {}, {}

    def layers(x, clock):
        n = x.shape[0]
        clocks = torch.arange(n, device="cuda") + clock
        for i in range(case["layers"]):
            full = (i + 1) % 5 == 0
            D = case["gD"] if full and case["gD"] else case["D"]
            nkv, ls, theta = case["nkv"], wseed + 64 * (i + 1), THETA_FULL if full else THETA
            y = _rms(x)
            q, k, v = ((y @ _synth_q4(h * D, H, ls + j).T).view(n, h, D) for j, h in enumerate((nq, nkv, nkv)))
            q, k, v = _rope(_rms(q), clocks, D, theta), _rope(_rms(k), clocks, D, theta), _rms(v)
            if i not in kc:
                kc[i], vc[i] = ((torch.empty((0, nkv, D), dtype=torch.float64, device="cuda"),) * 2 if prefill else
                                (kp[i].double().view(-1, nkv, D), vp[i].double().view(-1, nkv, D)))
            kc[i], vc[i] = torch.cat([kc[i], k]), torch.cat([vc[i], v])
            window = 0 if full else (1024 if prefill else 512)
            a = _attend(q, kc[i], vc[i], clock, window).flatten(1)
            x = x + _rms(a @ _synth_q4(H, nq * D, ls + 3).T)
            y = _rms(x)
            act = _gelu(y @ _synth_q4(I, H, ls + 4).T) * (y @ _synth_q4(I, H, ls + 5).T)
            x = x + _rms(act @ _synth_q4(H, I, ls + 6).T)
        return _rms(x[-1])

    def logits(y):
        out = []
        for r0 in range(0, V, 16384):
            r = torch.arange(r0, min(V, r0 + 16384), device="cuda")
            w = rows_of(r).view(len(r), H // 32, 32)
            amax = w.abs().amax(2, keepdim=True)
            q = w * (127 / amax)
            q = torch.trunc(q + 0.5 * q.sign()).clamp(-128, 127)     # halves away from zero
            out.append((q.double() * (amax / 127).double()).flatten(1) @ y)
        return torch.cat(out)

    scale = math.sqrt(H)
    if prefill:
        y = logits(layers(rows_of(tok).double() * scale, 0))
        return [y, (30 * torch.tanh(y / 30)).topk(64).values]
    y = None
    for i in range(case["tokens"]):
        y = logits(layers(rows_of(tok).double() * scale, case["clock"] + i))
        tok = y.argmax().view(1)
    return [None, y]
