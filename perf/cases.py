"""Performance cases: the calls that a user of this package makes, with sizes
from the repository's own configurations (the 40M model's QK, V and Know
pools, the scaled Know pool) and the ranges around them.

A case is a dict of plain values; ``kind`` names the entry point:

* ``forward``   one bound ``SrwPlan`` call (bf16), the layer's forward;
* ``pools``     the QK (two routes) and V pools of one attention layer as one
                ``SrwBatchPlan`` call;
* ``train``     ``make_sharded_srw`` / ``_paired`` / ``_v401`` on float32
                tensors, forward and backward;
* ``inference`` ``srw_inference``, float32 end to end;
* ``model_forward`` / ``model_prefill`` / ``model_decode``: ``DawnModel``.
"""

import math

import torch

import __graft_entry__

srw = __graft_entry__.load_package()

DEV = "cuda:0"
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
MAX_CHUNK = 12500          # the N-chunk that the training script passes
LB_WEIGHT, DEAD_WEIGHT = 0.01, 0.01
VOCAB, LAYERS, HEADS, MAX_SEQ = 32000, 12, 6, 512
N_QK, N_V, N_KNOW, D40, DR40 = 1580, 2600, 25200, 384, 128


def listed():
    return [
        # the Know pool's forward over 8 x 512 tokens: the package's headline call
        dict(name="know_forward", kind="forward", T=4096, D=384, dr=384, N=25200, gate="v41", stats="onepass",
             tau=-0.5, cached=False),
        # the QK and V pools of one attention layer over the same tokens
        dict(name="attention_forward", kind="pools", T=4096, D=384, dr=384, NQK=1580, NV=2600, stats="onepass",
             cached=False),
        # the scaled Know pool: a wide layer with 2% of its units passing, the largest call
        dict(name="wide_forward", kind="forward", T=16384, D=1024, dr=1024, N=100000, gate="v41", stats="onepass",
             tau=1.55, cached=False),
        # one training step through the Know pool
        dict(name="know_train", kind="train", B=8, S=512, R=1, D=384, dr=384, N=25200, gate="v41", tau=-0.5),
        # one training step through the QK pool, both routes, behind the model's router width
        dict(name="qk_train", kind="train", B=8, S=512, R=2, D=384, dr=128, N=1580, gate="v41", tau=-0.5),
        # the legacy v4.0.1 layer's training step on the same pool as know_train
        dict(name="v401_train", kind="train", B=8, S=512, R=1, D=384, dr=384, N=25200, gate="gelu_v401", tau=-0.5),
        # a training step of a wider model's layer, ragged in tokens and units
        dict(name="wide_train", kind="train", B=4, S=509, R=1, D=1024, dr=256, N=20011, gate="v41", tau=0.5),
        # float32 inference through the Know pool
        dict(name="know_inference_f32", kind="inference", T=4096, D=384, dr=384, N=25200, tau=-0.5),
        # decoding 64 sequences: the Know pool call of one layer, 3% of the units passing
        dict(name="decode_know", kind="forward", T=64, D=384, dr=128, N=25200, gate="v41", stats="centered",
             tau=1.38, cached=True),
        # decoding one sequence: the QK and V calls of one layer, the smallest call
        dict(name="decode_attention", kind="pools", T=1, D=384, dr=128, NQK=1580, NV=2600, stats="centered",
             cached=True),
        # the 40M model's forward over 8 sequences (evaluation)
        dict(name="model_forward", kind="model_forward", B=8, S=512),
        # one decode step of the 40M model for 64 sequences, 300 positions in the cache
        dict(name="model_decode", kind="model_decode", B=64, S=300),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """Another case of the listed ranges: other token and unit counts (odd
    ones among them), widths, routes, gates and pass rates."""
    kind = rng.choice(["forward", "forward", "pools", "train", "train", "inference", "decode", "model_forward",
                       "model_prefill", "model_decode"])
    if kind == "forward":
        D, dr = rng.choice([(384, 384), (384, 128), (128, 128), (1024, 1024), (1024, 256)])
        return dict(kind="forward", T=_log_int(rng, 200, 12000), D=D, dr=dr, N=_log_int(rng, 600, 40000),
                    gate="gelu_v401" if D < 1024 and rng.random() < 0.2 else "v41",
                    stats=rng.choice(["onepass", "centered"]), tau=round(rng.uniform(-0.5, 1.5), 2), cached=False)
    if kind == "decode":
        if rng.random() < 0.5:
            return dict(kind="forward", T=_log_int(rng, 1, 128), D=384, dr=128, N=_log_int(rng, 1000, 30000),
                        gate="v41", stats="centered", tau=round(rng.uniform(-0.5, 1.5), 2), cached=True)
        return dict(kind="pools", T=_log_int(rng, 1, 64), D=384, dr=128, NQK=_log_int(rng, 500, 4000),
                    NV=_log_int(rng, 500, 6000), stats="centered", cached=True)
    if kind == "pools":
        return dict(kind="pools", T=_log_int(rng, 200, 8000), D=384, dr=rng.choice([128, 384]),
                    NQK=_log_int(rng, 500, 4000), NV=_log_int(rng, 500, 6000), stats="onepass", cached=False)
    if kind == "train":
        R = rng.choice([1, 1, 2])
        if R == 2:
            D, dr, N, gate = 384, 128, _log_int(rng, 500, 6000), rng.choice(["v41", "v41", "gelu_v401"])
        else:
            D, dr = rng.choice([(384, 384), (384, 128), (128, 64), (1024, 256)])
            N = _log_int(rng, 1000, 18000 if D == 1024 else 30000)
            gate = "v41" if D == 1024 else rng.choice(["v41", "v41", "gelu_v401"])
        return dict(kind="train", B=rng.randint(1, 4 if D == 1024 else 8), S=rng.randint(64, 500), R=R, D=D, dr=dr,
                    N=N, gate=gate, tau=round(rng.uniform(-0.5, 1.0), 2))
    if kind == "inference":
        D, dr = rng.choice([(384, 384), (384, 128), (1024, 256)])
        return dict(kind="inference", T=_log_int(rng, 64, 4000), D=D, dr=dr, N=_log_int(rng, 600, 25000),
                    tau=round(rng.uniform(-0.5, 1.5), 2))
    if kind == "model_decode":
        return dict(kind=kind, B=_log_int(rng, 1, 96), S=rng.randint(1, 500))
    return dict(kind=kind, B=rng.randint(1, 8), S=rng.randint(17, 500))


# -- inputs -------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _rms_rows(t):
    return t / torch.sqrt(torch.mean(t * t, dim=-1, keepdim=True) + 1e-6)


def _unit_rows(g, n, d):
    t = torch.randn(n, d, generator=g, device=DEV)
    return t / torch.linalg.vector_norm(t, dim=-1, keepdim=True)


def _pool(g, T, R, D, dr, N, tau, dtype):
    """The repository's synthetic pool inputs: RMS-normalised x, E ~ N(0, 1/dr),
    unit read and write rows; h is x itself where the score reads x."""
    e = (torch.randn(N, dr, generator=g, device=DEV) / math.sqrt(dr)).to(dtype)
    r, w = _unit_rows(g, N, D).to(dtype), _unit_rows(g, N, D).to(dtype)
    x = _rms_rows(torch.randn(T, D, generator=g, device=DEV)).to(dtype)
    if R == 1 and dr == D:
        h = x
    else:
        h = _rms_rows(torch.randn(T, R, dr, generator=g, device=DEV)).to(dtype)
    off = tau + 0.05 * torch.randn(T, R, generator=g, device=DEV)
    return x, h, e, off, r, w


def _model(seed):
    cfg = srw.DawnConfig(vocab_size=VOCAB, d_model=D40, n_layers=LAYERS, n_heads=HEADS, max_seq_len=MAX_SEQ,
                         d_route=DR40, n_qk=N_QK, n_v=N_V, n_know=N_KNOW, max_chunk_size=MAX_CHUNK)
    return cfg, srw.init_params(cfg, seed)


def _caches(g, B, S):
    """Keys and values of S positions, as unit-normal as the scaled pools'
    outputs are, zero behind them."""
    out = []
    for _ in range(2):
        c = torch.zeros(LAYERS, B, HEADS, MAX_SEQ, D40 // HEADS, device=DEV)
        c[:, :, :, :S] = 0.5 * torch.randn(LAYERS, B, HEADS, S, D40 // HEADS, generator=g, device=DEV)
        out.append(c)
    return out


def _inputs(case, seed):
    g, k = _gen(seed), case["kind"]
    if k == "forward":
        return _pool(g, case["T"], 1, case["D"], case["dr"], case["N"], case["tau"], BF16)
    if k == "pools":
        qk = _pool(g, case["T"], 2, case["D"], case["dr"], case["NQK"], -0.5, BF16)
        v = _pool(g, case["T"], 1, case["D"], case["dr"], case["NV"], -0.5, BF16)
        x = qk[0]  # both pools read the layer's one input
        return qk, (x, x if v[1] is v[0] else v[1]) + v[2:]
    if k == "train":
        x, h, e, off, r, w = _pool(g, case["B"] * case["S"], case["R"], case["D"], case["dr"], case["N"],
                                   case["tau"], F32)
        B, S, R = case["B"], case["S"], case["R"]
        lead = (B, S) if R == 1 else (B, S, 2)
        xs = x.reshape(B, S, -1)
        hs = xs if h is x else h.reshape(*lead, -1)
        d_out = torch.randn(*lead, case["D"], generator=g, device=DEV)
        return xs, hs, e, off.reshape(*lead, 1), r, w, d_out
    if k == "inference":
        x, h, e, off, r, w = _pool(g, case["T"], 1, case["D"], case["dr"], case["N"], case["tau"], F32)
        return x, h.reshape(case["T"], -1), e, off, r, w
    if k == "model_decode":
        ids = torch.randint(0, VOCAB, (case["B"],), generator=g, device=DEV)
        return (ids, *_caches(g, case["B"], case["S"]))
    return (torch.randint(0, VOCAB, (case["B"], case["S"]), generator=g, device=DEV),)


def _chunk(N, stats):
    return srw.chunk_plan(N, MAX_CHUNK)[1] if stats == "onepass" else 0


def prepare(case, seed):
    k, inp = case["kind"], _inputs(case, seed)
    if k == "forward":
        plan = srw.SrwPlan(*inp, gate=case["gate"], stats=case["stats"], chunk_size=_chunk(case["N"], case["stats"]))
        if case["cached"]:  # a decode loop: the pool was packed by an earlier step
            plan.launch()
        return dict(kind=k, cached=case["cached"], plan=plan)
    if k == "pools":
        qk, v = inp
        plans = [srw.SrwPlan(*qk, stats=case["stats"], chunk_size=_chunk(case["NQK"], case["stats"])),
                 srw.SrwPlan(*v, stats=case["stats"], chunk_size=_chunk(case["NV"], case["stats"]))]
        batch = srw.SrwBatchPlan(plans)
        if case["cached"]:
            batch.launch()
        return dict(kind=k, cached=case["cached"], batch=batch)
    if k == "train":
        x, h, e, off, r, w, d_out = inp
        if case["gate"] == "v41":
            make = srw.make_sharded_srw if case["R"] == 1 else srw.make_sharded_srw_paired
        else:
            make = srw.make_sharded_srw_v401 if case["R"] == 1 else srw.make_sharded_srw_paired_v401
        leaves = [t.requires_grad_(True) for t in ((x, e, off, r, w) if h is x else (x, h, e, off, r, w))]
        return dict(kind=k, gate=case["gate"], fused=make(None, max_chunk_size=MAX_CHUNK), args=(x, h, e, off, r, w),
                    leaves=leaves, d_out=d_out, d_lb=torch.tensor(LB_WEIGHT, device=DEV),
                    d_dead=torch.tensor(DEAD_WEIGHT, device=DEV))
    if k == "inference":
        return dict(kind=k, args=inp)
    cfg, params = _model(seed)
    return dict(kind=k, model=srw.DawnModel(params, cfg, DEV), inp=inp, S=case["S"])


def run(state):
    k = state["kind"]
    if k == "forward":
        plan = state["plan"]
        plan.launch(pool_cached=state["cached"])
        return _plan_out(plan)
    if k == "pools":
        state["batch"].launch(pool_cached=state["cached"])
        return [_plan_out(p) for p in state["batch"].plans]
    if k == "train":
        res = state["fused"](*state["args"])
        if state["gate"] == "v41":  # the terms of the training loss: out, score_lb, dead_penalty
            terms, cot = (res[0], res[3], res[18]), (state["d_out"], state["d_lb"], state["d_dead"])
        else:
            terms, cot = (res[0], res[3]), (state["d_out"], state["d_lb"])
        grads = torch.autograd.grad(terms, state["leaves"], cot)
        # with the diagnostics that a training loop logs (score_skew and score_kurt are differences of
        # nearly equal moments and hold no digits to compare)
        names = dict(active_frac=1, gate_max=2, score_std=4, gate_sum=5, active_n=6, strong_frac=7, boundary_frac=8,
                     z_mean_active=9, tau_mean=10, z_lt_075=11, z_lt_030=12, entropy=15)
        return dict(terms=[t.detach() for t in terms], grads=list(grads),
                    diag={n: res[i].detach() for n, i in names.items() if i < len(res)})
    if k == "inference":
        return srw.srw_inference(*state["args"])
    if k == "model_forward":
        return state["model"].forward(*state["inp"])
    if k == "model_prefill":
        logits, cK, cV, _ = state["model"].prefill(*state["inp"])
        return logits, cK, cV
    logits, cK, cV, _ = state["model"].decode_step(*state["inp"], state["S"])
    return logits, cK, cV


def _plan_out(p):
    return dict(out=p.out, gate_sum=p.gate_sum, den=p.den, n_active=p.n_active, pass_mask=p.pass_mask)


# -- what a pass cannot do without ----------------------------------------------

def _layer_work(T, R, D, dr, N, size, h_is_x=False):
    flops = 2.0 * T * N * (R * dr + D + R * D)  # score, read (shared by the routes), write
    b = size * (N * (dr + 2 * D) + T * D + (0 if h_is_x else T * R * dr) + T * R * D) + 4 * T * R
    return dict(bytes=float(b), flops=flops)


def work(case):
    k = case["kind"]
    if k in ("forward", "inference"):
        size = 2 if k == "forward" else 4
        w = _layer_work(case["T"], 1, case["D"], case["dr"], case["N"], size, case["dr"] == case["D"])
        if k == "forward":
            w["bytes"] += case["T"] * (12 + 8 * ((case["N"] + 63) // 64))
        return w
    if k == "pools":
        a = _layer_work(case["T"], 2, case["D"], case["dr"], case["NQK"], 2)
        b = _layer_work(case["T"], 1, case["D"], case["dr"], case["NV"], 2, case["dr"] == case["D"])
        masks = case["T"] * (36 + 8 * (2 * ((case["NQK"] + 63) // 64) + (case["NV"] + 63) // 64))
        return dict(bytes=a["bytes"] + b["bytes"] + masks, flops=a["flops"] + b["flops"])
    if k == "train":
        T = case["B"] * case["S"]
        w = _layer_work(T, case["R"], case["D"], case["dr"], case["N"], 4, case["R"] == 1 and case["dr"] == case["D"])
        # backward: two products for each of the forward's (the inputs and their gradients once more)
        return dict(bytes=2.0 * w["bytes"] + 4.0 * T * case["R"] * case["D"], flops=3.0 * w["flops"])
    T = case["B"] * (1 if k == "model_decode" else case["S"])
    layer = [_layer_work(T, 2, D40, DR40, N_QK, 2), _layer_work(T, 1, D40, DR40, N_V, 2),
             _layer_work(T, 1, D40, DR40, N_KNOW, 2)]
    flops = LAYERS * (sum(w["flops"] for w in layer) + 2.0 * T * D40 * (4 * DR40 + 4 + D40))
    keys = case["S"] + 1 if k == "model_decode" else case["S"] / 2
    flops += LAYERS * 4.0 * T * keys * D40 + 2.0 * T * D40 * VOCAB
    pools = 2.0 * (N_QK + N_V + N_KNOW) * (DR40 + 2 * D40)  # the layers share them
    b = pools + 4.0 * (VOCAB * D40 + T * VOCAB) + LAYERS * 4.0 * D40 * (D40 + 4)
    if k == "model_decode":
        b += LAYERS * 8.0 * case["B"] * (case["S"] + 1) * D40
    if k == "model_prefill":
        b += LAYERS * 8.0 * case["B"] * MAX_SEQ * D40
    return dict(bytes=b, flops=flops)


def tolerance(case):
    k = case["kind"]
    if k == "inference":  # measured 9e-7 from 64 bits
        return {"rel": 1e-5}
    # bf16 scores, gates and products: a sum in another order moves a score to
    # the neighbouring bf16 value, and with it counts of single units (2e-3 to
    # 8e-3 from 64 bits, whole models 4e-3)
    if k.startswith("model"):
        return {"rel": 1e-2, "max": 0.4}
    return {"rel": 1e-2, "max": 0.4, "differ": 0.01}


# -- the same in 64 bits ----------------------------------------------------------

class _RoundScores(torch.autograd.Function):
    """The layer's scores are bf16 numbers by definition (a threshold reads
    them); their gradient passes through."""

    @staticmethod
    def forward(ctx, s):
        return s.to(BF16).to(F64)

    @staticmethod
    def backward(ctx, g):
        return g


def _layer64(x, h, e, off, r, w, gate, round_scores, full=False):
    """One route's layer in float64: x [T, D], h [T, dr], off [T, 1]."""
    s = h @ e.T
    if round_scores:
        s = _RoundScores.apply(s)
    mean = s.mean(-1, keepdim=True)
    std = torch.sqrt(((s - mean) ** 2).mean(-1, keepdim=True)) + 1e-8
    raw = s - (mean + off * std)
    if gate == "v41":
        m = raw - 0.5
        inten = 1e-4 + torch.clamp(m - 0.01, 0.0, 10.0)
        g = torch.sigmoid(500.0 * m) * inten
        den = torch.clamp_min(inten.sum(-1, keepdim=True), 1.0)
    else:
        r = r / (torch.linalg.vector_norm(r, dim=-1, keepdim=True) + 1e-8)
        w = w / (torch.linalg.vector_norm(w, dim=-1, keepdim=True) + 1e-8)
        z = raw / std
        g = torch.where(z > 0, z * (0.5 * (1.0 + torch.erf(z / math.sqrt(2.0)))), torch.zeros((), dtype=F64, device=DEV))
        den = torch.clamp_min(g.sum(-1, keepdim=True), 1.0)
    out = ((g * (x @ r.T)) @ w) / den
    if not full:
        return out, g.sum(-1, keepdim=True), den
    return out, g.sum(-1, keepdim=True), den, s, std


def _in64(*ts):
    """The values that the layer reads: its operands are bf16."""
    return [t.to(BF16).to(F64) for t in ts]


def _rows(T, N):
    return max(1, min(T, int(2e8 // N)))


def _forward64(x, h, e, off, r, w, gate, round_scores, dtype):
    """(out [T, R, D], gate_sum, den [T, R]) of h [T, R, dr] or x itself."""
    cast = _in64 if dtype == BF16 else (lambda *ts: [t.to(F64) for t in ts])
    hh = x[:, None] if h is x else h
    e, r, w = cast(e, r, w)
    outs, step = [], _rows(x.shape[0], e.shape[0])
    for a in range(0, x.shape[0], step):
        b = a + step
        got = [_layer64(*cast(x[a:b], hh[a:b, j]), e, off[a:b, j:j + 1].to(F64), r, w, gate, round_scores)
               for j in range(hh.shape[1])]
        outs.append([torch.stack([g[i] for g in got], 1) for i in range(3)])
    return [torch.cat([o[i] for o in outs]) for i in range(3)]


def _plan64(inp, gate="v41"):
    out, gs, den = _forward64(*inp, gate, True, BF16)
    return dict(out=out, gate_sum=gs[..., 0], den=den[..., 0], n_active=None, pass_mask=None)


def _train64(case, inp):
    x, h, e, off, r, w, d_out = inp
    T, R = case["B"] * case["S"], case["R"]
    same = h is x
    x2, e2, r2, w2 = (t.requires_grad_(True) for t in _in64(x.reshape(T, -1), e, r, w))
    h2 = x2 if same else _in64(h.reshape(T * R, -1))[0].requires_grad_(True)
    o2 = off.reshape(T * R, 1).to(F64).requires_grad_(True)
    hs, os_ = h2.reshape(T, R, -1), o2.reshape(T, R, 1)
    got = [_layer64(x2, hs[:, j], e2, os_[:, j], r2, w2, case["gate"], True, full=True) for j in range(R)]
    out = torch.stack([g[0] for g in got], 1)
    unit = sum(g[3].mean(0) for g in got) / R
    mean = unit.mean()
    var = (unit ** 2).mean() - mean ** 2
    lb = var / (mean ** 2 + var + 1e-2)
    leaves = [x2, e2, o2, r2, w2] if same else [x2, h2, e2, o2, r2, w2]
    loss = (out.reshape(d_out.shape) * d_out.to(F64)).sum() + LB_WEIGHT * lb
    grads = torch.autograd.grad(loss, leaves)
    want = [x, e, off, r, w] if same else [x, h, e, off, r, w]
    grads = [g.reshape(t.shape) for g, t in zip(grads, want)]
    terms = [out.detach().reshape(d_out.shape), lb.detach()] + ([None] if case["gate"] == "v41" else [])
    std = torch.stack([g[4].detach() for g in got]).mean()
    gsum = torch.stack([g[1].detach() for g in got]).mean()
    return dict(terms=terms, grads=grads, diag=dict(score_std=std, gate_sum=gsum))


def _ln64(x, p):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + 1e-6) * p["scale"] + p["bias"]


def _attend64(q, k, v, mask):
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    if mask is not None:
        s = s.masked_fill(~mask, float("-inf"))
    return torch.matmul(torch.softmax(s, -1), v)


def _model64(case, seed):
    k, inp = case["kind"], _inputs(case, seed)
    cfg, params = _model(seed)
    p = _to64(params)
    rt, pool = p["router"], p["neuron_pool"]
    B, S = case["B"], 1 if k == "model_decode" else case["S"]
    pos0 = case["S"] if k == "model_decode" else 0
    T, H, dh, dr = B * S, HEADS, D40 // HEADS, DR40
    x = (p["token_emb"]["embedding"][inp[0].reshape(B, S)] + p["pos_emb"]["embedding"][pos0:pos0 + S][None])
    x = x.reshape(T, D40)
    cK = torch.zeros(LAYERS, B, H, MAX_SEQ, dh, dtype=F64, device=DEV)
    cV = torch.zeros_like(cK)
    if k == "model_decode":
        cK.copy_(inp[1])
        cV.copy_(inp[2])
    mask = torch.ones(S, S, dtype=torch.bool, device=DEV).tril() if S > 1 else None

    def call(name, n, h, off):
        out = _forward64(n, h, pool[name + "_emb"], off, pool[name + "_read"], pool[name + "_write"], "v41", True, BF16)
        return out[0] * pool[name + "_scale"]

    def heads(t):
        return t.reshape(B, S, H, dh).transpose(1, 2)

    for i in range(LAYERS):
        bp = p["block_%d" % i]
        n = _ln64(x, bp["norm1"])
        h_all = n @ rt["proj_attn"]["kernel"] + rt["proj_attn"]["bias"]
        t_all = n @ rt["tau_attn"]["kernel"] + rt["tau_attn"]["bias"]
        qk = call("qk", n, h_all[:, :2 * dr].reshape(T, 2, dr), t_all[:, :2])
        v = call("v", n, h_all[:, 2 * dr:].reshape(T, 1, dr), t_all[:, 2:])
        q, kk, v = heads(qk[:, 0]), heads(qk[:, 1]), heads(v[:, 0])
        cK[i, :, :, pos0:pos0 + S], cV[i, :, :, pos0:pos0 + S] = kk, v
        a = _attend64(q, cK[i, :, :, :pos0 + S], cV[i, :, :, :pos0 + S], mask)
        x = x + a.transpose(1, 2).reshape(T, D40) @ bp["attn"]["expand_O"]["kernel"]
        n = _ln64(x, bp["norm2"])
        h = n @ rt["proj_know"]["kernel"] + rt["proj_know"]["bias"]
        x = x + call("know", n, h.reshape(T, 1, dr), n @ rt["tau_know"]["kernel"] + rt["tau_know"]["bias"])[:, 0]
    logits = _ln64(x, p["norm"]) @ p["token_emb"]["embedding"].T
    if k == "model_forward":
        return logits.reshape(B, S, VOCAB)
    if k == "model_prefill":
        return logits.reshape(B, S, VOCAB), cK, cV
    return logits, cK, cV


def _to64(t):
    return {k: _to64(v) for k, v in t.items()} if isinstance(t, dict) else t.to(DEV, F64)


def exact(case, seed):
    """What run() returns, in float64 plain torch: the operands that the layer
    rounds to bf16 (its inputs and its scores) rounded, nothing else."""
    k = case["kind"]
    with torch.no_grad() if k != "train" else torch.enable_grad():
        if k.startswith("model"):
            return _model64(case, seed)
        inp = _inputs(case, seed)
        if k == "forward":
            return _plan64(inp, case["gate"])
        if k == "pools":
            return [_plan64(p) for p in inp]
        if k == "train":
            return _train64(case, inp)
        x, h, e, off, r, w = inp
        return _forward64(x, x if h.data_ptr() == x.data_ptr() else h[:, None], e, off, r, w, "v41", False, F32)[0][:, 0]
