"""GPU: SRW_FLAG_DIAG on the tiled-GEMM family -- the drop-in's forward at the
widths the fused kernels do not take -- against the scalar kernels
(models/dawn_spatial_v41_exp.py:434-552).

Counts use thresholds on the sigmoid's argument (the exact inverse of the act
thresholds) and a score may round to the neighbouring bf16 value under another
fp32 order, so counts agree to 2 + 1e-3 N; sums to what those scores move
(power sums: 2% of sum k |s|^(k-1) ulp(s), at least two scores)."""

from __future__ import annotations

import pytest
import torch

from oracle import srw_ref
from tests.parity import bf16_ulp, rel_fro
from tests.test_gpu_mfma import _diag_scores

pytestmark = pytest.mark.gpu

BF = torch.bfloat16
CASES = [
    # T, D, dr, N, routes, max_chunk, seed
    (1, 192, 64, 33, 1, 12500, 1),        # one row, a unit past one lane's four
    (33, 384, 384, 256, 1, 12500, 2),     # h other than x at the fused widths; one whole slice
    (48, 1024, 256, 1030, 1, 515, 3),     # two chunks, a slice of six units
    (97, 640, 128, 511, 2, 12500, 4),     # paired rows, ragged rows and units
    (130, 128, 128, 48, 1, 24, 5),        # chunks shorter than a 32-unit tile
]


def _call(pkg, dev, case, **kw):
    T, D, dr, N, R, max_chunk, seed = case
    inp = pkg.inputs.make_pool_inputs(pkg.inputs.PoolShape(T=T, D=D, N=N, dr=dr, routes=R), seed=seed)
    inp["tau_offset"].uniform_(-0.9, 0.3, generator=torch.Generator().manual_seed(seed))
    _, cs = srw_ref.chunk_plan(N, max_chunk)
    args = [inp[k].to(BF).to(dev) for k in ("x", "h", "emb")] + [inp["tau_offset"].to(dev)] + \
           [inp[k].to(BF).to(dev) for k in ("read", "write")]
    return inp, args, cs


@pytest.mark.parametrize("case", CASES, ids=lambda c: "T{}D{}dr{}N{}R{}c{}".format(*c[:6]))
def test_tiled_diagnostics_match_generic(pkg, dev, case):
    T, D, dr, N, R, _, _ = case
    print(f"[gpu] tiled diagnostics {case}", flush=True)
    inp, args, cs = _call(pkg, dev, case)
    fast = pkg.srw_forward(*args, chunk_size=cs, diag=True, tiled=True)
    slow = pkg.srw_forward(*args, chunk_size=cs, diag=True, emulate=True)
    torch.cuda.synchronize()
    assert fast["path"] == "tiled_bf16" and slow["path"] == "generic"
    f = {k: v.cpu() for k, v in fast.items() if isinstance(v, torch.Tensor)}
    g = {k: v.cpu() for k, v in slow.items() if isinstance(v, torch.Tensor)}
    assert rel_fro(f["out"].float(), g["out"].float()) <= 5e-3
    assert torch.allclose(f["den"], g["den"], rtol=2e-4)
    assert torch.allclose(f["gate_sum"], g["gate_sum"], rtol=2e-3, atol=1e-6)
    assert int((f["n_active"] - g["n_active"]).abs().max()) <= 2
    col = pkg._capi.TDIAG_INDEX
    td_f, td_g = f["token_diag"], g["token_diag"]
    sc = _diag_scores(inp, False, R)
    # a score that rounds the other way moves the mean by its ulp / N and the
    # std by at most |s - mean| / std (below 5 here) times that, tau by their
    # sum; at most two such scores a row
    flip = 2 * 6 * float(bf16_ulp(sc.abs().max())) / N
    for n in ("s_mean", "s_std", "tau"):
        assert torch.allclose(td_f[..., col[n]], td_g[..., col[n]], rtol=1e-4, atol=1e-5 + flip), n
    for k, n in ((3, "sum_s3"), (4, "sum_s4")):
        each = k * sc.abs() ** (k - 1) * bf16_ulp(sc)  # what one score that rounds the other way moves
        sens = each.sum(dim=-1).reshape(td_g[..., 0].shape)
        bound = 0.02 * sens + 2 * each.amax(dim=-1).reshape(sens.shape) + 1e-5 * (sc.abs() ** k).sum(dim=-1).reshape(sens.shape)
        assert ((td_f[..., col[n]] - td_g[..., col[n]]).abs() <= bound).all(), n
    for n in ("gate_max", "int_max", "int_sum"):
        assert torch.allclose(td_f[..., col[n]], td_g[..., col[n]], rtol=2e-3, atol=1e-6), n
    m = sc.reshape(T, R, N) - td_g[..., col["tau"]][..., None] - 0.5
    gt = torch.sigmoid(500.0 * m) * (1e-4 + torch.clamp(m - 0.01, 0.0, 10.0))
    mag = (gt * torch.log(gt + 1e-8)).abs().sum(dim=-1)
    d = (td_f[..., col["g_log_g"]] - td_g[..., col["g_log_g"]]).abs()
    assert (d <= 1e-3 + 2e-3 * td_g[..., col["g_log_g"]].abs() + 1e-4 * mag).all()
    for n in ("n_strong", "n_boundary", "n_band075", "n_band030", "n_int_cap"):
        assert ((td_f[..., col[n]] - td_g[..., col[n]]).abs() <= 2 + 1e-3 * N).all(), n
    assert torch.allclose(f["unit_diag"][:, 0], g["unit_diag"][:, 0], rtol=1e-3, atol=1e-3 * (T * R) ** 0.5)
    assert torch.allclose(f["unit_diag"][:, 1], g["unit_diag"][:, 1], rtol=2e-3, atol=1e-6)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "T{}D{}dr{}N{}R{}c{}".format(*c[:6]))
def test_tiled_diagnostics_round_out_once(pkg, dev, case):
    """out is as exact as the scalar kernels': the chunks' sums are not rounded
    to bf16 before the division.  What is left against them is the order of
    the fp32 sums, which moves an element to the neighbouring bf16 value now
    and then, and gates of scores that round the other way; a second rounding
    of every element is 2^-9 / sqrt(3) rms or more over a binade, 1.1e-3."""
    print(f"[gpu] tiled diagnostics, rounding {case}", flush=True)
    _, args, cs = _call(pkg, dev, case)
    outs = []
    for general in (False, True):
        plan = pkg.SrwPlan(*args, chunk_size=cs, diag=True, tiled=True)
        if general:
            plan._desc.flags |= pkg._capi.SRW_FLAG_NO_FAST
        plan.launch()
        outs.append(plan.out.float().cpu())
        assert plan.path == ("generic" if general else "tiled_bf16")
    assert rel_fro(outs[0], outs[1]) <= 1e-3


def test_diagnostics_kept_on_generic(pkg, dev):
    """What the tiled diagnostics do not cover keeps the scalar kernels: gate
    constants under which gate and intensity are not non-decreasing in the
    score, centred statistics, the dense gate output."""
    _, args, _ = _call(pkg, dev, CASES[1])
    print("[gpu] diagnostics on the generic kernels", flush=True)
    for kw in (dict(consts=pkg.GateConfig(sharpness=-500.0)), dict(consts=pkg.GateConfig(epsilon=-1e-4)),
               dict(stats="centered"), dict(want_gate=True)):
        assert pkg.srw_forward(*args, diag=True, **kw)["path"] == "generic", kw


def test_noalloc_diagnostics_beyond_the_scratch(pkg, dev):
    """srw_forward_noalloc with diagnostics whose tiled workspace exceeds the
    library's scratch runs on the generic kernels, which need none: its results
    are srw_forward's under SRW_FLAG_NO_FAST bit for bit (the units' score sums
    come from atomics in no fixed order: to rounding)."""
    import ctypes
    C = pkg._capi
    T, D, dr, N = 8, 1024, 64, 33000  # W^T alone is 68 MB
    _, args, _ = _call(pkg, dev, (T, D, dr, N, 1, 40000, 6))
    print("[gpu] noalloc diagnostics", flush=True)
    plan = pkg.SrwPlan(*args, diag=True)
    assert plan.ws_bytes > 64 << 20
    plan.launch()
    assert plan.path == "tiled_bf16"
    keys = ("out", "gate_sum", "den", "n_active", "pass_mask", "token_diag", "unit_diag")
    plan._desc.flags |= C.SRW_FLAG_NO_FAST
    plan.launch()
    assert plan.path == "generic"
    torch.cuda.synchronize()
    want = {k: getattr(plan, k).clone() for k in keys}
    plan._desc.flags &= ~C.SRW_FLAG_NO_FAST
    for k in keys:
        getattr(plan, k).fill_(-7)
    C.check(plan._lib.srw_forward_noalloc(ctypes.byref(plan._desc), ctypes.byref(plan._tens), ctypes.byref(plan._outs),
                                          ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    assert C.last_path() == "generic"
    for k in keys[:-1]:
        assert torch.equal(getattr(plan, k), want[k]), k
    assert torch.equal(plan.unit_diag[:, 1], want["unit_diag"][:, 1])
    # eight scores a unit, in any order: seven additions of at most the sum of their sizes
    inp_s = (args[1][:, 0].float() @ args[2].float().T).abs().sum(0)
    assert ((plan.unit_diag[:, 0] - want["unit_diag"][:, 0]).abs() <= 7 * 2.0 ** -24 * 1.01 * inp_s).all()


def test_plan_with_h_equal_x_holds_its_own_workspace(pkg, dev):
    """With diagnostics at d_route == d_model, h == x runs on the fused kernels:
    its plan does not allocate the tiled family's larger workspace."""
    _, args, cs = _call(pkg, dev, (2048, 384, 384, 2600, 1, 2600, 7))
    print("[gpu] diagnostics plan, h == x", flush=True)
    same = pkg.SrwPlan(args[0], args[0], *args[2:], chunk_size=cs, diag=True)
    other = pkg.SrwPlan(*args, chunk_size=cs, diag=True)
    for p in (same, other):
        p.launch()
    assert same.path.startswith("mfma") and other.path == "tiled_bf16"
    assert same.ws_bytes < other.ws_bytes == pkg._capi.workspace_size(same._desc)
