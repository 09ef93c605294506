"""GPU: srw_diag_summary (the result tuple's values in two launches) against
the torch form of the same formulas in float64 (srw._diag_tuple,
srw._diag_tuple_v401: models/dawn_spatial_v41_exp.py:588-635, 862-907), and
srw_cast_bf16 against torch's casts, bit for bit.

Per-token values are float32 quotients (a few ulp); scalars are sums in double
of float32 terms, rounded once: 1e-6 relative, beside the 1e-6 absolute that
skew and kurtosis (differences of moments) lose in their columns' scale."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [
    # B, S, N, routes, gate
    (1, 1, 33, 1, "v41"),           # one row, one workgroup each
    (3, 171, 257, 2, "v41"),        # a unit past one workgroup, averaged routes
    (1, 33001, 64, 1, "v41"),       # more rows than 128 workgroups' first pass
    (2, 100, 40001, 2, "v41"),      # more units than 128 workgroups' first pass
    (2, 129, 300, 1, "gelu_v401"),
    (1, 257, 511, 2, "gelu_v401"),
]


def _plan(pkg, dev, B, S, N, R, gate):
    T, D = B * S, 64
    bf = dict(dtype=torch.bfloat16, device=dev)
    return pkg.SrwPlan(torch.zeros(T, D, **bf), torch.zeros(T, R, D, **bf), torch.zeros(N, D, **bf),
                       torch.zeros(T, R, device=dev), torch.zeros(N, D, **bf), torch.zeros(N, D, **bf),
                       gate=gate, diag=True, want_mask=False)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}S{}N{}R{}{}".format(*c))
def test_summary_matches_torch_form(pkg, dev, case):
    from dawn_srw_amd import srw
    B, S, N, R, gate = case
    print(f"[gpu] diag summary {case}", flush=True)
    plan = _plan(pkg, dev, B, S, N, R, gate)
    g = torch.Generator(device=dev).manual_seed(B + S + N)
    td = plan.token_diag
    td.uniform_(0.5, 2.0, generator=g)
    td[..., 3:5] = N * td[..., 3:5]                     # power sums
    td[..., 7:11] = torch.randint(0, N + 1, td[..., 7:11].shape, generator=g, device=dev).float()
    td[..., 11] -= 1.0                                  # sum g log g: either sign
    plan.gate_sum.uniform_(0.0, 5.0, generator=g)
    plan.gate_sum[0] = 0.0                              # the entropy's guard
    plan.n_active.random_(0, N + 1, generator=g)
    plan.n_active[-1] = 0                               # the quotients' guards
    plan.unit_diag.normal_(generator=g)                 # negative mean scores, dead units among them
    if gate == "v41":
        got = srw._fused_diag(plan, N, B, S, R, 0.01, False)
    else:
        got = srw._fused_diag(plan, N, B, S, R, 0.0, True)
    res = {k: (v.double().cpu() if torch.is_tensor(v) and v.is_floating_point() else v)
           for k, v in plan.results().items()}
    res["n_active"] = plan.n_active.cpu()
    # the torch form widens n_active to float32; counts are exact there
    want = srw._diag_tuple(res, N, B, S, R, 0.01) if gate == "v41" else srw._diag_tuple_v401(res, N, B, S, R)
    assert len(got) == len(want)
    for i, (a, b) in enumerate(zip(got, want)):
        assert a.shape == b.shape and a.dtype == torch.float32, i
        assert torch.allclose(a.cpu().double(), b.double(), rtol=2e-6, atol=1e-6), (i, a.flatten()[:4], b.flatten()[:4])


def test_summary_keeps_nan(pkg, dev):
    from dawn_srw_amd import srw
    plan = _plan(pkg, dev, 2, 130, 300, 1, "v41")
    for t in (plan.token_diag, plan.gate_sum, plan.unit_diag):
        t.fill_(1.0)
    plan.n_active.fill_(1)
    plan.token_diag[259, 0, 12] = float("nan")          # int_max of the last row
    plan.unit_diag[299, 0] = float("nan")
    got = srw._fused_diag(plan, 300, 2, 130, 1, 0.01, False)
    print("[gpu] diag summary nan", flush=True)
    assert torch.isnan(got[19]) and torch.isnan(got[2]) and torch.isnan(got[17])
    assert not torch.isnan(got[13])


@pytest.mark.parametrize("gate,R", [("v41", 1), ("v41", 2), ("gelu_v401", 2)])
def test_summary_of_infinities(pkg, dev, gate, R):
    """An infinity or NaN in any column comes out where the torch form gives
    one (relu(inf) times a dead unit's 0 among them), and nowhere else."""
    from dawn_srw_amd import srw
    B, S, N = 1, 70, 60
    print(f"[gpu] diag summary infinities {gate} R{R}", flush=True)
    v401 = gate != "v41"
    for v in (float("inf"), float("-inf"), float("nan")):
        for name, at in ([("token_diag", (33, 0, k)) for k in range(14)] + [("gate_sum", (33, 0))]
                         + [("unit_diag", (u, k)) for u in (7, 8) for k in (0, 1)]):
            plan = _plan(pkg, dev, B, S, N, R, gate)
            g = torch.Generator(device=dev).manual_seed(5)
            plan.token_diag.uniform_(0.5, 2.0, generator=g)
            plan.gate_sum.uniform_(0.5, 5.0, generator=g)
            plan.n_active.random_(1, N + 1, generator=g)
            plan.unit_diag.normal_(generator=g)
            plan.unit_diag[7, 1], plan.unit_diag[8, 1] = 0.0, 1.0  # a dead unit and one that is not
            getattr(plan, name)[at] = v
            res = plan.results()
            want = srw._diag_tuple_v401(res, N, B, S, R) if v401 else srw._diag_tuple(res, N, B, S, R, 0.01)
            got = srw._fused_diag(plan, N, B, S, R, 0.0 if v401 else 0.01, v401)
            for i, (a, b) in enumerate(zip(got, want)):
                assert torch.equal(torch.isnan(a), torch.isnan(b)), (v, name, at, i, a.flatten()[:1], b.flatten()[:1])
                inf = torch.isinf(b)
                assert torch.equal(torch.isinf(a), inf) and torch.equal(a[inf], b[inf]), (v, name, at, i)


def test_cast_bf16_bit_equal(pkg, dev):
    from dawn_srw_amd import layer
    g = torch.Generator(device=dev).manual_seed(3)
    big = torch.randn(70001, generator=g, device=dev)
    big[:5] = torch.tensor([float("inf"), float("-inf"), 3.3e38, 1e-40, -0.0], device=dev)
    ts = [big, big[1:], big[4:4 + 2048], torch.empty(0, 8, device=dev), big[:3],
          torch.randn(33, 65, generator=g, device=dev).t(), big[:7].double(), big[:9].bfloat16(),
          torch.randn(5, 5, generator=g, device=dev), big[2:2053], big[8:16]]
    print("[gpu] cast_bf16", flush=True)
    got = layer.cast_bf16(ts, dev)
    for a, t in zip(got, ts):
        assert a.dtype == torch.bfloat16 and a.is_contiguous()
        assert torch.equal(a, t.to(torch.bfloat16).contiguous())
    nan = layer.cast_bf16([torch.full((20,), float("nan"), device=dev)], dev)[0]
    assert torch.isnan(nan).all()
