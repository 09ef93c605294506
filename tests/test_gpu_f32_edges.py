"""GPU: the fp32 tiled family against the layer in float64
(models/dawn_spatial_v41_exp.py:1713-1738), at the edges of its tiles (256
units x 64 tokens, 128-unit moments, 32-wide lines) and of the operands'
ranges.

Bar: 1e-5 relative, the fp32 path's, for the output; every row by its own norm
to 2e-4, or to what the roundings of a score do to it: a row without a passing
unit (gates of 1e-4 and less) has its largest gates at margins where the gate
moves by the slope 500 times the score's error.  That is a chain of K / 2
additions at partial sums of about |h| |e| / sqrt(K), sqrt(64) 2^-25 = 2^-22 of
them at K = 128; the worst of some thousand scores lies within four times that."""

from __future__ import annotations

import math

import pytest
import torch

from tests.parity import REL_F32, gate_close, rel_fro, unpack_mask

pytestmark = pytest.mark.gpu

CASES = [
    # T, D, dr, N, routes, stats, gate, seed
    (256, 128, 128, 33, 1, "centered", "v41", 1),       # half a unit tile's moments empty
    (257, 160, 192, 300, 1, "centered", "v41", 2),      # a token past a tile, an odd unit tile
    (300, 384, 128, 511, 1, "onepass", "v41", 3),
    (200, 384, 384, 1030, 2, "centered", "v41", 4),     # paired rows
    (400, 256, 1152, 640, 1, "centered", "v41", 5),     # long score rows, one unit tile past the second
    (270, 128, 128, 385, 1, "centered", "gelu_v401", 6),
]


def _inputs(case, dev):
    T, D, dr, N, R, _, _, seed = case
    g = torch.Generator(device=dev).manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    x, h, e = rn(T, D), rn(T, R, dr), rn(N, dr) / math.sqrt(dr)
    r, w = rn(N, D), rn(N, D)
    r, w = r / r.norm(dim=-1, keepdim=True), w / w.norm(dim=-1, keepdim=True)
    off = torch.empty(T, R, device=dev).uniform_(-0.9, 1.5, generator=g)
    off[::7] = 8.0                                      # rows without a passing unit
    return [x, h, e, off, r, w]


def _want(args, gate="v41"):
    x, h, e, off, r, w = (t.double() for t in args)
    outs, margins, sizes = [], [], []
    for j in range(h.shape[1]):
        s = h[:, j] @ e.T
        mean = s.mean(-1, keepdim=True)
        std = ((s - mean) ** 2).mean(-1, keepdim=True).sqrt() + 1e-8
        raw = s - (mean + off[:, j:j + 1] * std)
        if gate == "v41":
            m = raw - 0.5
            inten = 1e-4 + (m - 0.01).clamp(0.0, 10.0)
            gt, den = torch.sigmoid(500.0 * m) * inten, inten.sum(-1, keepdim=True).clamp_min(1.0)
            rr, ww = r, w
        else:
            m = raw
            z = raw / std
            gt = torch.where(z > 0, z * 0.5 * (1 + torch.erf(z / math.sqrt(2))), torch.zeros_like(z))
            den = gt.sum(-1, keepdim=True).clamp_min(1.0)
            rr, ww = (t / (t.norm(dim=-1, keepdim=True) + 1e-8) for t in (r, w))
        outs.append((gt * (x @ rr.T)) @ ww / den)
        margins.append(m)
        sizes.append(h[:, j].norm(dim=-1) * e.norm(dim=-1).max() / math.sqrt(e.shape[1]))
    return torch.stack(outs, 1), torch.stack(margins, 1), torch.stack(sizes, 1)


def _check(got, want, margin, size, N, what=""):
    err = rel_fro(got["out"].cpu(), want.cpu())
    num, norm = (got["out"].double() - want).norm(dim=-1), want.norm(dim=-1)
    # every row by its own norm, but rows whose gates (and so norm) lie 1e-25
    # below the others': an fp32 gate leaves its normal range at 1e-38
    big = norm > 1e-25 * norm.max()
    row, bar = num[big] / norm[big], (500.0 * 2.0 ** -20 * size[big]).clamp_min(20 * REL_F32)
    print(f"  {what} rel err {err:.2e}, worst row {row.max().item():.2e}", flush=True)
    assert err <= REL_F32 and (row <= bar).all()
    clear = margin.abs() > 1e-5
    mask = unpack_mask(got["pass_mask"], N).to(margin.device)
    assert torch.equal(mask[clear], (margin > 0)[clear])


@pytest.mark.parametrize("case", CASES, ids=lambda c: "T{}D{}dr{}N{}R{}{}{}".format(*c[:7]))
def test_edges_match_float64(pkg, dev, case):
    T, D, dr, N, R, stats, gate, _ = case
    print(f"[gpu] f32 edges {case}", flush=True)
    args = _inputs(case, dev)
    got = pkg.srw_forward(*args, stats=stats, gate=gate)
    torch.cuda.synchronize()
    assert got["path"] == "tiled_f32"
    _check(got, *_want(args, gate), N)


def test_operand_ranges(pkg, dev):
    """Scales far from one, rows of zeros, units 2^20 apart and elements far
    below their row's largest."""
    case = (260, 128, 128, 200, 1, "centered", "v41", 7)
    print("[gpu] f32 edges ranges", flush=True)
    for name, f, g in (("small", 2.0 ** -20, 1.0), ("large", 2.0 ** 20, 1.0), ("units", 1.0, 4.0),
                       ("apart", 1.0, 2.0 ** 20), ("out", 2.0 ** 40, 1.0)):
        args = _inputs(case, dev)
        args[0] *= f
        args[4] /= f
        args[5] *= f
        args[4][::3] *= g
        args[5][1::3] /= g
        args[0][5] = 0.0
        args[4][7] = 0.0
        args[5][9] = 0.0
        args[0][11, 1:] *= 1e-6
        got = pkg.srw_forward(*args, stats="centered")
        torch.cuda.synchronize()
        _check(got, *_want(args), 200, name)


def test_infinities_match_generic(pkg, dev):
    """An infinity or NaN in any operand gives what products of fp32 numbers
    give, on a fresh pool and on a cached one, and leaves the other rows and
    the next call as they were."""
    case = (256, 128, 128, 140, 1, "centered", "v41", 8)
    print("[gpu] f32 edges infinities", flush=True)
    inf, nan = float("inf"), float("nan")
    for k, at, v in ((0, (3, 5), inf), (1, (4, 0, 7), nan), (2, (9, 1), -inf), (4, (100, 127), inf), (5, (0, 0), nan),
                     (3, (6, 0), inf), (3, (7, 0), -inf), (3, (8, 0), nan)):
        args = _inputs(case, dev)
        args[k][at] = v
        got = pkg.srw_forward(*args, stats="centered")["out"]
        ref = pkg.srw_forward(*args, stats="centered", force_generic=True)["out"]
        torch.cuda.synchronize()
        assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref)), k
        ok = torch.isfinite(ref)
        assert torch.equal(got[torch.isinf(ref)], ref[torch.isinf(ref)])
        if ok.any():
            assert rel_fro(got[ok].cpu(), ref[ok].cpu()) <= REL_F32
    args = _inputs(case, dev)
    plan = pkg.SrwPlan(*args, stats="centered")
    plan.launch()
    first = plan.out.clone()
    keep = args[0].clone()
    args[0][3, 5] = inf
    plan.launch(pool_cached=True)
    bad = plan.out.clone()
    args[0].copy_(keep)
    plan.launch(pool_cached=True)
    torch.cuda.synchronize()
    ref_rows = torch.arange(256, device=dev) != 3
    assert not torch.isfinite(bad[3]).any() and rel_fro(bad[ref_rows].cpu(), first[ref_rows].cpu()) <= REL_F32
    assert torch.equal(plan.out, first)


def test_dense_gate(pkg, dev):
    case = (256, 128, 128, 300, 1, "centered", "v41", 9)
    print("[gpu] f32 edges dense gate", flush=True)
    args = _inputs(case, dev)
    a = pkg.srw_forward(*args, stats="centered", want_gate=True)
    b = pkg.srw_forward(*args, stats="centered", want_gate=True, force_generic=True)
    torch.cuda.synchronize()
    assert a["path"] == "tiled_f32"
    ok, _ = gate_close(a["gate"][:, 0].cpu(), b["gate"][:, 0].cpu(), args[1][:, 0].cpu(), args[2].cpu())
    assert ok


def test_noalloc_equals_forward(pkg, dev):
    """A call whose workspace just fits the no-allocation scratch is accepted
    and equal to srw_forward's bit for bit."""
    import ctypes
    C = pkg._capi
    T, D, N = 400, 384, 7000
    print("[gpu] f32 edges noalloc", flush=True)
    args = _inputs((T, D, D, N, 1, "centered", "v41", 10), dev)
    plan = pkg.SrwPlan(*args, stats="centered")
    assert plan.ws_bytes <= C.NOALLOC_SCRATCH_BYTES
    plan.launch()
    want = plan.out.clone()
    plan.out.zero_()
    C.check(plan._lib.srw_forward_noalloc(ctypes.byref(plan._desc), ctypes.byref(plan._tens), ctypes.byref(plan._outs),
                                          ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    assert torch.equal(plan.out, want)
