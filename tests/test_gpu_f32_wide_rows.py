"""GPU: fp32 calls whose rows have elements of very different size, against
the layer in float64 (models/dawn_spatial_v41_exp.py:1713-1738).

One channel of x (or of h) is 2^16 to 2^24 where the pool's rows are zero, so
every product's value comes from the elements far below it: an operand held in
24 bits per element keeps them whatever the large one is, one held relative to
its row's largest element does not.  The thresholds lie so low that every unit
passes with a margin of several, where the gate is linear in the score.

Bar: 1e-6.  A product of K = 384 fp32 terms is within 2.5e-7 of its norm
(192 chained additions of two), the write product of 300 units 2.2e-7, a
score (K = 128) 1.4e-7 of a gate of about its own size, the threshold's and
the quotient's roundings 6e-8 each: 4e-7 together."""

from __future__ import annotations

import math

import pytest
import torch

from tests.parity import rel_fro

pytestmark = pytest.mark.gpu

BAR = 1e-6


def _inputs(dev, T, D, dr, N, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    r, w = rn(N, D), rn(N, D)
    r, w = r / r.norm(dim=-1, keepdim=True), w / w.norm(dim=-1, keepdim=True)
    return [rn(T, D), rn(T, 1, dr), rn(N, dr) / math.sqrt(dr), torch.full((T, 1), -6.0, device=dev), r, w]


def _want(args):
    x, h, e, off, r, w = (t.double() for t in args)
    s = h[:, 0] @ e.T
    mean = s.mean(-1, keepdim=True)
    std = ((s - mean) ** 2).mean(-1, keepdim=True).sqrt() + 1e-8
    m = s - (mean + off * std) - 0.5
    inten = 1e-4 + (m - 0.01).clamp(0.0, 10.0)
    den = inten.sum(-1, keepdim=True).clamp_min(1.0)
    return (torch.sigmoid(500.0 * m) * inten * (x @ r.T)) @ w / den


@pytest.mark.parametrize("power", [0, 16, 20, 24])
@pytest.mark.parametrize("where", ["x", "h"])
def test_rows_with_one_large_channel(pkg, dev, where, power):
    print(f"[gpu] f32 wide rows {where} 2^{power}", flush=True)
    args = _inputs(dev, 300, 384, 128, 300, 11)
    if power:
        a, b = (args[0], args[4]) if where == "x" else (args[1][:, 0], args[2])
        a[:, 5] = 2.0 ** power
        b[:, 5] = 0.0
    got = pkg.srw_forward(*args, stats="centered")
    torch.cuda.synchronize()
    assert got["path"] == "tiled_f32"
    err = rel_fro(got["out"][:, 0].cpu(), _want(args).cpu())
    print(f"  rel err {err:.2e}", flush=True)
    assert err <= BAR
