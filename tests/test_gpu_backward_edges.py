"""GPU: the backward's gradient products, whose operands with k as rows are
read transposed out of LDS, at the edges of their 64-k blocks and 256 / 192
column tiles (models/dawn_spatial_v41_exp.py:415-635 under jax.value_and_grad),
against the oracle's VJP: every gradient within the backward's 2e-2."""

from __future__ import annotations

import pytest
import torch

from oracle import srw_ref, srw_vjp
from tests.parity import rel_fro

pytestmark = pytest.mark.gpu

BF = torch.bfloat16
CASES = [
    # T, D, dr, N, seed
    (1, 64, 64, 33, 1),        # one row, less than a block of either k
    (64, 384, 384, 64, 2),     # whole blocks
    (65, 384, 128, 257, 3),    # one row, one unit past a tile
    (127, 256, 64, 191, 4),    # one short of a block; D of one 256-wide tile
    (130, 192, 192, 700, 5),   # one 192-wide tile
    (90, 1024, 320, 130, 6),   # four 256-wide tiles, a 64-column remainder of the route
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "T{}D{}dr{}N{}".format(*c[:4]))
def test_gradients_at_block_edges(pkg, dev, case):
    T, D, dr, N, seed = case
    print(f"[gpu] backward edges {case}", flush=True)
    inp = pkg.inputs.make_pool_inputs(pkg.inputs.PoolShape(T=T, D=D, N=N, dr=dr), seed=seed)
    inp["tau_offset"].uniform_(-0.9, 0.3, generator=torch.Generator().manual_seed(seed))
    x, e, r, w = (inp[k].to(BF) for k in ("x", "emb", "read", "write"))
    h, tau = inp["h"].to(BF), inp["tau_offset"]
    d_out = torch.randn(T, 1, D, generator=torch.Generator().manual_seed(seed + 9))
    ref = srw_ref.fused_gate_srw(x.float()[None], h[:, 0].float()[None], e.float(), tau[None], r.float(), w.float(),
                                 max_chunk_size=40000)
    out = ref[0].reshape(T, 1, D).to(BF)
    # gradients into sentinels: columns and rows past an array are not written
    g = pkg.srw_backward(*(t.to(dev) for t in (x, h, e, tau, r, w, out, d_out)), 0.5, 0.25)
    torch.cuda.synchronize()
    v = srw_vjp.fused_gate_srw_vjp(x.float(), h[:, 0].float(), e.float(), tau, r.float(), w.float(), d_out[:, 0], 0.5,
                                   0.25, max_chunk_size=40000)
    for k in ("dx", "dh", "demb", "dread", "dwrite"):
        err = rel_fro(g[k].cpu().reshape(v[k].shape), v[k])
        print(f"  {k}: {err:.2e}", flush=True)
        assert err <= 2e-2, k


def test_infinite_last_row_stays_in_its_place(pkg, dev):
    """A non-finite last token or unit meets only its own gradients' products:
    the rows past the last are zeros, not copies of it."""
    T, D, N = 65, 128, 100
    print("[gpu] backward, infinite last rows", flush=True)
    inp = pkg.inputs.make_pool_inputs(pkg.inputs.PoolShape(T=T, D=D, N=N, dr=64), seed=8)
    t = [inp[k].to(BF).to(dev) for k in ("x", "h", "emb")] + [inp["tau_offset"].to(dev)] + \
        [inp[k].to(BF).to(dev) for k in ("read", "write")]
    t[0][-1, 3] = float("inf")
    out = torch.zeros(T, 1, D, dtype=BF, device=dev)
    g = pkg.srw_backward(*t, out, torch.ones(T, 1, D, device=dev))
    torch.cuda.synchronize()
    assert torch.isfinite(g["dx"][:-1]).all() and torch.isfinite(g["dh"][:-1]).all()
    keep = torch.arange(D, device=dev) != 3
    assert torch.isfinite(g["dread"][:, keep]).all()    # x.r is infinite in P and dP.x, not in d(xr)
