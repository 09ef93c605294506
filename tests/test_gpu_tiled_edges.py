"""The tiled family's tile epilogues at the edges of their 128 x 128 wave
tiles: scores and P go through the GEMM's LDS stages in whole lines, so rows
past the last token, unit columns past the padded row and waves with no unit
at all must neither be stored nor counted; one k block (64 wide) takes the
score loads from the GEMM's prologue.  Against the CPU oracle
(models/dawn_spatial_v41_exp.py:415-635) at the family's own bar.
"""

from __future__ import annotations

import pytest

from oracle import srw_ref
from tests.test_gpu_mfma import _check, _gpu, _inputs, _oracle

pytestmark = pytest.mark.gpu

CASES = [
    # T, D, dr, N, max_chunk, seed
    (1, 64, 64, 33, 12500, 61),      # one k block, one token, half a padded row
    (257, 192, 64, 257, 12500, 62),  # one row and one unit into the next tiles
    (127, 576, 192, 385, 150, 63),   # odd k blocks, the second wave column one unit wide, three chunks
    (129, 320, 320, 128, 12500, 64),  # a wave column with no unit
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "T{}D{}dr{}N{}c{}".format(*c[:5]))
def test_tiled_tile_edges(pkg, dev, case):
    T, D, dr, N, max_chunk, seed = case
    print(f"[gpu] tiled edges {case}", flush=True)
    inp = _inputs(pkg, T, D, dr, N, dr == D, seed)
    _, cs = srw_ref.chunk_plan(N, max_chunk)
    got = _gpu(pkg, dev, inp, cs, tiled=True)
    assert got["path"] == "tiled_bf16"
    ref, tr = _oracle(inp, max_chunk)
    _check(got, ref, tr, T, N, D)
