"""GPU: the backward's elementwise work with a token's row held in a
workgroup's registers, at the edges of its splits (units per row: 2 048, 4 096,
8 192, 12 288, 20 480, 28 672 for one route, the first four for two; longer
rows take the two-pass kernels), v4.1 and v4.0.1, with and without the
forward's residuals, against the oracle's gradients (within 2e-2, the
backward's bar: bf16 products rounded as the oracle rounds them)."""

from __future__ import annotations

import pytest

from tests.test_gpu_backward import test_backward_paired_matches_oracle as paired_v41
from tests.test_gpu_backward_edges import test_gradients_at_block_edges as single_v41
from tests.test_gpu_backward_v401 import test_v401_backward_matches_oracle_autograd as any_v401

pytestmark = pytest.mark.gpu

ONE = [63, 2048, 2049, 4097, 8193, 12289, 20481, 28672, 28673]
TWO = [2048, 2049, 4097, 8193, 12288, 12289]


@pytest.mark.parametrize("N", ONE)
def test_one_route(pkg, dev, N):
    single_v41(pkg, dev, (5, 64, 64, N, N))


@pytest.mark.parametrize("N", TWO)
def test_two_routes(pkg, dev, N):
    paired_v41(pkg, dev, (3, 64, 64, N, N))


@pytest.mark.parametrize("residuals", [False, True], ids=["recompute", "residuals"])
@pytest.mark.parametrize("R,N", [(1, 2049), (1, 20480), (1, 28673), (2, 2049), (2, 12288), (2, 12289)])
def test_v401(pkg, dev, R, N, residuals):
    any_v401(pkg, dev, (4, 128, 64, N, False, R, N, 40000), residuals)
