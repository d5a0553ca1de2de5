"""The K2 + Kf sums do not depend on the order in which a block's Sobol points
are handed to the lanes: one launch over n points against the sum of launches
over 64 points each (which always run in the sequence's own order)."""

import pytest
import torch

from nlo_bk_optimized_amd import device as dev
from nlo_bk_optimized_amd.bk import MV, BKConfig
from nlo_bk_optimized_amd.bk.evolution import uniform_edges

pytestmark = pytest.mark.gpu


# below a block, one block, whole blocks, blocks and a ragged rest (the border
# between both orders inside a launch), a first index that blocks do not divide
@pytest.mark.parametrize("precision", ["fp32", "fp64", "fp64_stable"])
@pytest.mark.parametrize("first,n", [(0, 37), (0, 128), (0, 4096), (0, 4096 * 3), (0, 10_000), (0, 16_411),
                                     (4096, 8192), (192, 5000)])
def test_sums_do_not_depend_on_the_order(precision, first, n):
    config = BKConfig(RPOINTS=11, MAXR=50.0)
    r = (1e-6 * torch.pow(torch.tensor((50.0 / 1e-6) ** (1 / 11), dtype=torch.float64),
                          torch.arange(12, dtype=torch.float64))).cuda()
    N = MV(qs0sqr=0.2).dipole_amplitude(r)
    t64, t32 = dev.spline_build(r, N)
    edges = uniform_edges(12, 50, r.device)
    table = dev.sobol_table(4, 5)

    def sums(at, count):
        return dev.bk_nlo(r, N, t64, t32, edges, table, count, config, first_index=at, precision=precision)[0]

    whole = sums(first, n)
    pieces = torch.stack([sums(first + k, min(64, n - k)) for k in range(0, n, 64)])
    # every sample is the same number in both; the pair-wise compensated sums
    # leave one rounding per block partial and per piece
    bound = 4 * torch.finfo(torch.float64).eps * pieces.abs().sum(0).clamp_min(1e-300)
    assert bool(((whole - pieces.sum(0)).abs() <= bound * max(1, n // 64) ** 0.5 + bound).all())
