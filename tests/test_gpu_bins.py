"""FP32 K2 + Kf over the whole range of bin counts, against the same samples in FP64."""

import pytest
import torch

from nlo_bk_optimized_amd import device as dev
from nlo_bk_optimized_amd.bk import MV, BKConfig
from nlo_bk_optimized_amd.bk.evolution import uniform_edges

pytestmark = pytest.mark.gpu
NODES = 24


def workload():
    r = (1e-6 * torch.pow(torch.tensor((100.0 / 1e-6) ** (1 / (NODES - 1)), dtype=torch.float64),
                          torch.arange(NODES, dtype=torch.float64))).cuda()
    return r, MV(qs0sqr=0.2).dipole_amplitude(r)


def close(got, want, bound):
    assert bool(torch.isfinite(got).all()) and float(want.norm()) > 0
    assert float((got - want).norm() / want.norm()) < bound


# The volume factor grows with the fourth power of the number of bins: the
# smallest, both sides of 2^128 at the former scale, the largest.
# An FP32 sample is good to about 50 eps (its kernels, splines and Jacobian),
# the norm over parents to a few 1e-6; 1e-4 leaves room for a single sample
# that carries a sum.
@pytest.mark.parametrize("bins", [2, 50, 217, 218, 255])
def test_fp32_sums_and_histograms(bins):
    r, N = workload()
    t64, t32 = dev.spline_build(r, N)
    config = BKConfig(RPOINTS=NODES - 1, MAXR=100.0, MC_BINS=bins)
    edges, table = uniform_edges(NODES, bins, r.device), dev.sobol_table(4, 3)

    def run(precision, **kwargs):
        return dev.bk_nlo(r, N, t64, t32, edges, table, 1 << 16, config, precision=precision, **kwargs)

    want, want_hist, want_count = run("fp64_stable", histogram=True)
    got, hist, count = run("fp32", histogram=True)
    close(got[:, 0], want[:, 0], 1e-4)
    assert torch.equal(count, want_count)
    close(hist, want_hist, 1e-4)
    close(run("fp32", sum_only=True)[0][:, 0], want[:, 0], 1e-4)


@pytest.mark.parametrize("bins", [2, 217, 218, 255])
def test_fp32_steps(bins):
    r, N = workload()
    config = BKConfig(RPOINTS=NODES - 1, MAXR=100.0, MC_BINS=bins)
    edges, table = uniform_edges(NODES, bins, r.device), dev.sobol_table(4, 3)
    change = {}
    for precision in ("fp32", "fp64_stable"):
        ev = dev.Evolver(r, edges, table, config, n_samples=1 << 16, precision=precision, rk_method="euler", step=0.1,
                         k1_rule="fixed")
        ev.state.copy_(N)
        ev.step()
        change[precision] = ev.state - N
    close(change["fp32"], change["fp64_stable"], 1e-4)
    batch = dev.BatchEvolver(torch.cat([r, r]), torch.cat([edges, edges]), [NODES, NODES], table, config,
                             n_samples=1 << 16, precision="fp32", rk_method="euler", step=0.1, k1_rule="fixed")
    batch.state.copy_(torch.cat([N, N]))
    batch.step()
    close(batch.state - torch.cat([N, N]), change["fp64_stable"].repeat(2), 1e-4)


# An angular bin across theta = pi is not folded: its half-angles reach beyond
# pi/2 and the difference of two of them beyond pi, the further the wider the
# bin and the more the grids of the two angles differ.
@pytest.mark.parametrize("first,second", [([0, 0.3, 1], [0, 0.55, 1]), ([0, 0.45, 0.98, 1], [0, 0.3, 0.52, 1])])
def test_fp32_angles_in_wide_bins(first, second):
    r, N = workload()
    t64, t32 = dev.spline_build(r, N)
    bins = len(first) - 1
    config = BKConfig(RPOINTS=NODES - 1, MAXR=100.0, MC_BINS=bins)
    edges, table = uniform_edges(NODES, bins, r.device), dev.sobol_table(4, 3)
    for d, e in ((2, first), (3, second)):
        edges[:, d] = torch.tensor(e, dtype=torch.float64, device=r.device)

    def run(precision):
        return dev.bk_nlo(r, N, t64, t32, edges, table, 1 << 16, config, precision=precision)[0][:, 0]

    # FP32's own error of these sums is 5e-7, the unfolded difference gave 1e-5 to 2e-5
    close(run("fp32"), run("fp64_stable"), 2e-6)
