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
