"""Batched DIS integration (nlo_dis_batch_run) on the GPU.

* One VEGAS integral in a batch equals the host-driven per-iteration driver
  (numerics.integration.vegas_device: one nlo_dis_vegas pass and one
  nlo_vegas_adapt per iteration, statistics on the host) at the same Sobol
  indices to 1e-12 relative (value and error; the block partition of the
  sums differs, so not bit for bit), with the same evaluation count and
  convergence decision.
* Points batched together equal the points run alone, bit for bit (each
  integral keeps its own plan), for GBW and for a BK-table dipole (whose LO
  term initialises the interpolation).
* The six qqbar-g integrals at the reference's benchmark point (GBW Qs0^2 = 1,
  lambda = 0.3, Q^2 = 9, x = 1e-3, charm m = 1.4, maxr = 5) against its
  20-worker C++ values with their errors
  (T/benchmarks/dis_fixed_sobol_all_qg.py:69-76).
"""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from nlo_bk_optimized_amd import device

    return device


def _gbw():
    from nlo_bk_optimized_amd.dipole import GBW

    return GBW(Qs0sqr=1.0, lambda_=0.3, gamma=1.0, x0=1.0)


@pytest.mark.parametrize("kind,precision,quark_mass,transverse", [
    ("T1", "fp64", 1.4, True), ("T2", "fp32", 0.14, True), ("ab", "fp32", 0.14, False),
    ("cd", "fp64", 1.27, False), ("I1", "fp32", 1.4, True), ("I2_nested", "fp32", 1.27, False),
    ("I3_nested", "fp32", 0.14, True), ("I2", "fp64", 1.4, True), ("I3", "fp64", 1.4, False),
])
def test_batch_item_equals_host_driven_vegas(dev, kind, precision, quark_mass, transverse):
    from nlo_bk_optimized_amd import _lib
    from nlo_bk_optimized_amd.dis.config import DISConfig, Quark, QuarkType
    from nlo_bk_optimized_amd.numerics.integration import vegas_device

    cfg = DISConfig(quarks=(Quark(QuarkType.C, quark_mass),), maxr=5.0)
    desc = dev.dis_desc(9.0, 1e-3, transverse, cfg.quarks, _gbw(), cfg)
    seed, samples, iters = 17, 3 * 4096 + 100, 5
    print(f"batch item {kind} {precision} m={quark_mass} T={transverse}", flush=True)
    want = vegas_device(desc, kind, samples_per_iteration=samples, max_iterations=iters, min_iterations=3,
                        bins=cfg.bins, epsrel=1e-9, seed=seed, precision=precision, first_index=128)
    item = _lib.DisItem()
    item.desc = desc
    item.contribution = _lib.DIS_KINDS[kind]
    item.method = _lib.NLO_DIS_METHOD_VEGAS
    item.n = samples
    item.sobol_table = 0
    item.max_iterations, item.min_iterations = iters, 3
    item.first_index = 128
    got = dev.dis_batch([item], [dev.sobol_table(_lib.DIS_DIMENSIONS[kind], seed)], bins=cfg.bins,
                        precision=precision, epsrel=1e-9, device="cuda").cpu()[0]
    assert float(got[0]) == pytest.approx(float(want.value), rel=1e-12, abs=0)
    assert float(got[1]) == pytest.approx(float(want.error), rel=1e-10, abs=0)
    assert int(got[2]) == want.n_eval and bool(got[3]) == want.converged


# Blocks of 256, 512 and 1024 samples stage them for tiles of 2048, blocks of
# 2048 are a tile: below, at and above a block, a tile and each change of the
# block size (512 blocks: 2^18, 2^19, 2^20), and a ragged last tile; all in one
# batch, so that one launch of a kind holds both sorts of blocks.
def test_batch_histogram_tiles(dev):
    from nlo_bk_optimized_amd import _lib
    from nlo_bk_optimized_amd.dis.config import DISConfig, Quark, QuarkType
    from nlo_bk_optimized_amd.numerics.integration import vegas_device

    cfg = DISConfig(quarks=(Quark(QuarkType.C, 1.4),), maxr=5.0)
    desc = dev.dis_desc(9.0, 1e-3, True, cfg.quarks, _gbw(), cfg)
    sizes = [2, 63, 256, 257, 2047, 2048, 2049, 4096 + 77, (1 << 18) - 5, (1 << 18) + 256, (1 << 19) + 3, (1 << 20) - 2048,
             (1 << 20) + 1]
    items = []
    for n in sizes:
        item = _lib.DisItem()
        item.desc, item.contribution, item.method = desc, _lib.DIS_KINDS["LO"], _lib.NLO_DIS_METHOD_VEGAS
        item.n, item.sobol_table, item.max_iterations, item.min_iterations, item.first_index = n, 0, 4, 4, 64
        items.append(item)
    got = dev.dis_batch(items, [dev.sobol_table(2, 5)], bins=cfg.bins, precision="fp64", epsrel=1e-12, device="cuda").cpu()
    for n, row in zip(sizes, got):
        print(f"samples {n}", flush=True)
        want = vegas_device(desc, "LO", samples_per_iteration=n, max_iterations=4, min_iterations=4, bins=cfg.bins,
                            epsrel=1e-12, seed=5, precision="fp64", first_index=64)
        # the same samples; refined edges agree to the fixed-point step of 2^-50
        assert float(row[0]) == pytest.approx(float(want.value), rel=1e-12, abs=0)
        assert float(row[1]) == pytest.approx(float(want.error), rel=1e-10, abs=0)
        assert int(row[2]) == want.n_eval


def test_gauss_legendre_item_equals_single_rule(dev):
    from nlo_bk_optimized_amd import _lib
    from nlo_bk_optimized_amd.dis.config import DISConfig, Quark, QuarkType
    from nlo_bk_optimized_amd.numerics.integration import gauss_legendre_device

    cfg = DISConfig(quarks=(Quark(QuarkType.LIGHT, 0.14), Quark(QuarkType.C, 1.27)))
    items, want = [], []
    for kind, transverse, quarks in (("LO", True, cfg.quarks), ("T0", True, cfg.quarks[:1]),
                                     ("Omega_L_const", False, cfg.quarks[1:]), ("LO", False, cfg.quarks)):
        desc = dev.dis_desc(12.0, 1e-4, transverse, quarks, _gbw(), cfg)
        for pts in (24, 17):
            it = _lib.DisItem()
            it.desc = desc
            it.contribution = _lib.DIS_KINDS[kind]
            it.method = _lib.NLO_DIS_METHOD_GAUSS_LEGENDRE
            it.n = pts
            items.append(it)
            want.append(gauss_legendre_device(desc, kind, points=pts, epsrel=cfg.epsrel, precision="fp64"))
    got = dev.dis_batch(items, [], bins=cfg.bins, precision="fp64", epsrel=cfg.epsrel, device="cuda").cpu()
    for row, w in zip(got, want):
        assert float(row[0]) == float(w.value) and float(row[1]) == float(w.error)
        assert int(row[2]) == w.n_eval and bool(row[3]) == w.converged


def _bk_dipole():
    from nlo_bk_optimized_amd import MV, BKConfig, solve_bk
    from nlo_bk_optimized_amd.dipole import BKDipole

    cfg = BKConfig(RPOINTS=63, MINR=1e-6, MAXR=1e2, MCINTPOINTS=4096, DE_SOLVER_STEP=0.5, RK_METHOD="rk2",
                   K1_RULE="fixed", PRECISION="fp32")
    table = solve_bk(MV(qs0sqr=0.2), 12.0, cfg, device="cuda", dtype=torch.float64, seed=0)
    return BKDipole(table, device="cuda")


@pytest.mark.parametrize("dipole_kind", ["gbw", "bk"])
def test_points_in_a_batch_equal_points_alone(dev, dipole_kind):
    from nlo_bk_optimized_amd.dis import DISConfig, DISOrder, F2, F2_batch, sigma_r, sigma_r_batch
    from nlo_bk_optimized_amd.dis.config import Quark, QuarkType

    dipole = _gbw() if dipole_kind == "gbw" else _bk_dipole()
    cfg = DISConfig(order=DISOrder.NLO, quarks=(Quark(QuarkType.LIGHT, 0.14), Quark(QuarkType.C, 1.27)),
                    maxeval=1 << 13, epsrel=1e-3)
    pts = [(torch.tensor(q), torch.tensor(x)) for q, x in ((3.0, 1e-3), (25.0, 1e-4), (80.0, 1e-2))]
    print(f"F2 batch of {len(pts)} points, {dipole_kind}", flush=True)
    batch = F2_batch(pts, dipole, cfg, seed=5)
    alone = [F2(q, x, dipole, cfg, seed=5) for q, x in pts]
    for b, a in zip(batch, alone):
        assert torch.equal(b.value, a.value) and torch.equal(b.error, a.error)
        assert b.n_eval == a.n_eval and b.converged == a.converged
        assert math.isfinite(float(b.value)) and float(b.error) > 0
    sb = sigma_r_batch(pts[::2], 318.0, dipole, cfg, seed=5)
    sa = [sigma_r(q, x, 318.0, dipole, cfg, seed=5) for q, x in pts[::2]]
    for b, a in zip(sb, sa):
        assert torch.equal(b.value, a.value) and torch.equal(b.error, a.error)


def test_qqbarg_terms_match_reference_cpp_values(dev):
    """T/benchmarks/dis_fixed_sobol_all_qg.py:69-76 (20-worker C++ nlodis):
    value and error of each raw qqbar-g integral; ours by VEGAS (FP32 path,
    nested I2 / I3 with 48 inner nodes) within 4 combined standard errors."""

    from nlo_bk_optimized_amd import _lib
    from nlo_bk_optimized_amd.dis.config import DISConfig, Quark, QuarkType

    ref = {
        ("L", "I1"): (0.10206739088678346, 0.0002535000977528945),
        ("L", "I2_nested"): (-0.024439455902300525, 0.00004764427185133986),
        ("L", "I3_nested"): (0.009414936380564324, 0.000026852425497947778),
        ("T", "I1"): (0.40263591173620866, 0.0017956984452001683),
        ("T", "I2_nested"): (-0.08719375357937224, 0.00026850014906050766),
        ("T", "I3_nested"): (0.04848797141670969, 0.00013338145018266037),
    }
    cfg = DISConfig(quarks=(Quark(QuarkType.C, 1.4),), maxr=5.0, nf_alphas=1, cuda_nested_points=48)
    items, tables, keys = [], [], []
    for k, ((pol, kind), _) in enumerate(ref.items()):
        it = _lib.DisItem()
        it.desc = dev.dis_desc(9.0, 1e-3, pol == "T", cfg.quarks, _gbw(), cfg)
        it.contribution = _lib.DIS_KINDS[kind]
        it.method = _lib.NLO_DIS_METHOD_VEGAS
        it.n = 1 << 19
        it.sobol_table = k
        it.max_iterations, it.min_iterations = 8, 3
        it.first_index = 0
        items.append(it)
        tables.append(dev.sobol_table(5, 3100 + k))
        keys.append((pol, kind))
    print("six qqbar-g terms at the reference benchmark point", flush=True)
    got = dev.dis_batch(items, tables, bins=32, precision="fp32", epsrel=1e-12, device="cuda").cpu()
    for (key, (value, error)), row in zip(ref.items(), got):
        ours, err = float(row[0]), float(row[1])
        pull = (ours - value) / math.hypot(err, error)
        print(f"{key}: {ours:.8f} +- {err:.2e} vs {value:.8f} +- {error:.2e} ({pull:+.2f} sigma)")
        assert abs(pull) <= 4.0, (key, ours, err, value, error)
