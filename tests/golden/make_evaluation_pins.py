"""Values of the plain evaluation of the integrands, recorded on an MI355X.

    python tests/golden/make_evaluation_pins.py OUTPUT_DIRECTORY

The FP64 integrands have samples whose terms cancel by many digits, where
another order of the same operations gives other digits.  The recorded numbers
are those of the formulas written out with the math library's functions and
IEEE operations (the library as built from commit ccae63a); later kernels keep
them.  Each section is one .npz next to this file.
"""

from __future__ import annotations

import sys

import numpy as np
import torch

from nlo_bk_optimized_amd import device as dev
from nlo_bk_optimized_amd._lib import DIS_DIMENSIONS
from nlo_bk_optimized_amd.bk import MV, BKConfig
from nlo_bk_optimized_amd.bk.config import RunningCouplingNLO
from nlo_bk_optimized_amd.bk.evolution import uniform_edges
from nlo_bk_optimized_amd.dipole import GBW, BKDipole, DipoleTable
from nlo_bk_optimized_amd.dis import DISConfig, DISOrder, Polarization, Quark, QuarkType, structure_functions_batch
from nlo_bk_optimized_amd.dis.fixed_sobol import gbw_qg_fixed_sobol_batch

NODES = 24
SOBOL_SEEDS = (109, 110, 215, 339)  # each with a sample next to a2 = b2 in some parent


def bk_sums() -> dict[str, np.ndarray]:
    """Per-parent K2 + Kf sums of the FP64 formula, by kernel instance."""

    r = (1e-6 * torch.pow(torch.tensor((100.0 / 1e-6) ** (1 / (NODES - 1)), dtype=torch.float64),
                          torch.arange(NODES, dtype=torch.float64))).cuda()
    N = MV(qs0sqr=0.2).dipole_amplitude(r)
    t64, t32 = dev.spline_build(r, N)
    edges = uniform_edges(NODES, 50, r.device)
    config = BKConfig(RPOINTS=NODES - 1, MAXR=100.0)
    parent = BKConfig(RPOINTS=NODES - 1, MAXR=100.0, RC_NLO=RunningCouplingNLO.PARENT_NLO)
    out = {}
    for seed in SOBOL_SEEDS:
        table = dev.sobol_table(4, seed)
        for name, kwargs, cfg in (("full", {}, config), ("sum", {"sum_only": True}, config),
                                  ("histogram", {"histogram": True}, config), ("parent", {}, parent)):
            sums = dev.bk_nlo(r, N, t64, t32, edges, table, 1 << 17, cfg, precision="fp64", **kwargs)[0]
            out[f"{name}_{seed}"] = sums[:, 0].cpu().numpy()
    ev = dev.BatchEvolver(torch.cat([r, r]), torch.cat([edges, edges]), [NODES, NODES], dev.sobol_table(4, 109), config,
                          n_samples=1 << 17, precision="fp64", rk_method="euler", step=0.1, k1_rule="fixed")
    state = torch.cat([N, N])
    ev.state.copy_(state)
    ev.step()
    out["batch_109"] = (ev.state - state).cpu().numpy()
    return out


def bk_grids() -> dict[str, np.ndarray]:
    """Importance grids after five FP64 refinements, for the production coupling
    and the coupling at the parent."""

    from nlo_bk_optimized_amd.bk.evolution import prepare

    out = {}
    for name, kw in (("production", {"PRECISION": "fp64"}),
                     ("parent", {"PRECISION": "fp64", "RC_NLO": RunningCouplingNLO.PARENT_NLO})):
        config = BKConfig(RPOINTS=NODES - 1, MAXR=100.0, MCINTPOINTS=20_000, K1_RULE="fixed", **kw)
        out[name] = prepare(MV(qs0sqr=0.2), config, device=torch.device("cuda"), seed=3).edges[1::4].cpu().numpy()
    return out


QUARK = Quark(QuarkType.C, 1.4)
DIPOLE = GBW(Qs0sqr=0.4, lambda_=0.25, gamma=1.0, x0=1.0)


def integrand_points(kinds, precision: str) -> dict[str, np.ndarray]:
    """Integrands at points that crowd towards the lower faces of the cube,
    where gluons are soft and the terms cancel."""

    out = {}
    for kind in kinds:
        gen = torch.Generator().manual_seed(DIS_DIMENSIONS[kind])
        u = torch.rand((512, DIS_DIMENSIONS[kind]), generator=gen, dtype=torch.float64)
        u = (u ** (1 + 3 * torch.rand(u.shape, generator=gen, dtype=torch.float64))).cuda()
        for transverse in (False, True):
            desc = dev.dis_desc(10.0, 1e-3, transverse, (QUARK,), DIPOLE, DISConfig(quarks=(QUARK,), maxr=5.0))
            out[f"{kind}_{'T' if transverse else 'L'}"] = dev.dis_integrand(desc, kind, u, precision=precision).cpu().numpy()
    return out


def nested_fp32() -> dict[str, np.ndarray]:
    """The nested terms in FP32, and the fixed-Sobol estimator that sums them."""

    out = integrand_points(("I2_nested", "I3_nested"), "fp32")
    q2, x = torch.tensor(10.0, dtype=torch.float32), torch.tensor(1e-3, dtype=torch.float32)
    entries = [(q2, x, pol, QUARK, 5) for pol in (Polarization.L, Polarization.T)]
    results = gbw_qg_fixed_sobol_batch(entries, DIPOLE, DISConfig(quarks=(QUARK,), maxr=5.0))
    rows = [r for f in results for r in (*f.contributions, f.total)]
    out["estimator"] = torch.stack([torch.stack([r.value, r.error]).double() for r in rows]).cpu().numpy()
    return out


def dis_fp64() -> dict[str, np.ndarray]:
    return integrand_points(DIS_DIMENSIONS, "fp64")


def dis_batch() -> dict[str, np.ndarray]:
    """Structure functions of a table whose saturation scale grows with rapidity:
    eight refinements of every grid, so that the last bit of a histogram tells."""

    r = 1e-6 * torch.pow(torch.tensor(1e8 ** (1 / 127), dtype=torch.float64), torch.arange(128, dtype=torch.float64))
    y = torch.arange(31, dtype=torch.float64) * 0.4
    qs2 = 0.3 * torch.exp(0.22 * y)[:, None]
    e = r * r * qs2 / 4 * torch.log(1 / (0.241 * r) + 8 * 2.7182818)
    N = torch.where(e < 1e-5, e, -torch.expm1(-e))
    dipole = BKDipole(DipoleTable(r=r.cuda(), y=y.cuda(), N=N.cuda(), x0=0.01))
    out = {}
    for dtype, maxeval in ((torch.float64, 80_000), (torch.float64, 290_000), (torch.float32, 290_000)):
        config = DISConfig(order=DISOrder.NLO, maxeval=maxeval, epsrel=1e-12,
                           quarks=(Quark(QuarkType.LIGHT, 0.14), Quark(QuarkType.C, 1.27)))
        points = [(torch.tensor(q2, dtype=dtype), torch.tensor(x, dtype=dtype)) for q2, x in ((3.0, 5e-3), (40.0, 2e-4))]
        pairs = structure_functions_batch(points, dipole, config, seed=44)
        out[f"{'f64' if dtype is torch.float64 else 'f32'}_{maxeval}"] = torch.stack(
            [torch.stack([f.value, f.error]).double() for p in pairs for f in p]).cpu().numpy()
    return out


SECTIONS = {"bk_fp64_sums": bk_sums, "bk_fp64_grids": bk_grids, "nested_fp32": nested_fp32, "dis_fp64": dis_fp64,
            "dis_batch": dis_batch}

if __name__ == "__main__":
    for section, values in SECTIONS.items():
        np.savez_compressed(f"{sys.argv[1]}/{section}.npz", **values())
        print(section, flush=True)
