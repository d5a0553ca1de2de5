"""The work that a program using this package has it do, as timed cases.

Every case goes through the package's entry points: rapidity steps of one or
many BK evolutions (``device.Evolver``, ``device.BatchEvolver``), a whole short
evolution (``solve_bk``), the DIS structure functions (``F2``, ``structure_functions_batch``), the GBW fixed-Sobol estimator, single
DIS VEGAS passes and the sampling kernels.  ``exact`` gives the same outputs in
64 bits with plain torch, for the cases whose result is a fixed sum.
"""

from __future__ import annotations

import math
import random

import torch

from nlo_bk_optimized_amd import device as dev
from nlo_bk_optimized_amd._lib import DIS_DIMENSIONS
from nlo_bk_optimized_amd.bk import BKConfig, MV, solve_bk
from nlo_bk_optimized_amd.dipole import GBW, BKDipole, DipoleTable
from nlo_bk_optimized_amd.dis import F2, DISConfig, DISOrder, Polarization, Quark, QuarkType, structure_functions_batch
from nlo_bk_optimized_amd.dis.fixed_sobol import gbw_qg_fixed_sobol_batch

F64 = torch.float64
LAMBDA = 0.241
STAGES = {"euler": 1, "rk2": 2, "kutta3": 3, "rk4": 4}


def _device() -> torch.device:
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# ------------------------------------------------------------------- cases


def listed() -> list[dict]:
    return [
        # one output step of solve_bk with the default configuration (float32:
        # Kutta's three stages, fixed K1 rule, 100 000 points per parent)
        {"name": "bk_step_default", "kind": "step", "R": 101, "maxr": 30.0, "n": 100_000, "precision": "fp32",
         "rk": "kutta3", "k1": "fixed", "dy": 0.2},
        # one step of the 256-node benchmark evolution
        {"name": "bk_step_256_f32", "kind": "step", "R": 256, "maxr": 100.0, "n": 1 << 20, "precision": "fp32",
         "rk": "rk2", "k1": "fixed", "dy": 0.1},
        # the same grid on the plain FP64 path (the reference's K2 / Kf formula)
        {"name": "bk_step_256_f64", "kind": "step", "R": 256, "maxr": 100.0, "n": 1 << 18, "precision": "fp64",
         "rk": "rk2", "k1": "fixed", "dy": 0.1},
        # the rule solve_bk takes by default on every grid but the 101-node one
        {"name": "bk_step_256_adaptive", "kind": "step", "R": 256, "maxr": 100.0, "n": 1 << 18, "precision": "fp32",
         "rk": "euler", "k1": "adaptive", "dy": 0.1},
        # the largest grid of the benchmarks
        {"name": "bk_step_1024_f32", "kind": "step", "R": 1024, "maxr": 100.0, "n": 1 << 22, "precision": "fp32",
         "rk": "euler", "k1": "fixed", "dy": 0.05},
        # several evolutions of uneven grids stepped together
        {"name": "bk_batch_uneven", "kind": "batch", "sizes": "128,201,256,333,400,511", "n": 1 << 16, "rk": "rk2",
         "dy": 0.1},
        # the first two steps of the 64-node FP64 workload from the initial
        # condition on, grid adaptation included: a small call, where launches
        # and host work count
        {"name": "bk_solve_64_f64", "kind": "solve", "R": 64, "n": 1 << 14, "precision": "fp64", "rk": "rk2",
         "dy": 0.1, "steps": 2},
        # one structure function at one point with the default NLO settings
        {"name": "dis_f2_gbw_f32", "kind": "f2", "maxeval": 2_000_000, "light": 0.14, "charm": 1.4},
        # a few points of the (Q^2, x) table workload on an evolved dipole
        {"name": "dis_batch_table_f32", "kind": "sigma", "points": 4, "maxeval": 1 << 19, "dtype": "f32"},
        # the same on the FP64 path (6- / 7-dimensional I2, I3)
        {"name": "dis_point_table_f64", "kind": "sigma", "points": 1, "maxeval": 1 << 18, "dtype": "f64"},
        # single VEGAS passes of the terms both paths evaluate in FP64
        {"name": "dis_terms_f64", "kind": "terms", "n": 1 << 20, "bins": 32, "mass": 1.27},
        # the reference's six-term qqbar-g workload, grid learning included
        {"name": "dis_fixed_sobol_gbw", "kind": "fixed", "quarks": 1, "maxr": 5.0},
    ]


def _loguniform(rng: random.Random, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["step", "step", "step", "batch", "solve", "f2", "sigma", "terms", "fixed"])
    if kind == "step":
        precision = rng.choice(["fp32", "fp32", "fp64"])
        k1 = rng.choice(["fixed", "fixed", "adaptive"])
        R = int(_loguniform(rng, 48, 1024 if k1 == "fixed" else 420))
        rk = rng.choice(["euler", "rk2", "kutta3", "rk4"])
        budget = (4e9 if precision == "fp32" else 5e8) / (R * STAGES[rk])
        n = int(_loguniform(rng, 1 << 13, min(budget, 1 << 22)))
        return {"kind": kind, "R": R, "maxr": rng.choice([30.0, 50.0, 100.0]), "n": n, "precision": precision,
                "rk": rk, "k1": k1, "dy": rng.choice([0.05, 0.1, 0.2])}
    if kind == "batch":
        sizes = [rng.randint(64, 512) for _ in range(rng.randint(2, 8))]
        return {"kind": kind, "sizes": ",".join(map(str, sizes)), "n": int(_loguniform(rng, 1 << 13, 1 << 17)),
                "rk": rng.choice(["rk2", "kutta3"]), "dy": 0.1}
    if kind == "solve":
        return {"kind": kind, "R": int(_loguniform(rng, 33, 256)), "n": int(_loguniform(rng, 1 << 12, 1 << 17)),
                "precision": rng.choice(["fp32", "fp64"]), "rk": rng.choice(["euler", "rk2"]), "dy": 0.1,
                "steps": rng.randint(1, 3)}
    if kind == "f2":
        return {"kind": kind, "maxeval": int(_loguniform(rng, 900_000, 4_000_000)),
                "light": rng.choice([0.002, 0.14]), "charm": rng.uniform(1.27, 1.5)}
    if kind == "sigma":
        dtype = rng.choice(["f32", "f32", "f64"])
        return {"kind": kind, "points": rng.randint(1, 6 if dtype == "f32" else 3),
                "maxeval": int(_loguniform(rng, 1 << 16, 1 << 19)), "dtype": dtype}
    if kind == "terms":
        return {"kind": kind, "n": int(_loguniform(rng, 1 << 14, 1 << 22)), "bins": rng.choice([32, 50]),
                "mass": rng.choice([0.14, 1.27, 1.4])}
    return {"kind": kind, "quarks": rng.randint(1, 3), "maxr": rng.uniform(5.0, 30.0)}


# ------------------------------------------------------------------ inputs


def _mv(seed: int, index: int = 0) -> dict:
    rng = random.Random(f"mv {seed} {index}")
    return {"qs0sqr": rng.uniform(0.1, 0.5), "gamma": rng.uniform(0.9, 1.2), "ec": rng.uniform(1.0, 20.0)}


def _amplitude(r: torch.Tensor, ic: dict, growth: float = 1.0) -> torch.Tensor:
    e = torch.pow(r * r * (ic["qs0sqr"] * growth), ic["gamma"]) / 4 * torch.log(1 / (r * LAMBDA) + ic["ec"] * 2.7182818)
    return torch.where(e < 1e-5, e, -torch.expm1(-e))


def _r_grid(R: int, maxr: float) -> torch.Tensor:
    return 1e-6 * torch.pow(torch.tensor((maxr / 1e-6) ** (1 / (R - 1)), dtype=F64), torch.arange(R, dtype=F64))


def _frozen_grids(r: torch.Tensor, bins: int) -> torch.Tensor:
    """Importance grids of the shape adaptation gives them: the log-distance
    dimensions gather around the parent's own size, the angles around 0."""

    u = torch.linspace(0, 1, 2001, dtype=F64)
    lo = math.log(0.5 * float(r[0]))
    width = math.log(2.0 * float(r[-1])) - lo
    centre = ((torch.log(r) - lo) / width)[:, None]
    radial = 0.25 + torch.exp(-0.5 * ((u - centre) / 0.09) ** 2) / 0.09
    angular = (0.6 + torch.exp(-u / 0.08) + torch.exp(-(1 - u) / 0.08)).expand_as(radial)
    out = []
    for density in (radial, radial, angular, angular):
        cdf = torch.cumulative_trapezoid(density, u, dim=1)
        cdf = torch.cat([torch.zeros_like(cdf[:, :1]), cdf], 1) / cdf[:, -1:]
        target = torch.linspace(0, 1, bins + 1, dtype=F64).expand(len(r), -1).contiguous()
        k = torch.searchsorted(cdf.contiguous(), target).clamp(1, u.numel() - 1)
        c0, c1 = cdf.gather(1, k - 1), cdf.gather(1, k)
        e = u[k - 1] + (target - c0) / (c1 - c0) * (u[k] - u[k - 1])
        e[:, 0], e[:, -1] = 0.0, 1.0
        out.append(e)
    return torch.stack(out, 1).contiguous()


def _bk_config(case: dict, R: int, maxr: float) -> BKConfig:
    return BKConfig(RPOINTS=R - 1, MINR=1e-6, MAXR=maxr, MCINTPOINTS=case["n"], DE_SOLVER_STEP=case["dy"],
                    PRECISION=case.get("precision", "fp32"), RK_METHOD=case["rk"])


def _table(seed: int) -> DipoleTable:
    """An evolved amplitude: the saturation scale grows with rapidity."""

    r = _r_grid(256, 100.0)
    y = torch.arange(0, 61, dtype=F64) * 0.2
    N = torch.stack([_amplitude(r, _mv(seed), math.exp(0.22 * float(v))) for v in y])
    return DipoleTable(r=r.cuda(), y=y.cuda(), N=N.cuda(), x0=0.01)


def _kinematics(seed: int, count: int) -> list[tuple[float, float]]:
    rng = random.Random(f"kinematics {seed}")
    return [(_loguniform(rng, 1.0, 100.0), _loguniform(rng, 2e-5, 1e-2)) for _ in range(count)]


def _gbw(seed: int) -> GBW:
    rng = random.Random(f"gbw {seed}")
    return GBW(Qs0sqr=rng.uniform(0.2, 1.0), lambda_=rng.uniform(0.2, 0.3), gamma=1.0, x0=1.0)


def _term_grid(kind: str, bins: int, seed: int) -> torch.Tensor:
    """A mildly refined grid per dimension."""

    gen = torch.Generator().manual_seed(seed)
    width = 0.5 + torch.rand(DIS_DIMENSIONS[kind], bins, generator=gen, dtype=F64)
    e = torch.cumsum(width, 1) / width.sum(1, keepdim=True)
    e[:, -1] = 1.0
    return torch.cat([torch.zeros_like(e[:, :1]), e], 1)


# (term, transverse) of the passes that run in FP64 on both paths
TERMS = (("T1", True), ("ab", False), ("I1", True), ("I1", False))


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "step":
        r = _r_grid(case["R"], case["maxr"])
        config = _bk_config(case, case["R"], case["maxr"])
        ev = dev.Evolver(r.cuda(), _frozen_grids(r, config.MC_BINS).cuda(), dev.sobol_table(4, seed), config,
                         n_samples=case["n"], precision=case["precision"], rk_method=case["rk"], step=case["dy"],
                         k1_rule=case["k1"])
        return {"kind": kind, "ev": ev, "N": _amplitude(r, _mv(seed)).cuda()}
    if kind == "batch":
        sizes = [int(v) for v in case["sizes"].split(",")]
        grids = [_r_grid(R, 100.0) for R in sizes]
        config = _bk_config(case, sizes[0], 100.0)
        ev = dev.BatchEvolver(torch.cat(grids).cuda(),
                              torch.cat([_frozen_grids(r, config.MC_BINS) for r in grids]).cuda(), sizes,
                              dev.sobol_table(4, seed), config, n_samples=case["n"], precision="fp32",
                              rk_method=case["rk"], step=case["dy"], k1_rule="fixed")
        N = torch.cat([_amplitude(r, _mv(seed, i)) for i, r in enumerate(grids)]).cuda()
        ev.state.copy_(N)
        ev.step()  # the first step chooses the launch shape for the steps that follow
        return {"kind": kind, "ev": ev, "N": N}
    if kind == "solve":
        return {"kind": kind, "ic": MV(**_mv(seed)), "config": _bk_config(case, case["R"], 100.0), "seed": seed,
                "maxy": case["dy"] * case["steps"], "dtype": torch.float32 if case["precision"] == "fp32" else F64}
    if kind == "f2":
        (q2, x), = _kinematics(seed, 1)
        config = DISConfig(order=DISOrder.NLO, maxeval=case["maxeval"],
                           quarks=(Quark(QuarkType.LIGHT, case["light"]), Quark(QuarkType.C, case["charm"])))
        return {"kind": kind, "Q2": torch.tensor(q2, dtype=torch.float32), "x": torch.tensor(x, dtype=torch.float32),
                "dipole": _gbw(seed), "config": config, "seed": seed}
    if kind == "sigma":
        dtype = torch.float32 if case["dtype"] == "f32" else F64
        config = DISConfig(order=DISOrder.NLO, maxeval=case["maxeval"], epsrel=1e-12,
                           quarks=(Quark(QuarkType.LIGHT, 0.14), Quark(QuarkType.C, 1.27)))
        points = [(torch.tensor(q, dtype=dtype), torch.tensor(x, dtype=dtype))
                  for q, x in _kinematics(seed, case["points"])]
        return {"kind": kind, "points": points, "dipole": BKDipole(_table(seed)), "config": config, "seed": seed}
    if kind == "terms":
        (q2, x), = _kinematics(seed, 1)
        quark = Quark(QuarkType.C if case["mass"] > 1 else QuarkType.LIGHT, case["mass"])
        config = DISConfig(quarks=(quark,), maxr=5.0)
        passes = [(dev.dis_desc(q2, x, transverse, (quark,), _gbw(seed), config), term,
                   _term_grid(term, case["bins"], seed).cuda(), dev.sobol_table(DIS_DIMENSIONS[term], seed))
                  for term, transverse in TERMS]
        return {"kind": kind, "passes": passes, "n": case["n"]}
    quarks = [Quark(QuarkType.C, 1.4), Quark(QuarkType.LIGHT, 0.14), Quark(QuarkType.B, 4.18)][:case["quarks"]]
    (q2, x), = _kinematics(seed, 1)
    q2t, xt = torch.tensor(q2, dtype=torch.float32), torch.tensor(x, dtype=torch.float32)
    entries = [(q2t, xt, pol, q, seed + i) for pol in (Polarization.L, Polarization.T) for i, q in enumerate(quarks)]
    return {"kind": "fixed", "entries": entries, "dipole": _gbw(seed),
            "config": DISConfig(quarks=tuple(quarks), maxr=case["maxr"])}


def run(state: dict):
    kind = state["kind"]
    if kind == "step":
        ev = state["ev"]
        ev.state.copy_(state["N"])
        ev.step()
        return {"N": ev.state, "K1": ev.k1, "K2Kf": ev.k2kf}
    if kind == "batch":
        ev = state["ev"]
        ev.state.copy_(state["N"])
        ev.step()
        return {"N": ev.state}
    if kind == "solve":
        t = solve_bk(state["ic"], state["maxy"], state["config"], dtype=state["dtype"], seed=state["seed"])
        return {"r": t.r, "y": t.y, "N": t.N}
    if kind == "f2":
        f = F2(state["Q2"], state["x"], state["dipole"], state["config"], seed=state["seed"])
        return {"value": f.value, "error": f.error}
    if kind == "sigma":
        pairs = structure_functions_batch(state["points"], state["dipole"], state["config"], seed=state["seed"])
        return {"value": torch.stack([f.value for p in pairs for f in p]),
                "error": torch.stack([f.error for p in pairs for f in p])}
    if kind == "terms":
        out = []
        for desc, term, edges, table in state["passes"]:
            sums, hist, count = dev.dis_vegas(desc, term, edges, table, state["n"])
            out.append({"sums": sums, "hist": hist, "count": count})
        return out
    results = gbw_qg_fixed_sobol_batch(state["entries"], state["dipole"], state["config"])
    rows = [r for f in results for r in (*f.contributions, f.total)]
    return {"value": torch.stack([r.value for r in rows]), "error": torch.stack([r.error for r in rows])}


# ------------------------------------------------------------ cost, tolerance

# Operations of one evaluation (a named function counts 1): a K2 + Kf sample,
# a K1 node, a DIS integrand sample, a node of the inner rule.
SAMPLE, NODE, TERM, INNER = 216, 90, 250, 180


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("step", "batch"):
        sizes = [case["R"]] if kind == "step" else [int(v) for v in case["sizes"].split(",")]
        flops = sum((R - 1) * (case["n"] * SAMPLE + (R - 1) * 192 * NODE) for R in sizes) * STAGES[case["rk"]]
        return {"bytes": sum(R * 8 * (4 * 51 + 5) for R in sizes), "flops": flops}
    if kind == "solve":  # five adaptation passes and the steps' right-hand sides
        R, stages = case["R"], case["steps"] * STAGES[case["rk"]]
        return {"bytes": R * 8 * (case["steps"] + 2),
                "flops": (R - 1) * ((5 + stages) * case["n"] * SAMPLE + stages * (R - 1) * 192 * NODE)}
    if kind == "f2":  # the dipole terms at three of eight iterations, the fixed-Sobol estimators
        return {"bytes": 256, "flops": 2 * 2 * 11 * case["maxeval"] * 3 // 8 * TERM + 4 * 851_968 * (TERM + 48 * INNER)}
    if kind == "sigma":
        inner = 48 * INNER if case["dtype"] == "f32" else 2 * INNER
        return {"bytes": 256 * 61 * 8, "flops": case["points"] * 2 * case["maxeval"] * (22 * TERM + 2 * (3 * TERM + 2 * inner))}
    if kind == "terms":
        return {"bytes": len(TERMS) * 5 * case["bins"] * 24, "flops": len(TERMS) * case["n"] * TERM}
    return {"bytes": 4096, "flops": 2 * case["quarks"] * 851_968 * (TERM + 48 * INNER)}


def tolerance(case: dict):
    """About four times the largest difference seen between ``run`` and
    ``exact``, or between two runs whose inputs differ by a rounding."""

    kind = case["kind"]
    if kind == "step":  # K2 + Kf: FP32 integrand 1.2e-5; FP64 reference formula 2.3e-11, more at few points
        return {"rel": 5e-5 if case["precision"] == "fp32" else 1e-9}
    if kind == "batch":  # 2.2e-6 where a rounding takes a node across N = 0.99999
        return {"rel": 1e-5}
    if kind == "solve":
        return {"rel": 1e-5 if case["precision"] == "fp32" else 1e-10}
    if kind == "sigma":  # grids refined from FP32 weights: 4.4e-5
        return {"rel": 2e-4 if case["dtype"] == "f32" else 1e-9}
    # f2 4.3e-5; the spread of seven replicates 4.1e-4
    return {"rel": {"f2": 2e-4, "terms": 1e-10, "fixed": 2e-3}[kind]}


# -------------------------------------------------- the same in plain torch


def _natural_spline(x: torch.Tensor, y: torch.Tensor) -> torch.Tensor:
    """Cubics {a, b, c, d} in x - x_i of the natural spline through (x, y)."""

    h = x[1:] - x[:-1]
    A = torch.diag(2 * (h[:-1] + h[1:])) + torch.diag(h[1:-1], 1) + torch.diag(h[1:-1], -1)
    s = (y[1:] - y[:-1]) / h
    m = torch.zeros_like(y)
    m[1:-1] = torch.linalg.solve(A, 6 * (s[1:] - s[:-1]))
    return torch.stack([y[:-1], s - h * (2 * m[:-1] + m[1:]) / 6, m[:-1] / 2, (m[1:] - m[:-1]) / (6 * h)], 1)


class _Spline:
    def __init__(self, x: torch.Tensor, value: torch.Tensor, below: float, above: float) -> None:
        self.x, self.below, self.above = x, below, above
        logs = torch.where(value > 0, torch.log(value.clamp_min(1e-300)), torch.full_like(value, -40.0))
        self.c = _natural_spline(x, logs)

    def __call__(self, lv: torch.Tensor) -> torch.Tensor:
        e = lv.clamp(self.x[0], self.x[-1])
        k = (torch.searchsorted(self.x, e.contiguous(), right=True) - 1).clamp(0, len(self.x) - 2)
        c, t = self.c[k], e - self.x[k]
        v = torch.exp(c[..., 0] + t * (c[..., 1] + t * (c[..., 2] + t * c[..., 3])))
        v = torch.where(lv < self.x[0], torch.full_like(v, self.below), v)
        return torch.where(lv > self.x[-1], torch.full_like(v, self.above), v)


B0 = (11 * 3.0 - 2 * 3.0) / (12 * math.pi)
MU0 = 10 * math.log(2.5)
LOG_SCALE = math.log(4 / LAMBDA**2)


def _alpha(log_d: torch.Tensor) -> torch.Tensor:
    right = 5 * (LOG_SCALE - 2 * log_d)
    return 1 / (B0 * 0.2 * torch.logaddexp(right, torch.full_like(right, MU0)))


def _j1_i1(s: torch.Tensor) -> torch.Tensor:
    """sum_k s^k / (k! (k+1)!): I1(2a)/a at s = a^2, J1(2a)/a at s = -a^2 (the
    trapezoidal rule on Bessel's integral where the series would cancel)."""

    term = torch.ones_like(s)
    total = term.clone()
    for k in range(1, 64):
        term = term * s / (k * (k + 1))
        total = total + term
    x = 2 * torch.sqrt((-s).clamp_min(0))
    m = 80
    j1 = torch.zeros_like(s)
    for k in range(m):
        t = 2 * math.pi * k / m
        j1 = j1 + torch.cos(t - x * math.sin(t))
    return torch.where(s < -4, 2 * j1 / m / x.clamp_min(1), total)


def _k1(x: torch.Tensor, N: torch.Tensor, p: int, sN: _Spline, rule) -> torch.Tensor:
    """K1 of parent p on the fixed 8 x 24 rule per log-r panel."""

    lr = x[p]
    r = torch.exp(lr)
    nr = torch.clamp(sN(lr), max=1.0)
    ar = _alpha(lr)
    gx, gw, gt, gv = rule
    half = (x[1:] - x[:-1]) / 2
    lz = ((x[1:] + x[:-1]) / 2)[:, None] + half[:, None] * gx
    w = (half[:, None] * gw).reshape(-1, 1)
    lz = lz.reshape(-1, 1)
    z = torch.exp(lz)
    v = (gt + 1) / 2
    s2 = torch.sin(math.pi * v * v / 2) ** 2
    xsq = (r - z) ** 2 + 4 * r * z * s2
    lx = torch.log(xsq) / 2
    nx, ny = torch.clamp(sN(lx), max=1.0), torch.clamp(sN(lz), max=1.0)
    ax, ay = _alpha(lx), _alpha(lz)
    lmin = torch.minimum(lx, lz)
    amin = torch.where(lmin <= lr, torch.where(lx <= lz, ax, ay), ar)
    rxy = r * r / (xsq * z * z)
    pref = 3 / (2 * math.pi**2) * ar
    lo = pref * (rxy + (ay / ax - 1) / (z * z) + (ax / ay - 1) / xsq)
    abar = amin * 3 / math.pi
    resum = _j1_i1(-abar * 4 * (lx - lr) * (lz - lr)) if float(r) > 1.01e-6 else torch.ones_like(lo)
    slog = -abar * (11 / 12) * torch.abs(math.log(0.65) + 2 * (lr - lmin))
    fin = ar * 3 / (4 * math.pi) * (67 / 9 - math.pi**2 / 3 - 10 / 9)
    value = (resum * torch.exp(slog) * lo - pref * rxy * slog + lo * fin) * (nx + ny - nr - nx * ny)
    return (value * (gv * math.pi * v) * 2 * z * z * w).sum()


def _log_ratio(r: torch.Tensor, z: torch.Tensor, lz: torch.Tensor, cos_t: torch.Tensor, xsq: torch.Tensor):
    u = r / z * (r / z - 2 * cos_t)
    return torch.where(u.abs() < 0.5, torch.log1p(u) / 2, torch.log(xsq) / 2 - lz)


def _k2kf(x, p, spline, of_s: bool, q, edges, bins) -> torch.Tensor:
    """Mean of the K2 + Kf integrand of parent p over the points q."""

    lo = x[0] - math.log(2.0)
    wr = x[-1] + math.log(2.0) - lo
    b = torch.clamp((q * bins).floor().long(), max=bins - 1)
    frac = q * bins - b
    jac, c = torch.ones_like(q[:, 0]), []
    for d in range(4):
        left, right = edges[d][b[:, d]], edges[d][b[:, d] + 1]
        width = wr if d < 2 else 2 * math.pi
        c.append((lo if d < 2 else 0.0) + width * (left + (right - left) * frac[:, d]))
        jac = jac * (bins * (right - left) * width)
    lz, lz2, t1, t2 = c
    lr = x[p]
    r, z, z2 = torch.exp(lr), torch.exp(lz), torch.exp(lz2)
    xsq = (r - z) ** 2 + 4 * r * z * torch.sin(t1 / 2) ** 2
    x2sq = (r - z2) ** 2 + 4 * r * z2 * torch.sin(t2 / 2) ** 2
    zsq = (z - z2) ** 2 + 4 * z * z2 * torch.sin((t1 - t2) / 2) ** 2
    lxy, lxy2 = _log_ratio(r, z, lz, torch.cos(t1), xsq), _log_ratio(r, z2, lz2, torch.cos(t2), x2sq)
    lx, lx2, lzz = lz + lxy, lz2 + lxy2, torch.log(zsq) / 2
    f = [spline(v) for v in (lx, lz, lx2, lz2, lzz)]
    nx, ny, nx2, ny2, nz = (1 - v for v in f) if of_s else f
    sx, sy, sx2, sy2, _ = f if of_s else [1 - v for v in f]
    L = lxy - lxy2
    e = torch.expm1(2 * L)
    h = torch.where(L.abs() < 1e-12, torch.ones_like(L), 2 * L / torch.where(e == 0, torch.ones_like(e), e))
    hm = h + 2 * L
    small = L.abs() < 0.1
    y = L * L
    g = torch.where(small, y * (1 / 3 + y * (-1 / 45 + y * (2 / 945 + y * (-1 / 4725 + y * (2 / 93555 - y * 1382 / 638512875))))),
                    L.abs() + torch.where(L >= 0, h, hm) - 1)
    A, Bq, C, D = z * z2 / zsq, r * r * z2 * z2 / (x2sq * zsq), r**4 / (xsq * x2sq), r * r * z * z / (xsq * zsq)
    a2g = 2 * A * A * g
    k = a2g - 4 * h * Bq + h * C + 2 * L * D
    ks = a2g - 4 * hm * D + hm * C - 2 * L * Bq
    dip, dips = sx * (nz + ny2 - ny - nz * ny2), sx2 * (nz + ny - ny2 - nz * ny)
    cut = 1e10 * (z * z2) ** 2
    k2 = (torch.where((k.abs() > cut) & (dip.abs() < 1e-10), 0.0, k * dip)
          + torch.where((ks.abs() > cut) & (dips.abs() < 1e-10), 0.0, ks * dips)) / 2
    kf = -((h * Bq - a2g) * sy * (nx - nx2) + (hm * D - a2g) * sy2 * (nx2 - nx)) / 2
    dmin = torch.minimum(torch.minimum(torch.minimum(lx, lz), torch.minimum(lx2, lz2)), lzz).clamp(max=float(lr))
    w = (k2 + kf) * (3 * _alpha(dmin)) ** 2 / (8 * math.pi**4) * jac
    return torch.where(torch.isfinite(w), w, torch.zeros_like(w)).sum() / len(q)


def _gauss(n: int, device) -> tuple[torch.Tensor, torch.Tensor]:
    import numpy as np

    x, w = np.polynomial.legendre.leggauss(n)
    return torch.tensor(x, device=device), torch.tensor(w, device=device)


def _exact_step(case: dict, seed: int, R: int, maxr: float, index: int, precision: str, k1: bool) -> dict:
    d = _device()
    r = _r_grid(R, maxr)
    N0 = _amplitude(r, _mv(seed, index)).to(d)
    edges = _frozen_grids(r, 50).to(d)
    x = torch.log(r).to(d)
    n = case["n"]
    q = torch.quasirandom.SobolEngine(4, scramble=True, seed=seed).draw(n, dtype=F64).to(d)
    gx, gw = _gauss(8, d)
    gt, gv = _gauss(24, d)

    def rhs(N: torch.Tensor):
        sN = _Spline(x, N.clamp(0, 1), 0.0, 1.0)
        spline = _Spline(x, (1 - N).clamp(0, 1), 1.0, 0.0) if precision == "fp64" else sN
        a, b = torch.zeros_like(N), torch.zeros_like(N)
        for p in range(1, R):
            if float(N[p]) <= 0.99999:
                if k1:
                    a[p] = _k1(x, N, p, sN, (gx, gw, gt, gv))
                for part in q.split(1 << 22):
                    b[p] += _k2kf(x, p, spline, precision == "fp64", part, edges[p], 50) * len(part) / n
        return a, b

    a = {"euler": [[]], "rk2": [[], [0.5]], "kutta3": [[], [0.5], [-1, 2]], "rk4": [[], [0.5], [0, 0.5], [0, 0, 1]]}
    b = {"euler": [1], "rk2": [0, 1], "kutta3": [1 / 6, 4 / 6, 1 / 6], "rk4": [1 / 6, 2 / 6, 2 / 6, 1 / 6]}
    K = []
    for row in a[case["rk"]]:
        N = N0 + case["dy"] * sum((c * k for c, k in zip(row, K)), torch.zeros_like(N0))
        ka, kb = rhs(N)
        K.append(ka + kb)
    out = (N0 + case["dy"] * sum(c * k for c, k in zip(b[case["rk"]], K))).clamp(0, 1)
    return {"N": out if k1 else None, "K1": ka if k1 else None, "K2Kf": kb}


def _k01(x: torch.Tensor):
    return torch.special.modified_bessel_k0(x), torch.special.modified_bessel_k1(x)


def _gbw_n(r, Y, d: GBW):
    return -torch.expm1(-((r * r * d.Qs0sqr * torch.exp(d.lambda_ * Y.clamp_min(math.log(1 / d.x0)))) ** d.gamma) / 4)


def _dis_alpha(r, flavours: int):
    arg = 4 / (LAMBDA * LAMBDA * r * r)
    a = 12 * math.pi / ((33 - 2 * flavours) * torch.log(arg))
    return torch.where((a > 0.7) | (arg < 1), torch.full_like(a, 0.7), a)


def _exact_term(term: str, transverse: bool, u, q2: float, xbj: float, m: float, maxr: float, flavours: int, d: GBW):
    Q = math.sqrt(q2)
    af = 4 / 3 / math.pi
    if term in ("T1", "ab"):
        z, r, xi = 1e-6 + u[:, 0] * (1 - 2e-6), maxr * u[:, 1], u[:, 2]
        kz = torch.sqrt(z * (1 - z) * q2 + m * m)
        k0, k1 = _k01(r * kz)
        if term == "ab":
            b2 = _k01(r * torch.sqrt(kz**2 + (1 - z) * xi / (1 - xi) * m * m))[0]
            b3 = _k01(r * torch.sqrt(kz**2 + z * xi / (1 - xi) * m * m))[0]
            res = 4 * q2 * (z * (1 - z)) ** 2 * k0 / xi * (-2 * torch.log(xi) / (1 - xi) + (1 + xi) / 2) * (2 * k0 - b2 - b3)
        else:
            res = torch.zeros_like(z)
            for zz in (z, 1 - z):
                sh = torch.sqrt(kz**2 + xi / (1 - xi) * (1 - zz) * m * m)
                s0, s1 = _k01(r * sh)
                pre = (2 * torch.log(xi) / (1 - xi) - (1 + xi) / 2) / xi
                v1 = pre * (sh * s1 - kz * k1) - (torch.log(xi) / (1 - xi) ** 2 + zz / (1 - xi) + zz / 2) * (1 - zz) * m * m / sh * s1
                vm = pre * (s0 - k0) + (-1.5 * (1 - zz) / (1 - xi) + (1 - zz) / 2) * s0
                res = res + kz * k1 * (z * z + (1 - z) ** 2) * v1 + m * m * k0 * vm
        Y = torch.full_like(r, math.log(1 + (1 - xbj) / xbj))
        f = _gbw_n(r, Y, d) * res * r * maxr * (1 - 2e-6) * _dis_alpha(r, flavours) * af
        return torch.where(torch.isfinite(f), f, torch.zeros_like(f))
    z2min = xbj / q2
    z1 = (1 - z2min) * u[:, 0]
    z2 = (1 - z1 - z2min) * u[:, 1] + z2min
    z0 = 1 - z1 - z2
    a01, a02 = maxr * u[:, 2], maxr * u[:, 3]
    s01, s02 = a01**2, a02**2
    s21 = (s01 + s02 - 2 * a01 * a02 * torch.cos(2 * math.pi * u[:, 4])).clamp_min(0)
    a21 = torch.sqrt(s21)
    Y = torch.log(q2 / xbj * z2)
    S = [1 - _gbw_n(v, Y, d) for v in (a01, a02, a21)]
    n012 = 1 - 9 / 8 * (S[1] * S[2] - S[0] / 9)
    dot = (s21 + s02 - s01) / 2
    a, b = z0 + z2, z1 + z2
    qj, qk = q2 * z1 * (1 - z1) + m * m, q2 * z0 * (1 - z0) + m * m
    lj, lk = z1 * z2 / z0, z0 * z2 / z1
    x3j, x3k = (z0 / a) ** 2 * s02 + s21 - 2 * z0 / a * dot, (z1 / b) ** 2 * s21 + s02 - 2 * z1 / b * dot
    sj, sk = x3j + z0 * z2 / (z1 * a * a) * s02, x3k + z1 * z2 / (z0 * b * b) * s21
    j23, k23 = dot - z0 / a * s02, -dot + z1 / b * s21
    jk23, kj23 = -s02 + z1 / b * dot, s21 - z0 / a * dot
    j33 = z0 / a * s02 + z1 / b * s21 - (1 + z0 * z1 / (a * b)) * dot
    (k0j, k1j), (k0k, k1k) = _k01(torch.sqrt(qj * sj)), _k01(torch.sqrt(qk * sk))
    (u0j, u1j), (u0k, u1k) = _k01(torch.sqrt(qj * s01)), _k01(torch.sqrt(qk * s01))
    eg = 1.7810724179901979852
    ej, ek = -torch.exp(-s02 / (s01 * eg)) / s02, -torch.exp(-s21 / (s01 * eg)) / s21
    tj, tk = 2 * z0 * a + z2 * z2, 2 * z1 * b + z2 * z2
    if transverse:
        pj, pk = tj / (a * a), tk / (b * b)
        cj, ck = pj * (1 - 2 * z1 * (1 - z1)) * qj, pk * (1 - 2 * z0 * (1 - z0)) * qk
        uv = cj * ej * u1j**2 + ck * ek * u1k**2 + m * m * (pj * ej * u0j**2 + pk * ek * u0k**2)
        mj, mk = qj + m * m * lj, qk + m * m * lk
        hj, hk = 4 * torch.sqrt(mj / sj) * _k01(torch.sqrt(mj * sj))[1], 4 * torch.sqrt(mk / sk) * _k01(torch.sqrt(mk * sk))[1]
        gj, gk = torch.sqrt(qj / sj) * k1j / s02, torch.sqrt(qk / sk) * k1k / s21
        cross = z2 * (z0 - z1) ** 2 * (j23 * k23 - kj23 * jk23) - (z1 * a + z0 * b) * (z0 * a + z1 * b) * dot * j33
        f = (4 / (a * b) * cross * gj * gk - a * z1 * z2 / (b * b) * j23 * hk * gj + b * z0 * z2 / (a * a) * k23 * hj * gk
             - z0**2 * z1 * z2 / a**3 * j23 * hj * gj + z1**2 * z0 * z2 / b**3 * k23 * hk * gk
             + (z0 * z2) ** 2 / (8 * a**4) * hj**2 + (z1 * z2) ** 2 / (8 * b**4) * hk**2) / 2
        fm = -m * m * ((2 * z0 + z2) * (2 * z1 + z2) + z2 * z2) * dot * k0j * k0k / (s02 * s21 * a * b)
        i1 = (cj / s02 * x3j / sj * k1j**2 + ck / s21 * x3k / sk * k1k**2
              + m * m * (pj / s02 * k0j**2 + pk / s21 * k0k**2) + f + fm)
    else:
        uv = 4 * q2 * (z1**2 * tj * ej * u0j**2 + z0**2 * tk * ek * u0k**2)
        i1 = 4 * q2 * (z1**2 * tj / s02 * k0j**2 + z0**2 * tk / s21 * k0k**2
                       - 2 * z0 * z1 * (z0 * (1 - z0) + z1 * (1 - z1)) * dot / (s02 * s21) * k0j * k0k)
    res = (_gbw_n(a01, Y, d) * uv + n012 * i1) * (1 - z2min) * (1 - z1 - z2min) * a01 * a02 * maxr**2 * 2 * math.pi
    res = res * _dis_alpha(torch.minimum(a01, torch.minimum(a02, a21)), flavours) * af / z2
    return torch.where((Y >= 0) & torch.isfinite(res), res, torch.zeros_like(res))


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("step", "batch"):
        sizes = [case["R"]] if kind == "step" else [int(v) for v in case["sizes"].split(",")]
        if sum(sizes) * case["n"] * STAGES[case["rk"]] > (6e8 if _device().type == "cuda" else 3e6):
            return None
        if sum(sizes) * STAGES[case["rk"]] > 4000:
            return None
        if kind == "step":
            if case["k1"] == "adaptive" and case["rk"] != "euler":
                return None
            return _exact_step(case, seed, case["R"], case["maxr"], 0, case["precision"], case["k1"] == "fixed")
        parts = [_exact_step(case, seed, R, 100.0, i, "fp32", True)["N"] for i, R in enumerate(sizes)]
        return {"N": torch.cat(parts)}
    if kind != "terms" or case["n"] > (1 << 22):
        return None
    (q2, x), = _kinematics(seed, 1)
    out, bins = [], case["bins"]
    for term, transverse in TERMS:
        dim = DIS_DIMENSIONS[term]
        e = _term_grid(term, bins, seed).to(_device())
        u = torch.quasirandom.SobolEngine(dim, scramble=True, seed=seed).draw(case["n"], dtype=F64).to(_device())
        b = torch.clamp((u * bins).floor().long(), max=bins - 1)
        pts, jac = [], torch.ones_like(u[:, 0])
        for k in range(dim):
            left, right = e[k][b[:, k]], e[k][b[:, k] + 1]
            pts.append(left + (right - left) * (u[:, k] * bins - b[:, k]))
            jac = jac * bins * (right - left)
        flavours = 1 if case["mass"] > 1 else 3
        w = _exact_term(term, transverse, torch.stack(pts, 1), q2, x, case["mass"], 5.0, flavours, _gbw(seed)) * jac
        hist = torch.stack([torch.bincount(b[:, k], w.abs(), minlength=bins) for k in range(dim)])
        count = torch.stack([torch.bincount(b[:, k], minlength=bins) for k in range(dim)]).to(F64)
        out.append({"sums": torch.stack([w.sum(), (w * w).sum()]), "hist": hist, "count": count})
    return out
