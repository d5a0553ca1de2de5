"""Special functions and the DIS coupling in FP64 where a quotient or a
logarithm leaves the ordinary numbers."""

import math

import pytest
import torch

from nlo_bk_optimized_amd import device as dev
from nlo_bk_optimized_amd.dipole import GBW
from nlo_bk_optimized_amd.dis import DISConfig, Quark, QuarkType

pytestmark = pytest.mark.gpu
INF, NAN = math.inf, math.nan


# K2 ~ 2 / x^2 overflows below 1.1e-154; K1 ~ 1 / x below 5.6e-309
@pytest.mark.parametrize("fn,x,want", [
    ("K0", 0.0, INF), ("K1", 0.0, INF), ("K2", 0.0, INF), ("K1", 1e-300, 1e300), ("K1", 1e-310, INF),
    ("K2", 1e-150, 2e300), ("K2", 1e-155, INF), ("K2", 1e-200, INF), ("K2", 1e-308, INF),
    ("K0", 800.0, 0.0), ("K1", 800.0, 0.0), ("K2", INF, 0.0), ("K0", NAN, NAN), ("K0", -1.0, NAN),
    ("Li2", -INF, -INF), ("Li2", -1e308, -math.pi**2 / 6 - math.log(1e308) ** 2 / 2), ("Li2", 0.0, 0.0),
    ("Li2", 1.0, math.pi**2 / 6), ("Li2", NAN, NAN)])
def test_special_functions(fn, x, want):
    got = float(dev.dis_special(fn, torch.tensor([x], dtype=torch.float64).cuda())[0])
    if math.isnan(want):
        assert math.isnan(got)
    else:
        assert got == want or abs(got - want) <= 1e-14 * abs(want)


def test_coupling_at_its_pole():
    """At r = 2 / Lambda the logarithm is exactly 0: the coupling is frozen there
    as it is on both sides."""

    scale = 4.0 / (0.241 * 0.241)
    r = math.sqrt(scale)
    assert scale / (r * r) == 1.0
    quark = Quark(QuarkType.C, 1.4)
    values = []
    for size in (r * (1 - 1e-9), r, r * (1 + 1e-9)):
        desc = dev.dis_desc(10.0, 1e-3, True, (quark,), GBW(Qs0sqr=0.4, lambda_=0.25, gamma=1.0, x0=1.0),
                            DISConfig(quarks=(quark,), maxr=2.0 * size))
        point = torch.tensor([[0.5, 0.5]], dtype=torch.float64).cuda()
        values.append(float(dev.dis_integrand(desc, "T0", point)[0]))
    assert values[1] / values[0] == pytest.approx(1.0, rel=1e-6)
    assert values[1] / values[2] == pytest.approx(1.0, rel=1e-6)
