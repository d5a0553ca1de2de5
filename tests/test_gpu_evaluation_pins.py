"""Results of the FP64 kernels against recorded values of the plain evaluation:
samples whose terms cancel keep their digits, whatever the kernels share or
reorder elsewhere."""

from pathlib import Path

import numpy as np
import pytest

from tests.golden import make_evaluation_pins as pins

pytestmark = pytest.mark.gpu
GOLDEN = Path(pins.__file__).parent


def recorded(section: str) -> dict[str, np.ndarray]:
    with np.load(GOLDEN / f"{section}.npz") as f:
        return {k: f[k] for k in f.files}


def test_bk_sums_keep_the_formula():
    want, got = recorded("bk_fp64_sums"), pins.bk_sums()
    assert want.keys() == got.keys()
    for name in want:
        # about eps times the cancellation of the remaining steps (a factor up to
        # 1e5 in some samples); a reordered cancellation gives 1e-8 to 1e-7 here
        error = np.linalg.norm(got[name] - want[name]) / np.linalg.norm(want[name])
        assert error < 1e-11, (name, error)
