"""Results of the kernels against recorded values of the plain evaluation:
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


def test_bk_grids_to_the_last_bit():
    """An edge that moves by an ulp draws other roundings from the cancelling
    samples of every later pass, up to 5e-8 of an evolved amplitude."""

    want, got = recorded("bk_fp64_grids"), pins.bk_grids()
    assert want.keys() == got.keys()
    for name in want:
        assert np.array_equal(got[name], want[name]), name


def test_nested_terms_in_fp32():
    want, got = recorded("nested_fp32"), pins.nested_fp32()
    assert want.keys() == got.keys()
    for name in want:
        if name != "estimator":
            assert np.array_equal(got[name], want[name]), name
    # the estimator also sums I1, in FP64: its rounding reaches the FP32 terms
    # through the learned grids (edges of 1e-15) and the spread of seven
    # replicates; another rounding of the FP32 samples gives 4e-7 here and up to 1e-4 elsewhere
    error = np.abs(got["estimator"] / want["estimator"] - 1)
    assert error.max() < 1e-9, error


def test_dis_integrands_in_fp64():
    want, got = recorded("dis_fp64"), pins.dis_fp64()
    assert want.keys() == got.keys()
    for name in want:
        assert np.array_equal(got[name], want[name]), name


def test_dis_batch_refinement():
    want, got = recorded("dis_batch"), pins.dis_batch()
    assert want.keys() == got.keys()
    for name in want:
        # same samples, grids and order: only the rounding of the blocks' partial
        # sums differs, an eps each; a histogram rounded otherwise gives 1e-12 to 1e-8
        error = np.abs(got[name] / want[name] - 1).max()
        assert error < 1e-14, (name, error)
