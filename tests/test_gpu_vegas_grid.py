"""Grid refinement on the device (nlo_vegas_adapt: parallel search of every
edge's interval) against a forward sweep over the cumulative sums, bit for bit:
bin counts below, at and above a wave and beyond the default LDS limit, flat and
peaked histograms, empty bins, an empty histogram, and sums that are no numbers."""

from __future__ import annotations

from fractions import Fraction

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _sweep(edges, hist, count, eps):
    bins = hist.size
    imp = hist / np.maximum(count, 1.0)
    sm = np.empty(bins)
    sm[0] = (imp[0] + imp[1]) / 2.0 + eps
    sm[-1] = (imp[-2] + imp[-1]) / 2.0 + eps
    for i in range(1, bins - 1):
        sm[i] = ((imp[i - 1] + imp[i]) + imp[i + 1]) / 3.0 + eps
    cum = np.concatenate([[0.0], np.empty(bins)])
    for i in range(bins):
        cum[i + 1] = cum[i] + sm[i]
    total = cum[-1]
    step = total / bins
    out, j = np.empty(bins + 1), 0
    for t in range(bins + 1):
        if not np.isfinite(total):
            target = np.nan
        elif t < (bins + 1) // 2:
            target = t * step
        else:  # one rounding, as a fused multiply-add
            target = float(Fraction(total) - Fraction(step) * (bins - t))
        while j < bins and target >= cum[j + 1]:
            j += 1
        b = min(j, bins - 1)
        out[t] = edges[b] + (target - cum[b]) / sm[b] * (edges[b + 1] - edges[b])
    out[0], out[-1] = 0.0, 1.0
    return out


@pytest.mark.parametrize("bins", [2, 3, 32, 63, 64, 65, 255, 2731, 4096])
def test_refined_edges_equal_a_forward_sweep(bins):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from nlo_bk_optimized_amd import device as dev

    print(f"vegas grid bins={bins}", flush=True)
    rng = np.random.default_rng(bins)
    eps = float(np.finfo(np.float64).eps)
    x = np.arange(bins)
    hist = np.stack([np.full(bins, 2.0), np.exp(-0.5 * ((x - bins / 3) / (1 + bins / 40)) ** 2),
                     rng.random(bins) * (rng.random(bins) < 0.2), np.zeros(bins),
                     np.where(x == bins // 2, np.nan, 1.0)])
    count = rng.integers(0, 5, hist.shape).astype(float)
    edges = np.sort(rng.random((hist.shape[0], bins + 1)), axis=1)
    edges[:, 0], edges[:, -1] = 0.0, 1.0

    def t(a):
        return torch.as_tensor(a, dtype=torch.float64, device="cuda")[None].contiguous()

    got = dev.vegas_adapt(t(edges), t(hist), t(count), eps).cpu().numpy().reshape(edges.shape)
    with np.errstate(invalid="ignore"):
        want = np.stack([_sweep(e, h, c, eps) for e, h, c in zip(edges, hist, count)])
    assert np.array_equal(got, want, equal_nan=True)


def test_threads_refine_grids_of_different_sizes():
    """Grids above the default LDS limit set the kernel's limit; threads with
    other sizes launch in between."""

    import threading

    from nlo_bk_optimized_amd import device as dev

    errors = []

    def refine(bins):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                hist = torch.rand((1, 1, bins), generator=torch.Generator().manual_seed(bins), dtype=torch.float64).cuda()
                count = torch.ones_like(hist)
                edges = torch.linspace(0, 1, bins + 1, dtype=torch.float64).reshape(1, 1, -1).cuda()
                first = dev.vegas_adapt(edges, hist, count, 1e-16)
                for _ in range(300):
                    out = dev.vegas_adapt(edges, hist, count, 1e-16)
                stream.synchronize()
                assert torch.equal(out, first)
        except Exception as e:  # noqa: BLE001
            errors.append((bins, e))

    threads = [threading.Thread(target=refine, args=(bins,)) for bins in (2800, 3400, 4096, 4000)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
