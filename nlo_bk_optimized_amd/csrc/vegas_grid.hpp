// VEGAS grid refinement for one dimension of one grid, shared by the
// standalone refinement kernel and the batched DIS integrator: the
// reference's operation order with no contraction, so both give the same
// bits.
#pragma once

#include <hip/hip_runtime.h>

namespace nlo {

// Importance of bin i: sum |w| / max(count, 1).
__device__ __forceinline__ double vegas_importance(const double* h, const double* c, int i) {
    return h[i] / fmax(c[i], 1.0);
}

// Smoothed importance of bin i (S/numerics/integration.py:828-833): 3-point
// mean inside, 2-point mean at the ends, plus eps.
__device__ __forceinline__ double vegas_smoothed(const double* h, const double* c, int bins, int i,
                                                 double eps) {
#pragma clang fp contract(off)
    double v;
    if (i == 0) {
        v = (vegas_importance(h, c, 0) + vegas_importance(h, c, 1)) / 2.0;
    } else if (i == bins - 1) {
        v = (vegas_importance(h, c, bins - 2) + vegas_importance(h, c, bins - 1)) / 2.0;
    } else {
        v = (vegas_importance(h, c, i - 1) + vegas_importance(h, c, i) + vegas_importance(h, c, i + 1)) /
            3.0;
    }
    return v + eps;
}

// _adapt_vegas_edges (S/numerics/integration.py:835-866) of one dimension:
// edges e[bins + 1], histogram hh[bins] and counts cc[bins] in, refined
// edges o[bins + 1] out (o must not alias e).  The linspace targets
// increase, and so do the cumulative sums, so searchsorted(cumulative, target,
// right) - 1 is the first interval whose end lies above the target.
//
// By the threads of one block (any number): the importances, the smoothing and
// each edge's search are parallel; the cumulative sums, whose order of addition
// fixes the bits, are one thread's.  scratch: kAdaptScratch(bins) doubles of
// LDS.  (One thread per row, with every value from global memory, took 58 us
// for a batch's grids and 124 us for 64 x 4 BK grids, a tenth of the runs that
// refine between short passes.)
__host__ __device__ constexpr int kAdaptScratch(int bins) { return 3 * bins + 2; }
constexpr int kMaxAdaptBins = 4096;

__device__ inline void vegas_adapt_block(const double* e, const double* hh, const double* cc, int bins, double eps,
                                         double* o, double* scratch) {
#pragma clang fp contract(off)
    double* sm = scratch;                // bins
    double* cum = scratch + bins;        // bins + 1
    double* ed = scratch + 2 * bins + 1;  // bins + 1
    for (int i = threadIdx.x; i < bins; i += blockDim.x) sm[i] = vegas_smoothed(hh, cc, bins, i, eps);
    for (int i = threadIdx.x; i <= bins; i += blockDim.x) ed[i] = e[i];
    __syncthreads();
    if (threadIdx.x == 0) {
        double total = 0.0;
        cum[0] = 0.0;
        for (int i = 0; i < bins; ++i) {
            total = total + sm[i];
            cum[i + 1] = total;
        }
    }
    __syncthreads();
    const double total = cum[bins], step = total / (double)bins;
    for (int t = threadIdx.x; t <= bins; t += blockDim.x) {
        const double target =
            t < (bins + 1) / 2 ? (double)t * step : fma(-step, (double)(bins - t), total);
        // largest j with cum[j] <= target (0 when a sum is no number)
        int lo = 0, hi = bins;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (target >= cum[mid])
                lo = mid;
            else
                hi = mid - 1;
        }
        const int b = lo < bins ? lo : bins - 1;
        const double frac = (target - cum[b]) / sm[b];
        o[t] = t == 0 ? 0.0 : (t == bins ? 1.0 : ed[b] + frac * (ed[b + 1] - ed[b]));
    }
}

}  // namespace nlo
