// Host: renumbering the points of a Sobol block so that the 64 lanes of a wave
// hold neighbouring points.
//
// The points of an aligned block of 2^bits indices are shift ^ (high part) ^ g
// for g in the span of the block's direction numbers, one per index bit; the
// gray code of the index runs over the whole span.  Any invertible change of
// basis of that span gives the same set of points in another order, and the
// kernels only see it as other direction numbers.  The natural basis spreads
// 64 consecutive points over the whole cube (that is what a Sobol sequence is
// for), so nearly every wave takes both sides of every data-dependent branch.
// Here the six lane bits take combinations of directions that vanish in the
// leading bits of every dimension, as many as the block has room for: the
// lanes of a wave then share one small cell of the cube and branch together.
#pragma once

#include <cstdint>
#include <cstring>

#include "nlo_gfx950.h"

namespace nlo {

constexpr int kLaneBits = 6;  // 64 lanes

// The largest block worth reordering for points [first, first + n): aligned
// to first, and whole blocks holding 15/16 of the points (the rest keeps the
// natural order).  0: no such block.
inline int coherent_bits(int64_t first, int64_t n) {
    for (int bits = 24; bits > kLaneBits; --bits) {
        const int64_t size = (int64_t)1 << bits;
        if (first % size == 0 && (n >> bits << bits) >= n - n / 16) return bits;
    }
    return 0;
}

// The reordered direction numbers of t for blocks of 2^bits indices into
// out[dim][30].  Constraint k asks bit k / dim (from the top) of dimension
// k % dim of the lane directions to be zero; constraints are taken in this
// order while the lane directions keep six dimensions.
inline void coherent_order(const nlo_sobol_table& t, int dim, int bits, uint32_t (*out)[NLO_SOBOL_BITS]) {
    // the constraints as rows over the index bits, in reduced echelon form:
    // row[i] is the only one with bit pivot[i]
    uint32_t row[NLO_SOBOL_BITS];
    int pivot[NLO_SOBOL_BITS];
    int rank = 0;
    for (int k = 0; k < dim * NLO_SOBOL_BITS && rank < bits - kLaneBits; ++k) {
        const int top = NLO_SOBOL_BITS - 1 - k / dim;
        uint32_t f = 0;
        for (int b = 0; b < bits; ++b) f |= ((t.direction[k % dim][b] >> top) & 1u) << b;
        for (int i = 0; i < rank; ++i)
            if ((f >> pivot[i]) & 1u) f ^= row[i];
        if (f == 0) continue;  // follows from the others
        const int p = 31 - __builtin_clz(f);
        for (int i = 0; i < rank; ++i)
            if ((row[i] >> p) & 1u) row[i] ^= f;
        row[rank] = f;
        pivot[rank++] = p;
    }
    // new basis of the index bits: the solutions (one per free bit) first, the
    // unit vectors of the pivots after them; together they span every index
    uint32_t basis[NLO_SOBOL_BITS];
    uint32_t pivots = 0;
    for (int i = 0; i < rank; ++i) pivots |= 1u << pivot[i];
    int m = 0;
    for (int b = 0; b < bits; ++b) {
        if ((pivots >> b) & 1u) continue;
        uint32_t v = 1u << b;
        for (int i = 0; i < rank; ++i)
            if ((row[i] >> b) & 1u) v |= 1u << pivot[i];
        basis[m++] = v;
    }
    for (int i = 0; i < rank; ++i) basis[m++] = 1u << pivot[i];
    for (int d = 0; d < dim; ++d) {
        for (int i = 0; i < NLO_SOBOL_BITS; ++i) {
            uint32_t v = t.direction[d][i];
            if (i < bits) {
                v = 0;
                for (int b = 0; b < bits; ++b)
                    if ((basis[i] >> b) & 1u) v ^= t.direction[d][b];
            }
            out[d][i] = v;
        }
    }
}

}  // namespace nlo
