// tile_chol.h -- Cholesky factor and inverse of one 32 x 32 tile by one wave, in registers.
//
// Shared by the dense reduced system (dense.h) and the windows (window_kernels.h).
#pragma once

#include "lm_kernels.h"

namespace mba {

constexpr int kTile = 32;

// 1 / sqrt of the pivot held by `lane`; *bad when it is not positive and finite (then 1).
template <typename F>
__device__ __forceinline__ F tile_pivot(F column, int lane, bool* bad) {
    const F d = read_lane(column, lane);
    const bool nonpos = !(d > (F)0) || !isfinite((double)d);
    *bad |= nonpos;
    return inv_sqrt(nonpos ? (F)1 : d);
}

// Lane r < 32 holds row r of a symmetric tile (lower part) in a, lane 32 + i row i of the identity.  On
// return a holds row r of L (entries past the diagonal are not meaningful) and row i of L^-T (zero
// before the diagonal).  The column operations of the right-looking factorization, applied to the
// identity stacked below the tile, give L^-T, so the inverse costs no instructions of its own.  The
// entries l_cj of the scaled column j are read from their lanes with v_readlane.  The next column is
// updated first and its pivot's reciprocal root started, so that chain runs under the other columns'
// updates.  Bound by the chain of 32 columns (a reciprocal root and up to 31 broadcasts each); a step
// of the 2250 x 2250 factorization, which it sets the time of: 17.9 -> 10.1 us in FP64, 15.1 -> 8.7
// in FP32, against masked updates and an inverse by forward substitution afterwards.  Returns false
// when a pivot is not positive and finite.
template <typename F>
__device__ __forceinline__ bool potrf_stacked(F (&a)[kTile]) {
    bool bad = false;
    F inv = tile_pivot(a[0], 0, &bad);
#pragma unroll
    for (int j = 0; j < kTile; ++j) {
        a[j] *= inv;
        if (j + 1 < kTile) {
            a[j + 1] = fma(-a[j], read_lane(a[j], j + 1), a[j + 1]);
            inv = tile_pivot(a[j + 1], j + 1, &bad);
        }
#pragma unroll
        for (int c = j + 2; c < kTile; ++c) a[c] = fma(-a[j], read_lane(a[j], c), a[c]);
    }
    return !bad;
}

}  // namespace mba
