// tile_chol.h -- Cholesky factor and inverse of one 32 x 32 tile by one wave, in registers, and the
// factor and solve of a small system by one workgroup on top of it.
//
// Shared by the dense reduced system (dense.h) and the windows (window_kernels.h).
#pragma once

#include "lm_kernels.h"
#include "mfma.h"

namespace mba {

constexpr int kTile = 32;

// 1 / sqrt(d) for the pivot chain: the hardware estimate r and one third-order step r (1 + e / 2 + 3 e^2 / 8),
// e = 1 - d r^2, four dependent operations.  The step leaves out 5 e^3 / 16 and more: 2^-67 of the result for the
// FP64 estimate's 23 bits (|e| < 2^-22), and less for the FP32 one's, so the result is as good as
// the roundings of the step itself, about one unit in the last place.
__device__ __forceinline__ double pivot_rsqrt(double d) {
    const double r = __builtin_amdgcn_rsq(d), e = fma(-d * r, r, 1.0);
    return fma(r * e, fma(e, 0.375, 0.5), r);
}
__device__ __forceinline__ float pivot_rsqrt(float d) {
    const float r = __builtin_amdgcn_rsqf(d), e = fmaf(-d * r, r, 1.0f);
    return fmaf(r * e, fmaf(e, 0.375f, 0.5f), r);
}

// 1 / sqrt of the pivot held by `lane`; *bad when it is not positive and finite (the result is then not
// meaningful and the caller discards the tile).
template <typename F>
__device__ __forceinline__ F tile_pivot(F column, int lane, bool* bad) {
    const F d = read_lane(column, lane);
    *bad |= !(d > (F)0) || !isfinite((double)d);
    return pivot_rsqrt(d);
}

// The values of lanes 0-15 of v in every row of 16 lanes (lo), and those of lanes 16-31 (hi).
__device__ __forceinline__ void spread_rows(unsigned v, unsigned* lo, unsigned* hi) {
    const auto half = __builtin_amdgcn_permlane32_swap(v, v, false, false);              // lanes 0-31 twice
    const auto row = __builtin_amdgcn_permlane16_swap(half[0], half[0], false, false);  // its even, its odd rows
    *lo = row[0];
    *hi = row[1];
}
__device__ __forceinline__ void spread_rows(float v, float* lo, float* hi) {
    unsigned a, b;
    spread_rows((unsigned)__float_as_int(v), &a, &b);
    *lo = __int_as_float((int)a);
    *hi = __int_as_float((int)b);
}
__device__ __forceinline__ void spread_rows(double v, double* lo, double* hi) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    unsigned l0, l1, h0, h1;
    spread_rows((unsigned)b, &l0, &l1);
    spread_rows((unsigned)(b >> 32), &h0, &h1);
    *lo = __longlong_as_double((long long)(((unsigned long long)h0 << 32) | l0));
    *hi = __longlong_as_double((long long)(((unsigned long long)h1 << 32) | l1));
}

// acc += (lane LANE of each row of b) * x, one instruction.  The assembler form is needed because the
// compiler does not fold a row broadcast into a multiply-add.  b must have been written at least two
// wait states earlier: row_operands_ready gives them to the values as they are formed; the compiler, which does
// not know that the assembler form reads b by DPP, could only break it by copying b in between, and
// tests/test_code_objects.py looks for that in the compiled kernels.
template <int LANE>
__device__ __forceinline__ void fma_row_lane(double& acc, double b, double x) {
    asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(b), "v"(x), "n"(LANE));
}
template <int LANE>
__device__ __forceinline__ void fma_row_lane(float& acc, float b, float x) {
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(b), "v"(x), "n"(LANE));
}
template <typename F>
__device__ __forceinline__ void row_operands_ready(F& a, F& b) {
    asm("s_nop 1" : "+v"(a), "+v"(b));
}

// a[c] += l_cj * x for c = C .. 31, the multipliers l_cj in lo (rows 0-15 of the tile) and hi (16-31).
template <int C, typename F>
__device__ __forceinline__ void update_columns(F (&a)[kTile], F lo, F hi, F x) {
    if constexpr (C < kTile) {
        fma_row_lane<C % 16>(a[C], C < 16 ? lo : hi, x);
        update_columns<C + 1, F>(a, lo, hi, x);
    }
}

// Columns J .. 31 of potrf_stacked; inv is 1 / l_JJ.
template <int J, typename F>
__device__ __forceinline__ void factor_columns(F (&a)[kTile], F inv, bool* bad) {
    a[J] *= inv;
    if constexpr (J + 1 < kTile) {
        F lo, hi;
        spread_rows(a[J], &lo, &hi);
        row_operands_ready(lo, hi);
        const F x = -a[J];
        fma_row_lane<(J + 1) % 16>(a[J + 1], J + 1 < 16 ? lo : hi, x);
        inv = tile_pivot(a[J + 1], J + 1, bad);
        update_columns<J + 2, F>(a, lo, hi, x);
        factor_columns<J + 1, F>(a, inv, bad);
    }
}

// Lane r < 32 holds row r of a symmetric tile (lower part) in a, lane 32 + i row i of the identity.  On
// return a holds row r of L (entries past the diagonal are not meaningful) and row i of L^-T (zero
// before the diagonal).  The column operations of the right-looking factorization, applied to the
// identity stacked below the tile, give L^-T, so the inverse costs no instructions of its own.  The
// multipliers l_cj of column j are copied into every row of 16 lanes once per column and enter the
// updates as row-broadcast operands; the next column is updated first and its pivot's reciprocal root
// started, so that chain runs under the other columns' updates.  Bound by instruction issue, 7,300
// cycles a tile of which the chain alone takes 3,000 (multipliers by v_readlane: 11,700; through LDS: 10,900).
// A step of one tile column of the 2250 x 2250 factorization, whose time it set: 17.9 -> 7.0 us in FP64 (late steps), 15.1 -> 7.8 in FP32 (all),
// against masked updates with v_readlane and an inverse by forward substitution afterwards.  Returns
// false when a pivot is not positive and finite.
template <typename F>
__device__ __forceinline__ bool potrf_stacked(F (&a)[kTile]) {
    bool bad = false;
    const F inv = tile_pivot(a[0], 0, &bad);
    factor_columns<0, F>(a, inv, &bad);
    return !bad;
}

// ---------------------------------------------------------------------------------------------
// A small system (n unknowns) by one workgroup of NT threads, FP64: the lower triangle of S packed by
// rows, element (i, j) at i (i + 1) / 2 + j, with the right-hand side as row n.  Row n goes through the
// factorization like any other, so it ends as L^-1 b and only the backward sweep remains.
//
// Tiles of 32 columns.  Wave 0 factors a diagonal tile in registers (potrf_stacked) and leaves its
// inverse X in the tile's place (L_kk itself is not needed again); all waves turn the rows below into
// L_ik = A_ik X_k', 16 rows at a time; then the next diagonal tile is updated, and wave 0 factors it while
// the others update the rest, 16 x 16 blocks on the matrix cores: three barriers per tile, and the chain
// is the tile factors (about 3 us each) plus a panel and one block's update.  Every entry is updated by the tiles in order by one
// wave, so the result does not depend on the workgroup size or on where the triangle is kept.
//
// kGlobal: the triangle is in global memory (barriers then order global accesses too).

__host__ __device__ __forceinline__ constexpr int tri(int i) { return i * (i + 1) / 2; }
// Doubles of the packed triangle of n unknowns with its right-hand side row.
__host__ __device__ __forceinline__ constexpr int small_system_doubles(int n) { return tri(n + 1); }

template <bool kGlobal>
__device__ __forceinline__ void small_barrier() {
    if (kGlobal)
        __syncthreads();
    else
        lds_barrier();
}

// A 16 x 16 block of the trailing update: rows r0.. (up to n), columns c0.. (below n, lower part):
// -= L[.][kb, kb + 32) L[.][kb, kb + 32)'.
__device__ __forceinline__ void small_update(double* L, int n, int kb, int r0, int c0) {
    using M = Mfma<double>;
    const int l = threadIdx.x & 63, l16 = l & 15, q = l >> 4;
    const double* pa = L + tri(min(r0 + l16, n)) + kb + q;
    const double* pb = L + tri(min(c0 + l16, n)) + kb + q;
    double a[8], b[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        a[s] = pa[4 * s];
        b[s] = pb[4 * s];
    }
    typename M::acc c;
    bool in[4];
    double* pc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int r = r0 + M::row(l, e), cc = c0 + l16;
        in[e] = r <= n && cc <= r && cc < n;
        pc[e] = L + tri(in[e] ? r : 0) + (in[e] ? cc : 0);
        c[e] = *pc[e];
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) c = M::mma(-a[s], b[s], c);
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (in[e]) *pc[e] = c[e];
}

// The panel of the whole tile kb: rows r0, r0 + step, ... (16 at a time, up to n) become A X', in place.
__device__ __forceinline__ void small_panel(double* L, int n, int kb, int r0, int step) {
    using M = Mfma<double>;
    const int l = threadIdx.x & 63, l16 = l & 15, q = l >> 4;
    if (r0 > n) return;
    double b[2][8];  // X is lower triangular: zero past column cc of row cc (the triangle holds other rows there)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int cc = 16 * h + l16;
        const double* pb = L + tri(kb + cc) + kb + q;
#pragma unroll
        for (int s = 0; s < 4 + 4 * h; ++s) {
            const double v = pb[4 * s];
            b[h][s] = 4 * s + q <= cc ? v : 0.0;
        }
    }
    for (; r0 <= n; r0 += step) {
        const double* pa = L + tri(min(r0 + l16, n)) + kb + q;
        double a[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) a[s] = pa[4 * s];
        typename M::acc c[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if (s < 4) c[0] = M::mma(a[s], b[0][s], c[0]);
            c[1] = M::mma(a[s], b[1][s], c[1]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = r0 + M::row(l, e);
            double* row = L + tri(min(r, n)) + kb + l16;
            if (r <= n) {
                row[0] = c[0][e];
                row[16] = c[1][e];
            }
        }
    }
}

// X_k z (kTranspose: X_k' z) for the last or any tile's m entries z = x[kb ..], by one wave: lane r < m (of
// either half) gets entry r.  Half h of the wave takes entries k = 16 h .. 16 h + 15 of the sum.
template <bool kTranspose>
__device__ __forceinline__ double small_tile_times(const double* L, int kb, int m, const double* z) {
    const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5, rr = min(r, m - 1);
    double v[16], x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int k = min(16 * h + i, m - 1);
        const int a = kTranspose ? k : rr, b = kTranspose ? min(rr, k) : min(k, rr);
        v[i] = L[tri(kb + a) + kb + b];
        x[i] = z[k];
    }
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int k = 16 * h + i;
        s = fma(k < m && (kTranspose ? r <= k : k <= r) ? v[i] : 0.0, x[i], s);
    }
    return s + __shfl_xor(s, 32, 64);
}

// Wave 0: factors diagonal tile kb (m columns) and stores its inverse there.
__device__ __forceinline__ void small_diag(double* L, int kb, int m, int* bad) {
    const int l = threadIdx.x & 63, r = l & 31;
    double a[kTile];
#pragma unroll
    for (int c = 0; c < kTile; ++c) a[c] = l == kTile + c ? 1.0 : 0.0;
    if (m == kTile) {
        // the whole row: entries past the diagonal are the next rows' (not meaningful, still in the triangle)
        const double* row = L + tri(kb + r) + kb;
        if (l < kTile)
#pragma unroll
            for (int c = 0; c < kTile; ++c) a[c] = row[c];
    } else {
        const double* row = L + tri(kb + min(r, m - 1)) + kb;
        if (l < kTile)
#pragma unroll
            for (int c = 0; c < kTile; ++c) {
                const double v = row[min(c, min(r, m - 1))];
                a[c] = r < m && c <= r ? v : (r == c ? 1.0 : 0.0);  // rows past m: the identity
            }
    }
    if (!potrf_stacked<double>(a) && l == 0) *bad = 1;
    if (l >= kTile)
#pragma unroll
        for (int i = 0; i < kTile; ++i)
            if (r <= i && i < m) L[tri(kb + i) + kb + r] = a[i];
}

template <int NT, bool kGlobal>
__device__ __forceinline__ void small_factor(double* L, int n, int* bad) {
    constexpr int NW = NT / 64;
    static_assert(NW > 3, "three waves update the next diagonal tile");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wave == 0) small_diag(L, 0, min(kTile, n), bad);
    for (int kb = 0; kb < n; kb += kTile) {
        const int m = min(kTile, n - kb), next = kb + m;
        small_barrier<kGlobal>();
        if (next >= n) {  // the right-hand side is the only row left
            if (wave == 0) {
                double* z = L + tri(n) + kb;
                const double y = small_tile_times<false>(L, kb, m, z);
                wave_sync_lds();
                if ((int)threadIdx.x < m) z[threadIdx.x] = y;
            }
            small_barrier<kGlobal>();
            break;
        }
        small_panel(L, n, kb, next + 16 * wave, 16 * NW);
        small_barrier<kGlobal>();
        const int T = (n - next) / 16 + 1, blocks = T * (T + 1) / 2;  // 16-row blocks of rows next .. n
        // block t is row block ti, column block tk: (0, 0), (1, 0), (1, 1) are the next diagonal tile
        if (wave < min(3, blocks)) small_update(L, n, kb, next + 16 * ((wave + 1) / 2), next + 16 * (wave / 2));
        small_barrier<kGlobal>();
        if (wave == 0) {
            small_diag(L, next, min(kTile, n - next), bad);
        } else {
            for (int t = 2 + wave; t < blocks; t += NW - 1) {
                int ti = (int)((sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f);
                while ((ti + 1) * (ti + 2) / 2 <= t) ++ti;
                while (ti * (ti + 1) / 2 > t) --ti;
                small_update(L, n, kb, next + 16 * ti, next + 16 * (t - ti * (ti + 1) / 2));
            }
        }
    }
}

// Row n (L^-1 b) <- L^-T of it: tiles from the last, x_k = X_k' z_k by wave 0, then z -= L_k.' x_k above, a
// thread per row (a tile's first column is at most 256), its 32 entries of L requested before x_k is
// there.
template <int NT, bool kGlobal>
__device__ __forceinline__ void small_backward(double* L, int n) {
    static_assert(NT >= 256, "one thread per row above a tile");
    __shared__ __align__(16) double xk[kTile];
    const int tid = threadIdx.x;
    double* x = L + tri(n);
    for (int kb = ((n - 1) / kTile) * kTile; kb >= 0; kb -= kTile) {
        const int m = min(kTile, n - kb);
        double lv[kTile];
        if (tid < kb)
#pragma unroll
            for (int c = 0; c < kTile; ++c) lv[c] = L[tri(kb + min(c, m - 1)) + tid];
        if (tid < 64) {
            const double s = small_tile_times<true>(L, kb, m, x + kb);
            wave_sync_lds();
            if (tid < kTile) xk[tid] = tid < m ? s : 0.0;
            if (tid < m) x[kb + tid] = s;
        }
        small_barrier<kGlobal>();
        if (tid < kb) {
            double s = 0.0;
#pragma unroll
            for (int c = 0; c < kTile; ++c) s = fma(lv[c], xk[c], s);
            x[tid] -= s;
        }
        small_barrier<kGlobal>();
    }
}

// Copies the lower triangle of a row-major S (leading dimension ld) and the right-hand side b into the
// packed triangle: a wave takes R rows at a time, all their loads in flight together (n <= 64 C = 320).
template <int NT>
__device__ __forceinline__ void small_load(const double* __restrict__ S, int ld, const double* __restrict__ b, int n, double* L) {
    constexpr int NW = NT / 64, R = 8, C = 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    for (int r0 = R * wave; r0 <= n; r0 += R * NW) {
        const int last = min(r0 + R - 1, n - 1);  // the longest row's last column
        double v[R][C];
#pragma unroll
        for (int k = 0; k < C; ++k)
            if (64 * k <= last)
#pragma unroll
                for (int g = 0; g < R; ++g) {
                    const int r = min(r0 + g, n);
                    const double* row = r < n ? S + (size_t)r * ld : b;
                    v[g][k] = row[min(64 * k + lane, last)];
                }
#pragma unroll
        for (int k = 0; k < C; ++k)
            if (64 * k <= last)
#pragma unroll
                for (int g = 0; g < R; ++g)
                    if (r0 + g <= n && 64 * k + lane <= min(r0 + g, n - 1)) L[tri(r0 + g) + 64 * k + lane] = v[g][k];
    }
}

}  // namespace mba
