// dense.h -- explicit reduced camera system and its dense Cholesky solve (the DENSE_SCHUR /
// SPARSE_SCHUR step of test_bundle_adjustment_ceres.cpp:97 for problems up to a few hundred cameras).
//
//   S = U* - sum_points sum_{i,j in track} W~_i Vinv_p W~_j'     (9 nc x 9 nc, FP64)
// is assembled without atomics.  The diagonal block of a camera that sees no point twice is the
// Schur-Jacobi block k_rhs_cam forms anyway, D_a^2 + sum J~'(I - G)J~.  For the others the ordered
// observation pairs (i, j) of a point with camera(i) <= camera(j) are listed per camera block (a, b)
// once per problem; one workgroup owns one 9x9 block and reduces its pair list in a fixed order
// (pair_block.h, the products the batched windows use too).  A pair contributes
// Jc~_i' (Hp_i Jp~_j') Jc~_j with Hp_i = Jp~_i Vinv_p, i.e. a 2x2 middle factor.
//
// The factorization is a tiled right-looking Cholesky (32 x 32 tiles), two tile columns a step: a
// diagonal tile is factored by one wave and its triangular inverse kept, the panel below is multiplied
// by that inverse (TRSM as a small GEMM) and the trailing lower tiles are updated (SYRK/GEMM); the
// products run on the matrix cores (v_mfma_f64_16x16x4f64, v_mfma_f32_16x16x4f32), and the trailing
// update also factors the next pair of diagonal tiles, so a step is one launch.  The panel is stored
// transposed in the upper tiles (the factorization reads only the lower ones; in FP64 the factor
// overwrites S).  The triangular solves work on diagonal blocks of sixteen tiles whose
// inverses are formed after the factorization: two launches per block and sweep, each a
// matrix-vector product over many workgroups.  In mixed precision the factor is
// FP32 and the step is refined in FP64 against the FP64 S (refine_steps iterations of
// r = b - S y, y += S_f^-1 r).
#pragma once

#include <algorithm>
#include <cmath>
#include <vector>

#include "lm_kernels.h"
#include "mfma.h"
#include "pair_block.h"
#include "solver.h"
#include "tile_chol.h"

namespace mba {

constexpr int kJs = 36;  // per-observation stride of Jc~ (18, by columns), Jp~ (6), Hp (6), I - G (3)
static_assert(kJs == RecLayout<kRecDense>::stride, "the dense record is pair_block's kRecDense");

// S <- the cameras' Schur-Jacobi blocks M_c (k_rhs_cam: D_c^2 plus every observation with itself) on the
// diagonal, zero elsewhere, an identity tail on the padding diagonal: kFillPerBlock entries a workgroup, in the
// launch of the records (a launch of its own, and one that wrote the solve's iteration count, were 15 us of a
// four-iteration solve of 8 cameras in 485).
constexpr int kFillPerBlock = 16 * kWG;
__device__ __forceinline__ void fill_S(double* __restrict__ S, int n, int ld, const double* __restrict__ M, int block) {
    const size_t end = std::min((size_t)ld * ld, (size_t)(block + 1) * kFillPerBlock);
    for (size_t i = (size_t)block * kFillPerBlock + threadIdx.x; i < end; i += kWG) {
        const int r = (int)(i / ld), c = (int)(i % ld);
        double v = (r == c && r >= n) ? 1.0 : 0.0;
        if (r < n && c < n && r / 9 == c / 9) v = M[81 * (size_t)(r / 9) + 9 * (r % 9) + c % 9];
        S[i] = v;
    }
}

// The pair products' records (kRecDense).  `parts` workgroups share a camera's observations: with one, 49
// cameras of 640 observations leave most of the chip idle (28 us against 10.5).  Bound by the stores: by the
// lanes that form the records, 48 us in FP64 and 32 in FP32 at 250 cameras and 1M observations, through LDS
// 40 and 18.  FP64 is held to three wavefronts a SIMD, not four: the g2o model's 134 registers then stay
// registers (10.0 us at 49 cameras, 10.5 with six of 128 spilled); the others need no more than 128.
template <typename Real, int M>
__global__ void __launch_bounds__(kWG, sizeof(Real) == 8 ? 3 : 4) k_dense_store(Dev<Real> d, Real* __restrict__ js, int parts, int n_store,
                                                        double* __restrict__ S, int n, int ld) {
    LMState* st = d.st;
    if (st->done || st->step_invalid) return;
    __shared__ Unit16 lds[kWaves][64 * kRecordRow];
    constexpr bool f64 = sizeof(Real) == 8;  // a record is two rows then, J~_c and the rest, else one
    if ((int)blockIdx.x >= n_store) {  // the workgroups after the records' fill S
        fill_S(S, n, ld, d.M, (int)blockIdx.x - n_store);
        return;
    }
    const int per_part = n_store / parts, part = blockIdx.x / per_part;
    const int c = xcd_remap(blockIdx.x - part * per_part, d.nc);
    if (c >= d.nc) return;
    const CameraPrep<Real> P = d.prep[c];
    Real sc[9];
    for (int i = 0; i < 9; ++i) sc[i] = (Real)d.sc[9 * (size_t)c + i];
    const int end = d.cam_off[c + 1], wave = threadIdx.x >> 6;
    // rounds of a workgroup's observations, every lane taking part in the stores
    for (int j0 = d.cam_off[c] + kWG * part + 64 * wave; j0 < end; j0 += kWG * parts) {
        const int j = j0 + (threadIdx.x & 63);
        Real Jc[18];
#pragma unroll
        for (int i = 0; i < 18; ++i) Jc[i] = (Real)0;
        if (j < end) {
            int p;
            Real r[2], Jp[6], h[6], ig[3];
            corrected_jacobian<Real, M>(d, P, j, p, r, Jc, Jp);
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                Jc[i] *= sc[i];
                Jc[9 + i] *= sc[i];
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const Real s = (Real)d.sp[3 * (size_t)p + i];
                Jp[i] *= s;
                Jp[3 + i] *= s;
            }
            sym3_mul<Real>(d.VinvR + 6 * (size_t)p, Jp, h);
            sym3_mul<Real>(d.VinvR + 6 * (size_t)p, Jp + 3, h + 3);
            point_complement<Real, Real>(d, p, Jp, ig[0], ig[1], ig[2]);
            const int at = f64 ? 0 : 9;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                stage_pair<Real>(lds[wave], at + i, Jp[2 * i], Jp[2 * i + 1]);
                stage_pair<Real>(lds[wave], at + 3 + i, h[2 * i], h[2 * i + 1]);
            }
            stage_pair<Real>(lds[wave], at + 6, ig[0], ig[1]);
            stage_pair<Real>(lds[wave], at + 7, ig[2], (Real)0);
            stage_pair<Real>(lds[wave], at + 8, (Real)0, (Real)0);
        }
        const int rows = min(64, end - j0);
        Real* out = js + kJs * (size_t)j0;
        if (f64) flush_records<kJs * (int)sizeof(Real) / 16, 9>(lds[wave], out, 9, rows);
#pragma unroll
        for (int i = 0; i < 9; ++i) stage_pair<Real>(lds[wave], i, Jc[i], Jc[9 + i]);  // the rows of column i adjacent
        flush_records<kJs * (int)sizeof(Real) / 16, 9>(lds[wave], out, 0, rows);
    }
}

// ---------------------------------------------------------------------------------------------
// Observation pairs of the camera blocks, built on the device from the camera-order point indices
// (ascending within a camera): for block (a, b) the pairs (i, j) with camera(i) = a, camera(j) = b and
// one point, in order of i, then j.  One wave per block finds each of camera a's points in camera b's
// list by binary search (the list, a few KB, stays in the wave's L1); blocks whose point ranges do not
// overlap end at once.  Two passes, counts and then the pairs at the offsets the host lays out from
// the counts: 0.25 ms for 250 cameras and 3.7M pairs, against 25 ms for enumerating them per point on one
// host thread.

// Number of observations [*first, *first + n) of the list co_pt[lo, hi) at point p.
__device__ __forceinline__ int find_point(const int* __restrict__ co_pt, int lo, int hi, int p, int* first) {
    const int end = hi;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (co_pt[mid] < p)
            lo = mid + 1;
        else
            hi = mid;
    }
    *first = lo;
    int n = 0;
    while (lo + n < end && co_pt[lo + n] == p) ++n;
    return n;
}

// count[a nc + b], a <= b: pairs of block (a, b); a == b counts every observation with itself.
__global__ void __launch_bounds__(kWG) k_pair_count(const int* __restrict__ cam_off, const int* __restrict__ co_pt, int nc,
                                                    int* __restrict__ count) {
    const int64_t t = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
    const int a = (int)(t / nc), b = (int)(t % nc), lane = threadIdx.x & 63;
    if (a >= nc || b < a) return;
    const int a0 = cam_off[a], a1 = cam_off[a + 1], b0 = cam_off[b], b1 = cam_off[b + 1];
    int n = 0;
    if (a1 > a0 && b1 > b0 && co_pt[a0] <= co_pt[b1 - 1] && co_pt[b0] <= co_pt[a1 - 1])
        for (int i = a0 + lane; i < a1; i += 64) {
            int first;
            n += find_point(co_pt, b0, b1, co_pt[i], &first);
        }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) n += __shfl_xor(n, m, 64);
    if (lane == 0) count[(size_t)a * nc + b] = n;
}

// The pairs of every listed block (camera a, camera b, first pair, end pair; camera -1: padding).
__global__ void __launch_bounds__(kWG) k_pair_emit(const int* __restrict__ cam_off, const int* __restrict__ co_pt,
                                                   const int4* __restrict__ blk, int nblocks, int2* __restrict__ pairs) {
    const int t = blockIdx.x * kWaves + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= nblocks) return;
    const int4 bk = blk[t];
    if (bk.x < 0) return;
    const int a1 = cam_off[bk.x + 1], b0 = cam_off[bk.y], b1 = cam_off[bk.y + 1];
    int out = bk.z;
    for (int i0 = cam_off[bk.x]; i0 < a1; i0 += 64) {
        const int i = i0 + lane;
        int first = 0, n = 0;
        if (i < a1) n = find_point(co_pt, b0, b1, co_pt[i], &first);
        int before = n;  // pairs of this round's earlier observations
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const int o = __shfl_up(before, m, 64);
            if (lane >= m) before += o;
        }
        const int total = __shfl(before, 63, 64);
        before -= n;
        for (int k = 0; k < n; ++k)
            if (out + before + k < bk.w) pairs[out + before + k] = make_int2(i, first + k);
        out += total;
    }
}

// One 9x9 block of the reduced camera system per workgroup of NW waves (the blocks' pair lists, the
// 36-value records of k_dense_store): pair_block in pair_block.h.  Bound by LDS accesses and the products'
// instructions once the blocks of neighbouring cameras run on one XCD; FP64 by its two wavefronts a SIMD
// (238 registers) as well, FP32 is held to the three its 168 allow.  At 250 cameras and 4.2M pairs 325 us (blocks
// in key order over all XCDs, the cameras' own blocks among them), 188 FP64 and 199 FP32 with sixteen
// pairs a stage, 156 and 99 with 32; at 49 cameras 78, 37 and 29 us, for a window of 8 cameras 62, 5.5 and 5.8.
template <typename Real, int NW>
constexpr size_t schur_blocks_lds() {
    return (size_t)NW * pair_stage_bytes<Real, kRecDense>() + (NW > 1 ? NW * 81 * sizeof(double) : 0);
}

template <typename Real, int NW>
__global__ void __launch_bounds__(64 * NW, sizeof(Real) == 4 ? 3 : 2) k_schur_blocks(Dev<Real> d, const Real* __restrict__ js,
                                                          const int4* __restrict__ blk, const int2* __restrict__ pairs,
                                                          double* __restrict__ S, int ld) {
    LMState* st = d.st;
    if (st->done || st->step_invalid) return;
    extern __shared__ __align__(16) unsigned char schur_lds_mem[];
    const int4 bk = blk[blockIdx.x];
    if (bk.x < 0) return;  // padding of an XCD's list
    constexpr int kStage = pair_stage_bytes<Real, kRecDense>();
    pair_block<Real, kRecDense, NW>(bk, pairs, js, d.dc2, S, ld,
                                    reinterpret_cast<Real*>(schur_lds_mem + (size_t)(threadIdx.x >> 6) * kStage),
                                    reinterpret_cast<double*>(schur_lds_mem + (size_t)NW * kStage));
}

// The FP32 copy of S that is factored: the lower 64 x 64 blocks, one workgroup each, 16 rows of four values a
// thread and turn; the factorization writes the upper tiles before anything reads them.  Bound by memory: 33 MB
// in 6.2 us at 2250 unknowns (5.2 TB/s), where the whole matrix, one value a thread, took 13.1 us (64 MB).
__global__ void __launch_bounds__(kWG) k_convert_S(const double* __restrict__ S, float* __restrict__ A, int ld, const LMState* st) {
    if (st->done || st->step_invalid) return;
    const int b = blockIdx.x;
    int i = (int)((sqrt(8.0 * b + 1.0) - 1.0) * 0.5);
    while ((i + 1) * (i + 2) / 2 <= b) ++i;
    while (i * (i + 1) / 2 > b) --i;
    const int j = b - i * (i + 1) / 2;
    const size_t first = (size_t)(64 * i + threadIdx.x / 16) * ld + 64 * j + 4 * (threadIdx.x % 16);
    static_assert(kWG == 256, "16 rows of 16 threads");
    double2 v[4][2];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const double2* src = reinterpret_cast<const double2*>(S + first + (size_t)(16 * t) * ld);
        v[t][0] = src[0];
        v[t][1] = src[1];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
        *reinterpret_cast<float4*>(A + first + (size_t)(16 * t) * ld) =
            make_float4((float)v[t][0].x, (float)v[t][0].y, (float)v[t][1].x, (float)v[t][1].y);
}

// ---------------------------------------------------------------------------------------------
// 32 x 32 tile products on the matrix cores.  A 16 x 16 block of the product X Y' of two 32-column
// tiles is one wave's eight v_mfma 16x16x4 steps: lane l supplies eight values of row row0 + l%16 of X
// and of row col0 + l%16 of Y (Mfma::load_row), the four lanes of a row cover it and every k in [0, 32)
// enters exactly once.  Accumulator element i of
// lane l is entry (row(l, i), l%16) of the block; the FP64 and FP32 instructions order rows
// differently.

// c + sign * X[16 si .., :] Y[16 sj .., :]' for 32-column tiles X (leading dimension ldx) and Y (ldy);
// rows start 8-element aligned.
template <typename F>
__device__ __forceinline__ typename Mfma<F>::acc tile_mma_nt(const F* __restrict__ X, int ldx, const F* __restrict__ Y,
                                                             int ldy, int si, int sj, typename Mfma<F>::acc c, F sign) {
    const int l = threadIdx.x & 63, q = l >> 4, r = l & 15;
    F xv[8], yv[8];
    Mfma<F>::load_row(X + (size_t)(16 * si + r) * ldx, q, xv);
    Mfma<F>::load_row(Y + (size_t)(16 * sj + r) * ldy, q, yv);
#pragma unroll
    for (int s = 0; s < 8; ++s) c = Mfma<F>::mma(sign * xv[s], yv[s], c);
    return c;
}

// A lane's operand of such a product, loaded ahead of it.
template <typename F>
__device__ __forceinline__ void tile_operand(const F* __restrict__ Y, int ldy, int sj, F (&yv)[8]) {
    Mfma<F>::load_row(Y + (size_t)(16 * sj + (threadIdx.x & 15)) * ldy, (threadIdx.x & 63) >> 4, yv);
}

// Factors the tile held in T (lower triangle used) with one wave and writes X = L^-1 (Dinv[k],
// row-major, zero above the diagonal); L itself is not kept, nothing reads a factored diagonal tile.
// Lane r < 32 keeps row r of the tile in registers, lane 32 + i row i of the identity: the column
// operations that turn the tile into L (column j scaled by 1 / l_jj, column c less l_cj times column j)
// turn the identity below it into L^-T, whose row i is column i of X, so the inverse costs no
// instructions of its own (potrf_stacked).  Entries above the tile's diagonal are
// updated with the rest and never read by another lane.  Returns false (and writes nothing) when a
// pivot is not positive and finite.  Only one whole wave may call it.  T has rows of kTile + 1, X of ldx.
template <typename F>
__device__ __forceinline__ bool potrf_tile_wave(const F* T, F* X, int ldx) {
    const int l = threadIdx.x & 63, r = l & 31;
    F a[kTile];
#pragma unroll
    for (int c = 0; c < kTile; ++c) a[c] = l == kTile + c ? (F)1 : (F)0;
    if (l < kTile)
#pragma unroll
        for (int c = 0; c < kTile; ++c) a[c] = T[r * (kTile + 1) + c];
    if (!potrf_stacked<F>(a)) return false;
    if (l >= kTile)
#pragma unroll
        for (int m = 0; m < kTile; ++m) X[m * ldx + r] = a[m];
    return true;
}

// LDS tiles of the kernels below: rows start 16-byte aligned.
template <typename F>
constexpr int kLdsPitch = kTile + 16 / (int)sizeof(F);
template <typename F>
constexpr int kLdsTile = kTile * kLdsPitch<F>;
constexpr int kStepThreads = 512;
template <typename F>
constexpr size_t step_pair_lds() {
    return 8 * kLdsTile<F> * sizeof(F);
}

// Factors the 64 x 64 diagonal block of tiles t, t + 1 from its tiles T00, T11 (rows of kTile + 1) and T10
// (kLdsPitch) in LDS; X is one tile more.  Leaves X_t and X_t+1 in Dinv and L_t+1,t in the lower tile (t + 1, t),
// transposed also in the upper one.  All kStepThreads threads call it, before a barrier on the tiles; all
// but the first wave run idle() while that factors tile t.  A pivot that fails sets step_invalid to `mark`.
template <typename F, typename Idle>
__device__ __forceinline__ void factor_pair(F* T00, F* T10, F* T11, F* X, F* __restrict__ A, int ld, int t,
                                            F* __restrict__ Dinv, LMState* st, int mark, Idle idle) {
    constexpr int PP = kLdsPitch<F>;
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, si = (w >> 1) & 1, sj = w & 1;
    lds_barrier();
    if (w > 0)
        idle();
    else if (!potrf_tile_wave<F>(T00, X, PP) && l == 0)
        st->step_invalid = mark;
    lds_barrier();
    F* L = T00;  // L_t+1,t takes its place, rows of kLdsPitch
    if (w < 4) {
        typename Mfma<F>::acc p = {0, 0, 0, 0};
        p = tile_mma_nt<F>(T10, PP, X, PP, si, sj, p, (F)1);
#pragma unroll
        for (int e = 0; e < 4; ++e) L[(16 * si + Mfma<F>::row(l, e)) * PP + 16 * sj + (l & 15)] = p[e];
    } else {
        for (int idx = threadIdx.x - 256; idx < kTile * kTile; idx += 256)
            Dinv[(size_t)t * kTile * kTile + idx] = X[(idx / kTile) * PP + idx % kTile];
    }
    lds_barrier();
    if (w >= 4) {
        F* low = A + (size_t)(kTile * (t + 1)) * ld + kTile * t;
        F* up = A + (size_t)(kTile * t) * ld + kTile * (t + 1);
        for (int idx = threadIdx.x - 256; idx < kTile * kTile; idx += 256) {
            const int a = idx / kTile, b = idx % kTile;
            low[(size_t)a * ld + b] = L[a * PP + b];
            up[(size_t)a * ld + b] = L[b * PP + a];
        }
    } else if (si >= sj) {
        typename Mfma<F>::acc c = {0, 0, 0, 0};
        F* mine = T11 + (16 * si) * (kTile + 1) + 16 * sj + (l & 15);
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = mine[Mfma<F>::row(l, e) * (kTile + 1)];
        c = tile_mma_nt<F>(L, PP, L, PP, si, sj, c, (F)-1);
#pragma unroll
        for (int e = 0; e < 4; ++e) mine[Mfma<F>::row(l, e) * (kTile + 1)] = c[e];
    }
    lds_barrier();
    if (w == 0 && !potrf_tile_wave<F>(T11, Dinv + (size_t)(t + 1) * kTile * kTile, kTile) && l == 0) st->step_invalid = mark;
}

// The first diagonal block (later ones are factored by the trailing update).
template <typename F>
__global__ void __launch_bounds__(kStepThreads) k_potrf_pair(F* __restrict__ A, int ld, F* __restrict__ Dinv, LMState* st) {
    if (st->done || st->step_invalid) return;
    extern __shared__ __align__(16) unsigned char step_lds_mem[];
    F* const lds = reinterpret_cast<F*>(step_lds_mem);
    F *T00 = lds, *T10 = lds + kLdsTile<F>, *T11 = lds + 2 * kLdsTile<F>;
    for (int idx = threadIdx.x; idx < kTile * kTile; idx += kStepThreads) {
        const int a = idx / kTile, b = idx % kTile;
        T00[a * (kTile + 1) + b] = A[(size_t)a * ld + b];
        T10[a * kLdsPitch<F> + b] = A[(size_t)(kTile + a) * ld + b];
        T11[a * (kTile + 1) + b] = A[(size_t)(kTile + a) * ld + kTile + b];
    }
    factor_pair<F>(T00, T10, T11, lds + 3 * kLdsTile<F>, A, ld, 0, Dinv, st, 1, [] {});
}

// Step K of the factorization in one launch: tile columns k = 2 K and k + 1, one workgroup per lower 64 x 64
// block (I, J) of the trailing matrix, K < J <= I.  The panel tiles the update needs are formed in the
// workgroup from the unscaled A_ik, A_i,k+1 (rows of I and of J) and the kept inverses:
//   L_ik = A_ik X_k',   L_i,k+1 = (A_i,k+1 - L_ik L_k+1,k') X_k+1',
// staged in LDS, and A_ij -= L_ik L_jk' + L_i,k+1 L_j,k+1' follows, each wave on one 16 x 16 block of two
// tiles: the products and sums of two steps of one tile column each, in their order.  The workgroups of
// block column K + 1 store L' in the upper tiles, which the factorization does not read; the lower tiles of
// columns k and k + 1 still hold what other workgroups of this launch read, and k_panel_down copies the
// transposes into them once the factorization is done.  Block 0 (dispatched first) keeps its tiles in LDS
// and factors them, so the next step's diagonal factors cost no launch of their own.  A step is bound by
// that workgroup's chain, two tile factors (3 us each) behind two panels.  One launch per tile column paid the
// launch, the first loads and the trailing matrix's read and write twice: at 2250 unknowns the factorization
// took 832 us in FP64 and 552 in FP32, against 660 and 463; at 441, where the trailing matrix is small, 100
// against 104.
template <typename F>
__global__ void __launch_bounds__(kStepThreads, 4) k_step_pair(F* __restrict__ A, int ld, int K, F* __restrict__ Dinv,
                                                               LMState* st) {
    // Workgroup 0 may mark the step invalid while others start: the mark of this launch is left to later ones, so that
    // every wave of a workgroup decides alike.
    const int mark = K + 2, invalid = st->step_invalid;
    if (st->done || (invalid != 0 && invalid != mark)) return;
    constexpr int PP = kLdsPitch<F>, TS = kLdsTile<F>;
    extern __shared__ __align__(16) unsigned char step_lds_mem[];
    F* const P = reinterpret_cast<F*>(step_lds_mem);  // tiles 0-3: L_.k of the rows of I, J; 4-7: L_.,k+1
    const int b = blockIdx.x, w = threadIdx.x >> 6, l = threadIdx.x & 63;
    int ii = (int)((sqrt(8.0 * b + 1.0) - 1.0) * 0.5);
    while ((ii + 1) * (ii + 2) / 2 <= b) ++ii;
    while (ii * (ii + 1) / 2 > b) --ii;
    const int jj = b - ii * (ii + 1) / 2;
    const int k = 2 * K, i0 = k + 2 + 2 * ii, j0 = k + 2 + 2 * jj;  // first tiles of the step, of I and of J
    const bool diag = ii == jj;
    const int half = w >> 2, si = (w >> 1) & 1, sj = w & 1;
    // Panels: each wave a strip of 16 rows of I (waves 0-3) or of J (4-7, none on the diagonal), whose
    // operands pass from product to product through the strip's LDS rows, between the wave's own lanes.
    using Acc = typename Mfma<F>::acc;
    const int l16 = l & 15;
    if (w < 4 || !diag) {
        const int tile = (w >> 1) & 1, strip = w & 1, slot = 2 * (w >> 2) + tile;
        const F* row = A + (size_t)(kTile * ((w < 4 ? i0 : j0) + tile)) * ld + kTile * k;
        F xv[8], y[2][8];
        Acc p[2], a2[2];
        tile_operand<F>(row, ld, strip, xv);
#pragma unroll
        for (int sj = 0; sj < 2; ++sj) tile_operand<F>(Dinv + (size_t)k * kTile * kTile, kTile, sj, y[sj]);
#pragma unroll
        for (int sj = 0; sj < 2; ++sj)
#pragma unroll
            for (int e = 0; e < 4; ++e) a2[sj][e] = row[(size_t)(16 * strip + Mfma<F>::row(l, e)) * ld + kTile + 16 * sj + l16];
        F y2[2][8];
#pragma unroll
        for (int sj = 0; sj < 2; ++sj) tile_operand<F>(A + (size_t)(kTile * (k + 1)) * ld + kTile * k, ld, sj, y2[sj]);
        F* out = P + slot * TS + 16 * strip * PP + l16;
#pragma unroll
        for (int sj = 0; sj < 2; ++sj) {
            p[sj] = Acc{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < 8; ++s) p[sj] = Mfma<F>::mma(xv[s], y[sj][s], p[sj]);
#pragma unroll
            for (int e = 0; e < 4; ++e) out[Mfma<F>::row(l, e) * PP + 16 * sj] = p[sj][e];
        }
#pragma unroll
        for (int sj = 0; sj < 2; ++sj) tile_operand<F>(Dinv + (size_t)(k + 1) * kTile * kTile, kTile, sj, y[sj]);
        wave_sync_lds();
        tile_operand<F>(P + slot * TS, PP, strip, xv);
        out += 4 * TS;
#pragma unroll
        for (int sj = 0; sj < 2; ++sj) {
#pragma unroll
            for (int s = 0; s < 8; ++s) a2[sj] = Mfma<F>::mma(-xv[s], y2[sj][s], a2[sj]);
#pragma unroll
            for (int e = 0; e < 4; ++e) out[Mfma<F>::row(l, e) * PP + 16 * sj] = a2[sj][e];
        }
        wave_sync_lds();
        tile_operand<F>(P + (4 + slot) * TS, PP, strip, xv);
        wave_sync_lds();
#pragma unroll
        for (int sj = 0; sj < 2; ++sj) {
            p[sj] = Acc{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < 8; ++s) p[sj] = Mfma<F>::mma(xv[s], y[sj][s], p[sj]);
#pragma unroll
            for (int e = 0; e < 4; ++e) out[Mfma<F>::row(l, e) * PP + 16 * sj] = p[sj][e];
        }
    }
    // block (si, sj) of tile (i0 + u, j0 + v), less its products
    const F* Pj = P + (diag ? 0 : 2) * TS;
    auto load_block = [&](int u, int v, int si, int sj) {
        Acc c;
        const F* Aij = A + (size_t)(kTile * (i0 + u) + 16 * si) * ld + kTile * (j0 + v) + 16 * sj + l16;
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = Aij[(size_t)Mfma<F>::row(l, e) * ld];
        return c;
    };
    auto update_block = [&](int u, int v, int si, int sj, Acc c) {
        c = tile_mma_nt<F>(P + u * TS, PP, Pj + v * TS, PP, si, sj, c, (F)-1);
        return tile_mma_nt<F>(P + (4 + u) * TS, PP, Pj + (4 + v) * TS, PP, si, sj, c, (F)-1);
    };
    auto store_panel = [&](int first, int threads) {
        for (int idx = first; idx < 4 * kTile * kTile; idx += threads) {
            const int t = idx / (kTile * kTile), cc = idx / kTile % kTile, rr = idx % kTile;  // t: (column, row tile)
            A[(size_t)(kTile * (k + (t >> 1)) + cc) * ld + kTile * (i0 + (t & 1)) + rr] =
                P[(4 * (t >> 1) + (t & 1)) * TS + rr * PP + cc];
        }
    };
    if (b > 0) {
        Acc c[2];
        bool own[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            own[u] = !diag || u > half || (u == half && si >= sj);
            if (own[u]) c[u] = load_block(u, half, si, sj);
        }
        lds_barrier();
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (!own[u]) continue;
            c[u] = update_block(u, half, si, sj, c[u]);
            F* Aij = A + (size_t)(kTile * (i0 + u) + 16 * si) * ld + kTile * (j0 + half) + 16 * sj + l16;
#pragma unroll
            for (int e = 0; e < 4; ++e) Aij[(size_t)Mfma<F>::row(l, e) * ld] = c[u][e];
        }
        if (jj == 0) store_panel(threadIdx.x, kStepThreads);
        return;
    }
    // The next diagonal block, in LDS tiles that a diagonal workgroup's panels do not use.  Tile (0, 0) first,
    // by three waves; the others' blocks and the panel's store run while it is factored.
    F *T00 = P + 2 * TS, *T10 = P + 3 * TS, *T11 = P + 6 * TS;
    // waves 0-2: (0, 0) of tile (0, 0), then blocks (0, 0), (1, 0), (1, 1) of tile (1, 1) in waves 1-3; 4-7: tile (1, 0)
    auto put = [&](F* T, int pitch, int bi, int bj, Acc c) {
        F* out = T + 16 * bi * pitch + 16 * bj + l16;
#pragma unroll
        for (int e = 0; e < 4; ++e) out[Mfma<F>::row(l, e) * pitch] = c[e];
    };
    const int bi0 = w > 0, bj0 = w > 1;  // wave's block of tile (0, 0)
    const int bi1 = w > 1, bj1 = w > 2;  // and of tile (1, 1)
    Acc c0 = {0, 0, 0, 0}, c1 = {0, 0, 0, 0};
    if (w < 3) c0 = load_block(0, 0, bi0, bj0);
    if (w > 3)
        c1 = load_block(1, 0, si, sj);
    else if (w > 0)
        c1 = load_block(1, 1, bi1, bj1);
    lds_barrier();
    if (w < 3) put(T00, kTile + 1, bi0, bj0, update_block(0, 0, bi0, bj0, c0));
    factor_pair<F>(T00, T10, T11, P + 7 * TS, A, ld, k + 2, Dinv, st, mark, [&] {
        if (w > 3)
            put(T10, PP, si, sj, update_block(1, 0, si, sj, c1));
        else
            put(T11, kTile + 1, bi1, bj1, update_block(1, 1, bi1, bj1, c1));
        store_panel(threadIdx.x - 64, kStepThreads - 64);
    });
}

// After the factorization: L_ik = (tile (k, i))' into the lower tile (i, k), i > k (one workgroup per
// tile; the triangular sweeps and the block inverses read the lower tiles).
template <typename F>
__global__ void __launch_bounds__(256) k_panel_down(F* __restrict__ A, int ld, const LMState* st) {
    if (st->done || st->step_invalid) return;
    __shared__ F T[kTile][kTile + 1];
    const int b = blockIdx.x;
    int ii = (int)((sqrt(8.0 * b + 1.0) - 1.0) * 0.5);
    while ((ii + 1) * (ii + 2) / 2 <= b) ++ii;
    while (ii * (ii + 1) / 2 > b) --ii;
    const int k = b - ii * (ii + 1) / 2, i = ii + 1;  // k < i
    const F* Aki = A + (size_t)(kTile * k) * ld + kTile * i;
    F* Aik = A + (size_t)(kTile * i) * ld + kTile * k;
    for (int idx = threadIdx.x; idx < kTile * kTile; idx += 256) T[idx / kTile][idx % kTile] = Aki[(size_t)(idx / kTile) * ld + idx % kTile];
    lds_barrier();
    for (int idx = threadIdx.x; idx < kTile * kTile; idx += 256) Aik[(size_t)(idx / kTile) * ld + idx % kTile] = T[idx % kTile][idx / kTile];
}

// ---------------------------------------------------------------------------------------------
// Triangular solves.  The factor is cut into diagonal blocks of kSolveBlk tiles (512 rows); after the
// factorization k_block_inverse forms each block's inverse X = L_KK^-1, so a block of either sweep is
// one matrix-vector product with X (or X') and one with the panel below (above) it, both spread over
// the chip at one wave per kSweepRows rows.  A system of at most 512 unknowns is solved by two
// launches; 2250 unknowns by 18 (with 128-row blocks, whose product and panel one workgroup formed one
// after the other, the sweeps were 36 launches of 10-12 us: 405 us per solve against 80 us).
constexpr int kSolveBlk = 16;
constexpr int kSolveRows = kSolveBlk * kTile;

// Tiles of block K: [kSolveBlk K, min(kSolveBlk (K + 1), nt)).
__host__ __device__ __forceinline__ int solve_block_tiles(int K, int nt) {
    return nt - kSolveBlk * K < kSolveBlk ? nt - kSolveBlk * K : kSolveBlk;
}

// One workgroup per (block K, 16 columns of X = L_KK^-1): with j their tile, X_jj = Dinv_j and
// X_ij = -Dinv_i sum_{j<=k<i} L_ik X_kj for i = j+1, ... in order, in FP64 on the matrix cores.  The
// columns found so far are kept in LDS transposed (rows of X_kj' are the products' second operand);
// wave (row half si = w % 2, quarter w / 2) forms a 16 x 16 block of the sum over every fourth k, the
// quarters are added, and the first two waves multiply by Dinv_i.  L_ik is requested while row i - 1 is
// finished.  What bounds it is one CU's rate of reading L (measured in a copy with clock stamps: with 32
// columns a workgroup, whose column halves read L twice, issuing the loads took 40% of the time), hence
// the narrow columns: the five blocks of 2250 rows 97 -> 54 us in FP64, 75 -> 45 us in FP32.  X is stored row-major and transposed (XT), so
// both sweeps read rows; tiles above the diagonal are neither written nor read.
constexpr int kInvPitch = kTile + 2;
constexpr int kInvThreads = 512;
constexpr int kInvCols = 16;
inline size_t block_inverse_lds(int nt) {
    return ((size_t)(std::min(nt, kSolveBlk) + 1) * kInvCols * kInvPitch + 6 * 256) * sizeof(double);
}

// A lane's eight operands of a 32-column row stored in F, in the columns Mfma<double>::load_row takes.
template <typename F>
__device__ __forceinline__ void load_row_f64(const F* __restrict__ row, int q, F (&v)[8]) {
    const R2v<F>* p = reinterpret_cast<const R2v<F>*>(row) + q;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const R2v<F> t = p[4 * i];
        v[2 * i] = t.x;
        v[2 * i + 1] = t.y;
    }
}

template <typename F>
__global__ void __launch_bounds__(kInvThreads) k_block_inverse(const F* __restrict__ A, int ld, const F* __restrict__ Dinv,
                                                               F* __restrict__ Binv, F* __restrict__ BinvT, int nt,
                                                               const LMState* st) {
    if (st->done || st->step_invalid) return;
    extern __shared__ __align__(16) double inv_lds[];
    using M = Mfma<double>;
    constexpr int kHalves = kTile / kInvCols, kQuarters = 4;
    const int K = blockIdx.x / (kSolveBlk * kHalves), col = blockIdx.x % (kSolveBlk * kHalves);
    const int j = col / kHalves, bt = solve_block_tiles(K, nt), t0 = kSolveBlk * K;
    if (j >= bt) return;
    constexpr int TS = kInvCols * kInvPitch;  // doubles of a tile's 16 columns in LDS
    double* part = inv_lds;                   // partial sums of quarters 1-3, by lane
    double* Tt = inv_lds + 6 * 256;           // the sum, transposed
    double* Xc = Tt + TS;                     // X_ij' for i = j, j + 1, ...
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, q = l >> 4, c16 = l & 15;
    const int si = w & 1, quarter = w >> 1, cs = kInvCols * col;  // first column within the block
    F* X = Binv + (size_t)K * kSolveRows * kSolveRows;
    F* XT = BinvT + (size_t)K * kSolveRows * kSolveRows;
    {
        const int r = tid / kInvCols, c = tid % kInvCols;
        const F v = Dinv[(size_t)(t0 + j) * kTile * kTile + r * kTile + cs % kTile + c];
        X[(size_t)(kTile * j + r) * kSolveRows + cs + c] = v;
        Xc[c * kInvPitch + r] = (double)v;
    }
    // this wave's operands of row i: L_ik for its k = j + quarter + 4 m
    constexpr int kMine = kSolveBlk / kQuarters;
    F lr[kMine][8];
    auto request = [&](int i) {
        const F* Lrow = A + (size_t)(kTile * (t0 + i) + 16 * si + c16) * ld + kTile * t0;
#pragma unroll
        for (int m = 0; m < kMine; ++m)
            if (j + quarter + kQuarters * m < i) load_row_f64<F>(Lrow + kTile * (j + quarter + kQuarters * m), q, lr[m]);
    };
    if (j + 1 < bt) request(j + 1);
    lds_barrier();
    for (int i = j + 1; i < bt; ++i) {
        F dv[8];  // the row of Dinv_i the last product needs
        if (quarter == 0) load_row_f64<F>(Dinv + (size_t)(t0 + i) * kTile * kTile + (16 * si + c16) * kTile, q, dv);
        typename M::acc c = {0, 0, 0, 0};
#pragma unroll
        for (int m = 0; m < kMine; ++m) {
            const int k = j + quarter + kQuarters * m;
            if (k < i) {
                double xv[8];
                M::load_row(Xc + (size_t)(k - j) * TS + c16 * kInvPitch, q, xv);
#pragma unroll
                for (int s = 0; s < 8; ++s) c = M::mma((double)lr[m][s], xv[s], c);
            }
        }
        if (i + 1 < bt) request(i + 1);
        if (quarter > 0)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[((quarter - 1) * 2 + si) * 256 + e * 64 + l] = c[e];
        lds_barrier();
        if (quarter == 0)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                double t = c[e];
#pragma unroll
                for (int h = 0; h < 3; ++h) t += part[(h * 2 + si) * 256 + e * 64 + l];
                Tt[c16 * kInvPitch + 16 * si + M::row(l, e)] = t;
            }
        lds_barrier();
        if (quarter == 0) {
            double tv[8];
            M::load_row(Tt + c16 * kInvPitch, q, tv);
            typename M::acc x = {0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < 8; ++s) x = M::mma(-(double)dv[s], tv[s], x);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = 16 * si + M::row(l, e);
                X[(size_t)(kTile * i + r) * kSolveRows + cs + c16] = (F)x[e];
                Xc[(size_t)(i - j) * TS + c16 * kInvPitch + r] = x[e];
            }
        }
        lds_barrier();
    }
    const int rows = kTile * (bt - j);
    for (int e = tid; e < kInvCols * rows; e += kInvThreads) {
        const int cc = e / rows, r = e % rows;
        XT[(size_t)(cs + cc) * kSolveRows + kTile * j + r] = (F)Xc[(size_t)(r / kTile) * TS + cc * kInvPitch + r % kTile];
    }
}

// Dot products of kSweepRows consecutive rows with v, by one wave: s[g] = sum_{c in [c0, c1)}
// M[row0 + g][c] v[c] (every lane gets the sums).  Lane l takes columns c0 + l, + 64, ...; the loads of
// 256 columns of all rows are in flight together, with clamped columns (v = 0 there) and rows
// instead of branches around the loads.
constexpr int kSweepRows = 4;

template <typename F>
__device__ __forceinline__ void sweep_dot(const F* __restrict__ M, size_t ldm, int row0, int last_row, int c0, int c1,
                                          const double* __restrict__ v, int v_end, double (&s)[kSweepRows]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int g = 0; g < kSweepRows; ++g) s[g] = 0.0;
    for (int cb = c0; cb < c1; cb += 256) {
        F m[kSweepRows][4];
        double x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = cb + lane + 64 * u, cc = min(c, c1 - 1);
            const double t = v[min(cc, v_end - 1)];
            x[u] = c < c1 && c < v_end ? t : 0.0;
#pragma unroll
            for (int g = 0; g < kSweepRows; ++g) m[g][u] = M[(size_t)min(row0 + g, last_row) * ldm + cc];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int g = 0; g < kSweepRows; ++g) s[g] = fma((double)m[g][u], x[u], s[g]);
    }
#pragma unroll
    for (int g = 0; g < kSweepRows; ++g) s[g] = wave_sum(s[g]);
}

// Forward sweep, block K: y_K = X_K rhs_K (rhs: b for block 0, which has n entries; z afterwards).
template <typename F>
__global__ void __launch_bounds__(kWG) k_fwd_solve(const F* __restrict__ Binv, int nt, int K, const double* __restrict__ rhs,
                                                   int n, double* __restrict__ y, const LMState* st) {
    if (st->done || st->step_invalid) return;
    const int rows = kTile * solve_block_tiles(K, nt), kb = kSolveRows * K;
    const int r0 = kSweepRows * (blockIdx.x * kWaves + (threadIdx.x >> 6));
    if (r0 >= rows) return;
    double s[kSweepRows];
    sweep_dot<F>(Binv + (size_t)K * kSolveRows * kSolveRows, kSolveRows, r0, rows - 1, 0, kTile * (r0 / kTile + 1), rhs + kb,
                 n - kb, s);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int g = 0; g < kSweepRows; ++g) y[kb + r0 + g] = s[g];
}

// Rows below block K: z = rhs - L_{.K} y_K (rhs: b for block 0, z itself afterwards).
template <typename F>
__global__ void __launch_bounds__(kWG) k_fwd_rows(const F* __restrict__ A, int ld, int K, const double* rhs, int n,
                                                  const double* __restrict__ y, double* z, const LMState* st) {
    if (st->done || st->step_invalid) return;
    const int kb = kSolveRows * K;
    const int r0 = kb + kSolveRows + kSweepRows * (blockIdx.x * kWaves + (threadIdx.x >> 6));
    if (r0 >= ld) return;
    double s[kSweepRows];
    sweep_dot<F>(A + kb, ld, r0, ld - 1, 0, kSolveRows, y + kb, kSolveRows, s);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int g = 0; g < kSweepRows; ++g) z[r0 + g] = (r0 + g < n ? rhs[r0 + g] : 0.0) - s[g];
}

// Backward sweep, block K: t_K = X_K' y_K, also into x (added to it when accumulate != 0; rows below
// n only).
template <typename F>
__global__ void __launch_bounds__(kWG) k_bwd_solve(const F* __restrict__ BinvT, int nt, int K, const double* __restrict__ y,
                                                   double* __restrict__ t, double* __restrict__ x, int n, int accumulate,
                                                   int solves, LMState* st) {
    if (st->done || st->step_invalid) return;
    if (K == 0 && blockIdx.x == 0 && threadIdx.x == 0) st->pcg_iters = solves;  // linear solver iterations
    const int rows = kTile * solve_block_tiles(K, nt), kb = kSolveRows * K;
    const int r0 = kSweepRows * (blockIdx.x * kWaves + (threadIdx.x >> 6));
    if (r0 >= rows) return;
    double s[kSweepRows];
    sweep_dot<F>(BinvT + (size_t)K * kSolveRows * kSolveRows, kSolveRows, r0, rows - 1, kTile * (r0 / kTile), rows, y + kb, rows,
                 s);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int g = 0; g < kSweepRows; ++g) {
            const int row = kb + r0 + g;
            t[row] = s[g];
            if (row < n) x[row] = accumulate ? x[row] + s[g] : s[g];
        }
}

// Rows above block K: y -= L_{K.}' t_K, from the transposed panels in the upper tiles.
template <typename F>
__global__ void __launch_bounds__(kWG) k_bwd_rows(const F* __restrict__ A, int ld, int nt, int K, const double* __restrict__ t,
                                                  double* __restrict__ y, const LMState* st) {
    if (st->done || st->step_invalid) return;
    const int rows = kTile * solve_block_tiles(K, nt), kb = kSolveRows * K;
    const int r0 = kSweepRows * (blockIdx.x * kWaves + (threadIdx.x >> 6));
    if (r0 >= kb) return;
    double s[kSweepRows];
    sweep_dot<F>(A + kb, ld, r0, kb - 1, 0, rows, t + kb, rows, s);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int g = 0; g < kSweepRows; ++g) y[r0 + g] -= s[g];
}

// r = b - S y (FP64, S symmetric with its full n x n block stored); one wave per row.
__global__ void __launch_bounds__(kWG) k_residual(const double* __restrict__ S, int ld, const double* __restrict__ b,
                                                  const double* __restrict__ y, double* __restrict__ r, int n,
                                                  const LMState* st) {
    if (st->done || st->step_invalid) return;
    const int row = blockIdx.x * kWaves + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= n) return;
    double v = 0.0;
    for (int c = lane; c < n; c += 64) v += S[(size_t)row * ld + c] * y[c];
    v = wave_sum(v);
    if (lane == 0) r[row] = b[row] - v;
}

// The whole factor and solve of a small reduced system by one workgroup (tile_chol.h): S's lower
// triangle and b packed into LDS.  One launch in place of the tile steps, the block inverse and the sweeps.
constexpr int kSmallThreads = 512;
__global__ void __launch_bounds__(kSmallThreads) k_dense_small(const double* __restrict__ S, int ld, const double* __restrict__ b,
                                                               double* __restrict__ x, int n, LMState* st) {
    if (st->done || st->step_invalid) return;
    extern __shared__ __align__(16) double small_lds[];
    __shared__ int bad;
    if (threadIdx.x == 0) bad = 0;
    small_load<kSmallThreads>(S, ld, b, n, small_lds);
    lds_barrier();
    small_factor<kSmallThreads, false>(small_lds, n, &bad);
    if (bad) {
        if (threadIdx.x == 0) st->step_invalid = 1;
        return;
    }
    small_backward<kSmallThreads, false>(small_lds, n);
    for (int k = threadIdx.x; k < n; k += kSmallThreads) x[k] = small_lds[tri(n) + k];
    if (threadIdx.x == 0) st->pcg_iters = 1;  // linear solver iterations
}

// Reduced systems up to this size are factored in FP64 in both precisions: the factor costs a few
// microseconds there, and an FP32 factor of a small, nearly gauge-free system (a local window whose
// trust region has grown) would need a Krylov solve on top to reach the FP64 step.
constexpr int kDenseF64MaxN = 288;
// Systems up to this size (22 cameras, 159 KB of LDS) are factored and solved by one workgroup: 26 us at 8
// cameras and 71 at 22, against 35 and 85 for the tile steps, block inverse and sweeps; past it the
// triangle does not fit the LDS.
constexpr int kDenseSmallN = 198;

template <typename Real>
struct DenseSchur {
    int n = 0, ld = 0, nt = 0, nb = 0, nblocks = 0, refine = 0;
    bool f64 = true;  // factor in FP64 (FP64 solver, or a small system)
    DevBuf<Real> js;
    DevBuf<int4> blk;
    int store_parts = 1;  // workgroups of k_dense_store per camera
    int schur_waves = 2;  // waves per block of the pair products
    DevBuf<int2> pairs;
    DevBuf<double> S, r, z, y;
    DevBuf<float> Af, Dinvf, Binvf, BinvTf;
    DevBuf<double> Dinvd, Binvd, BinvTd;
    int64_t device_bytes() const {
        return js.bytes() + blk.bytes() + pairs.bytes() + S.bytes() + r.bytes() + z.bytes() + y.bytes() + Af.bytes() +
               Dinvf.bytes() + Binvf.bytes() + BinvTf.bytes() + Dinvd.bytes() + Binvd.bytes() + BinvTd.bytes();
    }

    // The blocks the pair kernel forms, from their pair counts: those of two different cameras that share
    // a point, and a camera's own block when it observes a point more than once (pairs x != y, which M_c
    // does not hold; the pair kernel then writes the whole block).  In launch order: workgroup k runs
    // on XCD k % 8; each XCD takes a contiguous eighth (by pairs) of the blocks sorted by groups of four
    // cameras on either side, so that the records of eight cameras, read once per pair, are re-read
    // from its own L2.  Padding entries have camera -1.
    int block_list(const Layout& L, const std::vector<int>& count, std::vector<int4>* out, int64_t* n_pairs) {
        constexpr int G = 4;
        const int nc = L.nc;
        std::vector<int4> take;  // pair counts in z until the offsets are known
        int64_t total = 0;
        for (int ga = 0; ga < nc; ga += G)
            for (int gb = ga; gb < nc; gb += G)
                for (int a = ga; a < std::min(ga + G, nc); ++a)
                    for (int b = std::max(gb, a); b < std::min(gb + G, nc); ++b) {
                        const int c = count[(size_t)a * nc + b];
                        if (a == b ? c == L.cam_off[a + 1] - L.cam_off[a] : c == 0) continue;
                        take.push_back(make_int4(a, b, c, 0));
                        total += c;
                    }
        if (total > INT32_MAX) return fail(BA_ERR_CAPACITY, "%lld observation pairs in the reduced system", (long long)total);
        std::vector<std::vector<int4>> xq(kXcds);
        int64_t seen = 0;
        for (const int4& t : take) {
            const int x = (int)std::min<int64_t>(kXcds - 1, (seen + t.z / 2) * kXcds / std::max<int64_t>(total, 1));
            xq[x].push_back(make_int4(t.x, t.y, (int)seen, (int)(seen + t.z)));
            seen += t.z;
        }
        size_t longest = 0;
        for (const auto& q : xq) longest = std::max(longest, q.size());
        out->assign(longest * kXcds, make_int4(-1, -1, 0, 0));
        for (int x = 0; x < kXcds; ++x)
            for (size_t k = 0; k < xq[x].size(); ++k) (*out)[k * kXcds + x] = xq[x][k];
        *n_pairs = total;
        // A workgroup of eight waves fills a CU's LDS with its staging areas, so it is taken only while
        // every block still has a CU of its own (28 blocks of 380 pairs: 5.8 us against 6.5 with four
        // waves).  Two waves otherwise: four such workgroups share a CU.
        schur_waves = (int)take.size() <= kCUs ? 8 : 2;
        return BA_OK;
    }

    // cam_off, co_pt: the solver's device copies of the layout's arrays, uploaded on s.
    int create(const Layout& L, const int* cam_off, const int* co_pt, const ba_options& o, hipStream_t s) {
        const int nc = L.nc;
        n = 9 * nc;
        nt = 2 * std::max(1, (n + 2 * kTile - 1) / (2 * kTile));  // whole 64 x 64 blocks
        ld = nt * kTile;
        nb = (nt + kSolveBlk - 1) / kSolveBlk;
        // two workgroups a CU, while a camera has rounds to share
        int most = 0;
        for (int c = 0; c < nc; ++c) most = std::max(most, L.cam_off[c + 1] - L.cam_off[c]);
        store_parts = std::max(1, std::min((2 * kCUs + nc - 1) / std::max(nc, 1), (most + kWG - 1) / kWG));
        f64 = sizeof(Real) == sizeof(double) || n <= kDenseF64MaxN;
        refine = f64 ? 0 : std::max(0, o.refine_steps);
        if (nc > 0) {
            DevBuf<int> dcount;
            std::vector<int> count((size_t)nc * nc);
            std::vector<int4> list;
            int64_t n_pairs = 0;
            BA_TRY(dcount.alloc(count.size()));
            hipLaunchKernelGGL(k_pair_count, dim3(div_up((int64_t)count.size(), kWaves)), dim3(kWG), 0, s, cam_off, co_pt, nc,
                               dcount.p);
            BA_HIP(hipGetLastError());
            BA_HIP(hipMemcpyAsync(count.data(), dcount.p, count.size() * sizeof(int), hipMemcpyDeviceToHost, s));
            BA_HIP(hipStreamSynchronize(s));
            BA_TRY(block_list(L, count, &list, &n_pairs));
            nblocks = (int)list.size();
            BA_TRY(blk.upload(list.data(), list.size(), s));
            BA_TRY(pairs.alloc((size_t)n_pairs));
            if (nblocks)
                hipLaunchKernelGGL(k_pair_emit, dim3(div_up(nblocks, kWaves)), dim3(kWG), 0, s, cam_off, co_pt,
                                   (const int4*)blk.p, nblocks, pairs.p);
            BA_HIP(hipGetLastError());
            BA_HIP(hipStreamSynchronize(s));
        }
        BA_TRY(js.alloc(kJs * (size_t)std::max(L.no, 1)));
        BA_TRY(S.alloc((size_t)ld * ld));
        BA_TRY(r.alloc(ld));
        BA_TRY(z.alloc(ld));
        BA_TRY(y.alloc(ld));
        const size_t binv = (size_t)nb * kSolveRows * kSolveRows;
        if (n <= kDenseSmallN) {
            BA_TRY(allow_dynamic_lds((const void*)k_dense_small, (int)(small_system_doubles(n) * sizeof(double))));
        } else if (f64) {
            BA_TRY(Dinvd.alloc((size_t)nt * kTile * kTile));
            BA_TRY(Binvd.alloc(binv));
            BA_TRY(BinvTd.alloc(binv));
            BA_TRY(allow_dynamic_lds((const void*)k_block_inverse<double>, (int)block_inverse_lds(nt)));
            BA_TRY(allow_dynamic_lds((const void*)k_potrf_pair<double>, (int)step_pair_lds<double>()));
            BA_TRY(allow_dynamic_lds((const void*)k_step_pair<double>, (int)step_pair_lds<double>()));
        } else {
            BA_TRY(Af.alloc((size_t)ld * ld));
            BA_TRY(Dinvf.alloc((size_t)nt * kTile * kTile));
            BA_TRY(Binvf.alloc(binv));
            BA_TRY(BinvTf.alloc(binv));
            BA_TRY(allow_dynamic_lds((const void*)k_block_inverse<float>, (int)block_inverse_lds(nt)));
        }
        BA_TRY(allow_dynamic_lds((const void*)k_schur_blocks<Real, 8>, (int)schur_blocks_lds<Real, 8>()));
        BA_HIP(hipStreamSynchronize(s));
        return BA_OK;
    }

    // x = (L L')^-1 b (accumulate: x += ...) by the blocked sweeps.
    template <typename F, typename SolverT>
    void solve(SolverT& sv, const F* A, const F* Binv, const F* BinvT, const double* b, double* x, int accumulate) {
        const LMState* st = sv.d.st;
        const int per = kSweepRows * kWaves;  // rows of a workgroup
        for (int K = 0; K < nb; ++K) {
            const double* rhs = K == 0 ? b : z.p;
            const int lim = K == 0 ? n : ld;
            sv.launch("fwd_solve", k_fwd_solve<F>, div_up(kTile * solve_block_tiles(K, nt), per), kWG, Binv, nt, K, rhs, lim,
                      y.p, st);
            const int below = ld - kSolveRows * (K + 1);
            if (below > 0)
                sv.launch("fwd_rows", k_fwd_rows<F>, div_up(below, per), kWG, A, ld, K, rhs, lim, (const double*)y.p, z.p, st);
        }
        for (int K = nb - 1; K >= 0; --K) {
            sv.launch("bwd_solve", k_bwd_solve<F>, div_up(kTile * solve_block_tiles(K, nt), per), kWG, BinvT, nt, K,
                      (const double*)y.p, z.p, x, n, accumulate, 1 + refine, sv.d.st);
            if (K > 0)
                sv.launch("bwd_rows", k_bwd_rows<F>, div_up(kSolveRows * K, per), kWG, A, ld, nt, K, (const double*)z.p, y.p, st);
        }
    }

    template <typename F, typename SolverT>
    void factor_and_solve(SolverT& sv, F* A, F* Dinv, F* Binv, F* BinvT) {
        auto& d = sv.d;
        sv.launch_shm("potrf", k_potrf_pair<F>, 1, kStepThreads, step_pair_lds<F>(), A, ld, Dinv, d.st);
        for (int K = 0; K + 1 < nt / 2; ++K) {
            const int m = nt / 2 - 1 - K;
            sv.launch_shm("step", k_step_pair<F>, m * (m + 1) / 2, kStepThreads, step_pair_lds<F>(), A, ld, K, Dinv, d.st);
        }
        sv.launch("panel_down", k_panel_down<F>, nt * (nt - 1) / 2, 256, A, ld, (const LMState*)d.st);
        sv.launch_shm("block_inverse", k_block_inverse<F>, nb * kSolveRows / kInvCols, kInvThreads, block_inverse_lds(nt), (const F*)A, ld,
                      (const F*)Dinv, Binv, BinvT, nt, (const LMState*)d.st);
        solve<F>(sv, A, Binv, BinvT, (const double*)d.bc, d.px, 0);
        for (int it = 0; it < refine; ++it) {
            sv.launch("residual", k_residual, div_up(n, kWaves), kWG, (const double*)S.p, ld, (const double*)d.bc,
                      (const double*)d.px, r.p, n, (const LMState*)d.st);
            solve<F>(sv, A, Binv, BinvT, (const double*)r.p, d.px, 1);
        }
    }

    template <int NW, typename SolverT>
    void enqueue_schur(SolverT& sv) {
        sv.launch_shm("schur_pairs", k_schur_blocks<Real, NW>, nblocks, 64 * NW, schur_blocks_lds<Real, NW>(), sv.d,
                      (const Real*)js.p, (const int4*)blk.p, (const int2*)pairs.p, S.p, ld);
    }

    template <typename SolverT>
    void enqueue_solve(SolverT& sv) {
        auto& d = sv.d;
        const int nc = d.nc;
        const size_t nn = (size_t)ld * ld;
        const int n_store = xcd_grid(nc) * store_parts;
        sv.launch("dense_store",
                  pick_model(d.model, k_dense_store<Real, kModelSnavely>, k_dense_store<Real, kModelSnavelyG2o>,
                             k_dense_store<Real, kModelStereo>),
                  n_store + (int)((nn + kFillPerBlock - 1) / kFillPerBlock), kWG, d, js.p, store_parts, n_store, S.p, n, ld);
        if (schur_waves == 8)
            enqueue_schur<8>(sv);
        else
            enqueue_schur<2>(sv);
        if (n <= kDenseSmallN) {
            sv.launch_shm("small_solve", k_dense_small, 1, kSmallThreads, small_system_doubles(n) * sizeof(double),
                          (const double*)S.p, ld, (const double*)d.bc, d.px, n, d.st);
        } else if (f64) {
            factor_and_solve<double>(sv, S.p, Dinvd.p, Binvd.p, BinvTd.p);
        } else {
            const int m = nt / 2;  // 64 x 64 blocks a side
            sv.launch("convert_S", k_convert_S, m * (m + 1) / 2, kWG, (const double*)S.p, Af.p, ld, (const LMState*)d.st);
            factor_and_solve<float>(sv, Af.p, Dinvf.p, Binvf.p, BinvTf.p);
        }
    }
};

}  // namespace mba
