// pair_block.h -- one 9x9 block of a reduced camera system from its observation pairs, by one wave.
//
// S_ab = [a == b] D_a^2 - sum_pairs J~_c,i' G_ij J~_c,j over the pairs (i, j) of observations of
// one point in cameras a and b, with G_ij = H_i J~_p,j' (H = J~_p V*^-1) for i != j and, for an
// observation with itself, -(I - G)_i (its share of U* folded in).  Used by the batched windows
// (records of 32 values, I - G formed from H and J~_p in working precision) and by the dense
// single-problem solver (records of 36 values with I - G formed in FP64 and stored).
//
// Per stage of 32 pairs the wave copies the record chunks the products read into its LDS staging area
// with 4-element vector loads, sixteen lanes to a pair (the next stage's records and the pair indices
// two stages ahead are in flight, requested in that order so that neither wait covers the other); then
// lane q of each half-wave takes pair q, the lower half columns 0-3 of all nine rows, the upper half
// columns 4-8, accumulating in registers (FP64); the partial sums of an entry are folded over the
// half-wave's lanes.  The block's entries are written to S (row-major, leading dimension ld, both
// triangles).  Every entry's sum runs in a fixed order (pair q, q + 32, ... per lane, then the fold),
// whatever wave or launch takes the block.  The dense solver, whose blocks are few and long, gives a
// block to a workgroup of several waves instead (NW below).
//
// LDS accesses bound it (60% of the time of a launch with sixteen pairs a stage, four column groups and
// 23 LDS instructions a stage, at 250 cameras and 4.2M pairs): with two column groups a pair's i record
// is read twice instead of four times, and in 16-byte units.
#pragma once

#include "lm_kernels.h"

namespace mba {

constexpr int kPairsPerStage = 32;

// Two consecutive record elements, read as one LDS access.
template <typename Real>
struct alignas(2 * sizeof(Real)) R2v {
    Real x, y;
};

// Record layouts.  Both keep J~_c by columns (the two residual rows of column c at 2c, 2c + 1).
//   kRecWindow: [J~_c 18][H 6][J~_p 6][2 unused]; i records read chunks 0-5, j records 0-4 and 6-7.
//   kRecDense:  [J~_c 18][J~_p 6][H 6][I - G: g00 g01 g11][3 unused]; i records read chunks 0-4 and
//               6-8 (J~_c, H, I - G), j records 0-5 (J~_c, J~_p).
// A pair's cp chunks (four values) are slots 0 .. cp - 1 of the staging area, the i record's ci first; h0 and
// jp0 are the half slots (two values) H and J~_p start at.
enum { kRecWindow = 0, kRecDense = 1 };
template <int LAYOUT>
struct RecLayout;
template <>
struct RecLayout<kRecWindow> {
    static constexpr int stride = 32, ci = 6, cp = 13, h0 = 9, jp0 = 22;
    static constexpr bool stored_complement = false;
    // chunk of the record in slot e
    __device__ static int chunk(int e) { return e < ci ? e : (e - ci < 5 ? e - ci : e - ci + 1); }
};
template <>
struct RecLayout<kRecDense> {
    static constexpr int stride = 36, ci = 8, cp = 14, h0 = 10, jp0 = 25;
    static constexpr bool stored_complement = true;
    __device__ static int chunk(int e) { return e < ci ? (e < 5 ? e : e + 1) : e - ci; }
};

// A wave's records on their way to memory go through LDS, so that neighbouring lanes write neighbouring
// 16-byte units: stored by the lanes that form them, each store instruction touches 64 records' lines, a
// part of a line at a time.  stage_pair puts two values of the lane's record, at pair `at` of its row of
// kRecordRow units; flush_records stores `step` units of every row, units u0 .. of the first n records at out.
typedef unsigned int Unit16 __attribute__((ext_vector_type(4)));
constexpr int kRecordRow = 9;  // odd: neighbouring rows start in different banks
template <typename Real>
__device__ __forceinline__ void stage_pair(Unit16* lds, int at, Real x, Real y) {
    reinterpret_cast<R2v<Real>*>(lds + kRecordRow * (threadIdx.x & 63))[at] = R2v<Real>{x, y};
}
template <int units, int step, typename Real>
__device__ __forceinline__ void flush_records(const Unit16* lds, Real* __restrict__ out, int u0, int n) {
    static_assert(step <= kRecordRow && step <= units, "a row's units");
    const int lane = threadIdx.x & 63;
    wave_sync_lds();
#pragma unroll 4
    for (int s = 0; s < step; ++s) {
        const int e = 64 * s + lane, rec = e / step, u = e - step * rec;
        if (rec < n) reinterpret_cast<Unit16*>(out)[(size_t)units * rec + u0 + u] = lds[kRecordRow * rec + u];
    }
    wave_sync_lds();
}

// The staging area holds 16-byte units (a slot in FP32, half a slot in FP64), unit u of pair k at
// u (32 + 1) + k: neighbouring pairs' units are adjacent for the reads, and a pair's units, which
// neighbouring lanes store, lie in different banks.  FP64 keeps the slots' second halves after all first ones.
constexpr int kUnitPitch = kPairsPerStage + 1;
template <typename Real>
constexpr int kUnitsPerSlot = 4 * (int)sizeof(Real) / 16;

// LDS bytes of a wave's staging area.
template <typename Real, int LAYOUT>
constexpr int pair_stage_bytes() {
    return kUnitsPerSlot<Real> * RecLayout<LAYOUT>::cp * kUnitPitch * 16;
}

// Values 2 half, 2 half + 1 of slot e of pair k.
template <typename Real, int LAYOUT>
__device__ __forceinline__ R2v<Real> stage_half(const Real* stage, int e, int half, int k) {
    constexpr int cp = RecLayout<LAYOUT>::cp;
    if constexpr (kUnitsPerSlot<Real> == 1)
        return *reinterpret_cast<const R2v<Real>*>(stage + 4 * (e * kUnitPitch + k) + 2 * half);
    else
        return *reinterpret_cast<const R2v<Real>*>(stage + 2 * ((half * cp + e) * kUnitPitch + k));
}

// All four values of slot e of pair k.
template <typename Real, int LAYOUT>
__device__ __forceinline__ void stage_slot(const Real* stage, int e, int k, R2v<Real>& lo, R2v<Real>& hi) {
    if constexpr (kUnitsPerSlot<Real> == 1) {
        const R4<Real> v = *reinterpret_cast<const R4<Real>*>(stage + 4 * (e * kUnitPitch + k));
        lo = R2v<Real>{v.x, v.y};
        hi = R2v<Real>{v.z, v.w};
    } else {
        lo = stage_half<Real, LAYOUT>(stage, e, 0, k);
        hi = stage_half<Real, LAYOUT>(stage, e, 1, k);
    }
}

// Six values from half slot s0 on.
template <typename Real, int LAYOUT, int s0>
__device__ __forceinline__ void stage_six(const Real* stage, int k, R2v<Real> (&v)[3]) {
    if constexpr (s0 & 1) {
        v[0] = stage_half<Real, LAYOUT>(stage, s0 / 2, 1, k);
        stage_slot<Real, LAYOUT>(stage, s0 / 2 + 1, k, v[1], v[2]);
    } else {
        stage_slot<Real, LAYOUT>(stage, s0 / 2, k, v[0], v[1]);
        v[2] = stage_half<Real, LAYOUT>(stage, s0 / 2 + 1, 0, k);
    }
}

// Copy round r of a stage: lane l takes slot l % 16 (the last one for the spare lanes) of pair
// 4 r + l / 16.  idx holds the stage's observation indices, i of pair k in lane k and j in lane 32 + k.
constexpr int kCopyRounds = kPairsPerStage / 4;
template <typename Real, int LAYOUT>
__device__ __forceinline__ R4<Real> pair_load_round(const Real* __restrict__ js, int idx, int r) {
    using RL = RecLayout<LAYOUT>;
    const int lane = threadIdx.x & 63, e = min(lane & 15, RL::cp - 1);
    const int o = __shfl(idx, 4 * r + (lane >> 4) + (e < RL::ci ? 0 : 32), 64);
    return reinterpret_cast<const R4<Real>*>(js + RL::stride * (size_t)o)[RL::chunk(e)];
}

template <typename Real, int LAYOUT>
__device__ __forceinline__ void pair_store_round(Real* stage, int r, const R4<Real>& v) {
    using RL = RecLayout<LAYOUT>;
    const int lane = threadIdx.x & 63, e = min(lane & 15, RL::cp - 1), k = 4 * r + (lane >> 4);
    if constexpr (kUnitsPerSlot<Real> == 1) {
        *reinterpret_cast<R4<Real>*>(stage + 4 * (e * kUnitPitch + k)) = v;
    } else {
        *reinterpret_cast<R2v<Real>*>(stage + 2 * (e * kUnitPitch + k)) = R2v<Real>{v.x, v.y};
        *reinterpret_cast<R2v<Real>*>(stage + 2 * ((RL::cp + e) * kUnitPitch + k)) = R2v<Real>{v.z, v.w};
    }
}

// One entry (r, c) of block bk, the pairs' sum v, into S.
__device__ __forceinline__ void pair_entry(const int4 bk, int r, int c, double v, const double* __restrict__ dc2, double* S,
                                           int ld) {
    const int ca = bk.x, cb = bk.y;
    const double s = (ca == cb && r == c ? dc2[9 * ca + r] : 0.0) - v;
    S[(size_t)(9 * ca + r) * ld + 9 * cb + c] = s;
    if (ca != cb) S[(size_t)(9 * cb + c) * ld + 9 * ca + r] = s;
}

// Block bk = (camera a, camera b, first pair, end pair) of the pair list `pairs` (observation
// indices (i, j) into the records js) into S; dc2 holds D^2 (added on the diagonal of a == b).
// NW > 1: the workgroup's NW waves take the block's stages in turn (wave w the stages w, w + NW, ...; each
// with its own staging area) and their sums are added in neighbouring pairs through sums (NW x 81 doubles
// of LDS); every wave of the workgroup must call it.
template <typename Real, int LAYOUT, int NW = 1>
__device__ __forceinline__ void pair_block(const int4 bk_all, const int2* __restrict__ pairs, const Real* __restrict__ js,
                                           const double* __restrict__ dc2, double* S, int ld, Real* stage,
                                           double* sums = nullptr) {
    using RL = RecLayout<LAYOUT>;
    using R2 = R2v<Real>;
    constexpr int PS = kPairsPerStage;
    static_assert(PS == 32 && RL::cp <= 16, "one pair per lane of a half-wave, one slot per lane of a row");
    const int wave = NW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    int4 bk = bk_all;
    bk.z = min(bk.z + PS * wave, bk.w);
    constexpr int kStride = NW * PS;  // pairs between two stages of a wave
    const int lane = threadIdx.x & 63, q = lane & 31, h = lane >> 5;
    const int c0 = 4 * h, nc = 4 + h;  // the lane's columns (a fifth slot of the lower half repeats column 4)
    const bool self = bk.x == bk.y;    // only there can an observation be paired with itself
    double acc[9][5];
#pragma unroll
    for (int r = 0; r < 9; ++r)
#pragma unroll
        for (int k = 0; k < 5; ++k) acc[r][k] = 0.0;
    const int npairs = bk.w - bk.z;  // up to the block's end, the other waves' stages among them
    const int nst = (npairs + kStride - 1) / kStride;
    // lane's index of a stage starting at pair b; lanes past the block's pairs repeat its last one, whose
    // products are not used
    auto load_idx = [&](int b) { return reinterpret_cast<const int*>(pairs)[2 * (size_t)min(b + q, bk.w - 1) + h]; };
    int idx = 0, idx_next = 0;
    R4<Real> rec[kCopyRounds];
    if (nst > 0) {
        idx = load_idx(bk.z);
        if (nst > 1) idx_next = load_idx(bk.z + kStride);
#pragma unroll
        for (int r = 0; r < kCopyRounds; ++r) rec[r] = pair_load_round<Real, LAYOUT>(js, idx, r);
    }
    for (int stg = 0; stg < nst; ++stg) {
        const int base = bk.z + stg * kStride;
        const int m = min(PS, bk.w - base);
#pragma unroll
        for (int r = 0; r < kCopyRounds; ++r) pair_store_round<Real, LAYOUT>(stage, r, rec[r]);
        bool same = false;
        if (self) same = __shfl(idx, q, 64) == __shfl(idx, 32 + q, 64);
        // the pair indices two stages ahead are requested before the next stage's records and
        // taken over after this stage's products, so that neither waits for the records (a wave's
        // loads complete in order)
        int idx_far = 0;
        if (stg + 1 < nst) {
            if (stg + 2 < nst) idx_far = load_idx(base + 2 * kStride);
#pragma unroll
            for (int r = 0; r < kCopyRounds; ++r) rec[r] = pair_load_round<Real, LAYOUT>(js, idx_next, r);
        }
        wave_sync_lds();
        if (q < m) {
            R2 hh[3], p[3];
            stage_six<Real, LAYOUT, RL::h0>(stage, q, hh);
            stage_six<Real, LAYOUT, RL::jp0>(stage, q, p);
            // H_i = [h0.x h0.y h1.x; h1.y h2.x h2.y], J~_p,j = [p0.x p0.y p1.x; p1.y p2.x p2.y]
            double G00 = (double)(hh[0].x * p[0].x + hh[0].y * p[0].y + hh[1].x * p[1].x);
            double G01 = (double)(hh[0].x * p[1].y + hh[0].y * p[2].x + hh[1].x * p[2].y);
            double G10 = (double)(hh[1].y * p[0].x + hh[2].x * p[0].y + hh[2].y * p[1].x);
            double G11 = (double)(hh[1].y * p[1].y + hh[2].x * p[2].x + hh[2].y * p[2].y);
            if (same) {
                if (RL::stored_complement) {
                    // an observation with itself: -(I - G) as formed in FP64 when the record was written
                    const R2 g0 = stage_half<Real, LAYOUT>(stage, 6, 1, q), g1 = stage_half<Real, LAYOUT>(stage, 7, 0, q);
                    G00 = -(double)g0.x;
                    G01 = G10 = -(double)g0.y;
                    G11 = -(double)g1.x;
                } else {
                    // an observation with itself carries its share of U*: J~c'(I - G)J~c, negated
                    // because the accumulated sum is subtracted
                    G00 -= 1.0;
                    G11 -= 1.0;
                }
            }
            R2 jc[5];
            stage_slot<Real, LAYOUT>(stage, RL::ci + 2 * h, q, jc[0], jc[1]);
            stage_slot<Real, LAYOUT>(stage, RL::ci + 2 * h + 1, q, jc[2], jc[3]);
            jc[4] = stage_half<Real, LAYOUT>(stage, RL::ci + 2 * h + 2, 0, q);
            double t0[5], t1[5];
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                t0[k] = G00 * (double)jc[k].x + G01 * (double)jc[k].y;
                t1[k] = G10 * (double)jc[k].x + G11 * (double)jc[k].y;
            }
#pragma unroll
            for (int r2 = 0; r2 < 5; ++r2) {
                R2 a[2];
                if (r2 < 4)
                    stage_slot<Real, LAYOUT>(stage, r2, q, a[0], a[1]);
                else
                    a[0] = stage_half<Real, LAYOUT>(stage, 4, 0, q);
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    if (2 * r2 + u < 9)
#pragma unroll
                        for (int k = 0; k < 5; ++k)
                            acc[2 * r2 + u][k] = fma((double)a[u].y, t1[k], fma((double)a[u].x, t0[k], acc[2 * r2 + u][k]));
            }
        }
        wave_sync_lds();
        idx = idx_next;
        idx_next = idx_far;
    }
    // the 45 sums over each half-wave: lane q gets numbers q and q + 32
    double sum[45];
#pragma unroll
    for (int e = 0; e < 45; ++e) sum[e] = acc[e / 5][e % 5];
    lane_fold<45, 5>(sum);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int e = q + 32 * u, r = e / 5, k = e - 5 * r, c = c0 + k;
        if (e < 45 && k < nc) {
            if (NW == 1)
                pair_entry(bk, r, c, sum[u], dc2, S, ld);
            else
                sums[81 * wave + 9 * r + c] = sum[u];
        }
    }
    if (NW > 1) {
        lds_barrier();
        for (int e = threadIdx.x; e < 81; e += 64 * NW) {
            double v[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w) v[w] = sums[81 * w + e];
#pragma unroll
            for (int h = 1; h < NW; h *= 2)
#pragma unroll
                for (int w = 0; w + h < NW; w += 2 * h) v[w] += v[w + h];
            pair_entry(bk, e / 9, e % 9, v[0], dc2, S, ld);
        }
    }
}

}  // namespace mba
