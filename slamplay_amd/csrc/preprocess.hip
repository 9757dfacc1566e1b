// preprocess.hip -- BALProblem::Normalize and ::Perturb on the parameters a solver holds on the
// device (utils/datasets/BALProblem.cpp:39-76,230-336).
//
// Built with -ffp-contract=off so every product and sum rounds as the host code's does; with that,
// the medians, the L1 distances, the scale and the point transform are bit-identical to the host
// Normalize, and the perturbation draws the same normals as the host Perturb (equal to the last ulp
// of log()).
#include <cmath>
#include <mutex>
#include <vector>

#include "preprocess.h"

namespace mba {
namespace {

// ---------------------------------------------------------------------------------------------
// glibc rand() (random_r.c, TYPE_3: degree 31, separation 3).  srand(seed) sets r_0 = seed (1 for
// 0) and r_i = 16807 r_{i-1} mod (2^31 - 1) for i < 31 by Schrage's method in 32-bit arithmetic,
// then r_31..r_33 = r_0..r_2 and r_i = r_{i-31} + r_{i-3} (mod 2^32) onwards; srand discards 310
// outputs, so rand() call k returns r_{344+k} >> 1.  The state (r_{i-31}, ..., r_{i-1}) evolves by
// a fixed 31x31 matrix over Z/2^32, which is what makes jump-ahead possible.
constexpr int kDeg = 31;
constexpr int kChunk = 31 * 8;   // draws per generator thread
constexpr int kJumps = 24;       // generator threads below 2^24
constexpr int kPairsPerThread = 4;
constexpr int kPairBlock = 256;
constexpr int kPairsPerBlock = kPairsPerThread * kPairBlock;
constexpr int kSelBlock = 256;

struct RandState {
    uint32_t s[kDeg];
};

// state before rand() call 0: (r_313, ..., r_343)
RandState glibc_seed_state(uint32_t seed) {
    std::vector<uint32_t> r(344);
    if (seed == 0) seed = 1;
    int32_t word = (int32_t)seed;
    r[0] = (uint32_t)word;
    for (int i = 1; i < kDeg; ++i) {
        const int64_t hi = word / 127773, lo = word % 127773;
        int64_t next = 16807 * lo - 2836 * hi;
        if (next < 0) next += 2147483647;
        word = (int32_t)next;
        r[i] = (uint32_t)word;
    }
    for (int i = kDeg; i < 34; ++i) r[i] = r[i - kDeg];
    for (int i = 34; i < 344; ++i) r[i] = r[i - 31] + r[i - 3];
    RandState st;
    for (int j = 0; j < kDeg; ++j) st.s[j] = r[313 + j];
    return st;
}

using Mat31 = std::vector<uint32_t>;  // row-major 31x31

Mat31 mat_mul(const Mat31& a, const Mat31& b) {
    Mat31 c(kDeg * kDeg, 0u);
    for (int i = 0; i < kDeg; ++i)
        for (int k = 0; k < kDeg; ++k) {
            const uint32_t aik = a[i * kDeg + k];
            if (!aik) continue;
            for (int j = 0; j < kDeg; ++j) c[i * kDeg + j] += aik * b[k * kDeg + j];
        }
    return c;
}

// Q_j = A^(kChunk 2^j) for j < kJumps, A the one-draw transition.
const std::vector<uint32_t>& jump_tables() {
    static std::vector<uint32_t> tables;
    static std::once_flag once;
    std::call_once(once, [] {
        Mat31 a(kDeg * kDeg, 0u), p(kDeg * kDeg, 0u);
        for (int j = 0; j + 1 < kDeg; ++j) a[j * kDeg + j + 1] = 1u;  // shift
        a[(kDeg - 1) * kDeg + 0] = 1u;                                // r_{i-31}
        a[(kDeg - 1) * kDeg + 28] = 1u;                               // r_{i-3}
        for (int j = 0; j < kDeg; ++j) p[j * kDeg + j] = 1u;
        Mat31 base = a;
        for (int e = kChunk; e; e >>= 1) {  // p = A^kChunk
            if (e & 1) p = mat_mul(p, base);
            base = mat_mul(base, base);
        }
        tables.reserve((size_t)kJumps * kDeg * kDeg);
        for (int j = 0; j < kJumps; ++j) {
            tables.insert(tables.end(), p.begin(), p.end());
            p = mat_mul(p, p);
        }
    });
    return tables;
}

// A workgroup gives the draws of 64 consecutive chunks.  The first one's start state by the jumps of the
// workgroup index's bits, in wave 0, one row of the 31 x 31 product per lane, while the other waves put
// Q_0..Q_5 into LDS; the others by doubling, chunks n .. 2n - 1 from 0 .. n - 1 with Q_log2(n), the 31 n rows
// spread over the threads.  Then one lane per chunk runs the recurrence 31 draws at a time with the state
// in registers (s[j] += s[j+28] for the first three, whose r_{i-3} is still the previous round's,
// s[j] += s[j-3] for the rest) into LDS, from where the workgroup stores its 15,872 words contiguously.
// Bound by latency, not by what it writes: 818,000 draws (3.3 MB) take 15 us (132 with a whole product
// per bit of the chunk index in every thread, 57 with one wave to a workgroup for all of this).
constexpr int kBlockChunks = 64;
constexpr int kBlockBits = 6;  // log2(kBlockChunks)
constexpr int kChunkRow = kChunk + 1;  // odd row stride: the lanes' rows start in distinct banks
constexpr int kStateRow = kDeg + 2;
__global__ void __launch_bounds__(256) k_rand_generate(RandState start, const uint32_t* __restrict__ tables,
                                                       int64_t n_draws, uint32_t* __restrict__ out) {
    __shared__ uint32_t lds[kBlockChunks * kChunkRow];  // first the states and Q_0..Q_5, then the draws
    static_assert(kBlockChunks * kStateRow + kBlockBits * kDeg * kDeg <= kBlockChunks * kChunkRow, "LDS of the start states");
    uint32_t* const state = lds;
    uint32_t* const Qs = lds + kBlockChunks * kStateRow;
    const int t = threadIdx.x;
    if (t >= 64) {
        constexpr int n = kBlockBits * kDeg * kDeg, per = (n + 191) / 192;
        uint32_t v[per];
#pragma unroll
        for (int i = 0; i < per; ++i) v[i] = tables[min(t - 64 + 192 * i, n - 1)];
#pragma unroll
        for (int i = 0; i < per; ++i)
            if (t - 64 + 192 * i < n) Qs[t - 64 + 192 * i] = v[i];
    } else {
        uint32_t mine = 0;  // entry t of the state
#pragma unroll
        for (int j = 0; j < kDeg; ++j) mine = t == j ? start.s[j] : mine;
        for (int q = kBlockBits; q < kJumps && ((int)blockIdx.x >> (q - kBlockBits)); ++q) {
            if (!(((int)blockIdx.x >> (q - kBlockBits)) & 1)) continue;
            const uint32_t* Q = tables + (size_t)q * kDeg * kDeg + (t < kDeg ? t : 0) * kDeg;
            uint32_t row[kDeg], acc = 0;
#pragma unroll
            for (int k = 0; k < kDeg; ++k) row[k] = Q[k];
#pragma unroll
            for (int k = 0; k < kDeg; ++k) acc += row[k] * (uint32_t)__builtin_amdgcn_readlane((int)mine, k);
            mine = acc;
        }
        if (t < kDeg) state[t] = mine;
    }
    __syncthreads();
    for (int q = 0; q < kBlockBits; ++q) {
        const int n = 1 << q;
        for (int e = t; e < kDeg * n; e += 256) {
            const int m = e / kDeg, i = e - kDeg * m;
            uint32_t acc = 0;
#pragma unroll
            for (int k = 0; k < kDeg; ++k) acc += Qs[q * kDeg * kDeg + i * kDeg + k] * state[m * kStateRow + k];
            state[(m + n) * kStateRow + i] = acc;
        }
        __syncthreads();
    }
    uint32_t s[kDeg];
#pragma unroll
    for (int j = 0; j < kDeg; ++j) s[j] = state[(t & 63) * kStateRow + j];
    __syncthreads();
    if (t < 64)
        for (int round = 0; round < kChunk / kDeg; ++round) {
#pragma unroll
            for (int j = 0; j < 3; ++j) s[j] += s[j + 28];
#pragma unroll
            for (int j = 3; j < kDeg; ++j) s[j] += s[j - 3];
#pragma unroll
            for (int j = 0; j < kDeg; ++j) lds[t * kChunkRow + round * kDeg + j] = s[j] >> 1;
        }
    __syncthreads();
    const int64_t first = (int64_t)blockIdx.x * (kBlockChunks * kChunk);
    const int n = (int)std::min<int64_t>(n_draws - first, kBlockChunks * kChunk);
    for (int e = t; e < n; e += 256) {
        const int c = e / kChunk;
        out[first + e] = lds[c * kChunkRow + e - c * kChunk];
    }
}

// BALProblem.cpp:39-55: x = 2 rand()/RAND_MAX - 1 for both coordinates, rejected when w >= 1 or 0.
__device__ __forceinline__ bool polar_pair(const uint32_t* __restrict__ draws, int64_t j, double* x1, double* w) {
    const double a = 2.0 * ((double)draws[2 * j] / 2147483647.0) - 1.0;
    const double c = 2.0 * ((double)draws[2 * j + 1] / 2147483647.0) - 1.0;
    const double ww = a * a + c * c;
    *x1 = a;
    *w = ww;
    return !(ww >= 1.0 || ww == 0.0);
}

// exclusive prefix sum over a 256-thread block; returns the block total in *total
__device__ __forceinline__ int block_exclusive_scan(int v, int* lds, int* total) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) lds[wave] = x;
    __syncthreads();
    int wave_off = 0, all = 0;
    for (int k = 0; k < kPairBlock / 64; ++k) {
        const int c = lds[k];
        if (k < wave) wave_off += c;
        all += c;
    }
    __syncthreads();
    *total = all;
    return wave_off + x - v;
}

__global__ void __launch_bounds__(kPairBlock) k_pairs_count(const uint32_t* __restrict__ draws, int64_t n_pairs,
                                                            int* __restrict__ counts) {
    __shared__ int lds[kPairBlock / 64];
    const int64_t p0 = (int64_t)blockIdx.x * kPairsPerBlock + (int64_t)threadIdx.x * kPairsPerThread;
    int c = 0;
    for (int k = 0; k < kPairsPerThread; ++k) {
        double x1, w;
        if (p0 + k < n_pairs && polar_pair(draws, p0 + k, &x1, &w)) ++c;
    }
    int total;
    block_exclusive_scan(c, lds, &total);
    if (threadIdx.x == 0) counts[blockIdx.x] = total;
}

// one block: counts -> exclusive offsets; total accepted pairs into *total
__global__ void __launch_bounds__(kPairBlock) k_pairs_scan(int* __restrict__ counts, int n, int* __restrict__ total) {
    __shared__ int lds[kPairBlock / 64];
    int carry = 0;
    for (int base = 0; base < n; base += kPairBlock) {
        const int i = base + (int)threadIdx.x;
        const int v = i < n ? counts[i] : 0;
        int tile;
        const int ex = block_exclusive_scan(v, lds, &tile);
        if (i < n) counts[i] = carry + ex;
        carry += tile;
    }
    if (threadIdx.x == 0) *total = carry;
}

__global__ void __launch_bounds__(kPairBlock) k_pairs_emit(const uint32_t* __restrict__ draws, int64_t n_pairs,
                                                           const int* __restrict__ offsets, int n_normals,
                                                           double* __restrict__ normals) {
    __shared__ int lds[kPairBlock / 64];
    const int64_t p0 = (int64_t)blockIdx.x * kPairsPerBlock + (int64_t)threadIdx.x * kPairsPerThread;
    double x1[kPairsPerThread], w[kPairsPerThread];
    bool ok[kPairsPerThread];
    int c = 0;
#pragma unroll
    for (int k = 0; k < kPairsPerThread; ++k) {
        ok[k] = p0 + k < n_pairs && polar_pair(draws, p0 + k, &x1[k], &w[k]);
        c += ok[k] ? 1 : 0;
    }
    int total;
    int idx = offsets[blockIdx.x] + block_exclusive_scan(c, lds, &total);
#pragma unroll
    for (int k = 0; k < kPairsPerThread; ++k)
        if (ok[k]) {
            if (idx < n_normals) normals[idx] = x1[k] * sqrt((-2.0 * log(w[k])) / w[k]);
            ++idx;
        }
}

// rotation.h:133-198 (AngleAxisRotatePoint), in the expression order of the host BALProblem code
__device__ __forceinline__ void rotate_point(const double aa[3], const double pt[3], double out[3]) {
    const double theta2 = aa[0] * aa[0] + aa[1] * aa[1] + aa[2] * aa[2];
    if (theta2 > 2.220446049250313080847e-16) {
        const double theta = sqrt(theta2);
        const double c = cos(theta), s = sin(theta);
        const double inv = 1.0 / theta;
        const double w[3] = {aa[0] * inv, aa[1] * inv, aa[2] * inv};
        const double wx[3] = {w[1] * pt[2] - w[2] * pt[1], w[2] * pt[0] - w[0] * pt[2], w[0] * pt[1] - w[1] * pt[0]};
        const double tmp = (w[0] * pt[0] + w[1] * pt[1] + w[2] * pt[2]) * (1.0 - c);
        for (int i = 0; i < 3; ++i) out[i] = pt[i] * c + wx[i] * s + w[i] * tmp;
    } else {
        const double wx[3] = {aa[1] * pt[2] - aa[2] * pt[1], aa[2] * pt[0] - aa[0] * pt[2], aa[0] * pt[1] - aa[1] * pt[0]};
        for (int i = 0; i < 3; ++i) out[i] = pt[i] + wx[i];
    }
}

// BALProblem.cpp:230-246: c = -R' t, through R(-aa)
__device__ __forceinline__ void camera_center(const double aa[3], const double t[3], double center[3]) {
    const double inv[3] = {-aa[0], -aa[1], -aa[2]};
    rotate_point(inv, t, center);
    for (int i = 0; i < 3; ++i) center[i] *= -1.0;
}

// BALProblem.cpp:248-261: t = -R c
__device__ __forceinline__ void center_translation(const double aa[3], const double center[3], double t[3]) {
    rotate_point(aa, center, t);
    for (int i = 0; i < 3; ++i) t[i] *= -1.0;
}

// BALProblem.cpp:305-336, points: X += n * sigma with the normals of the caller's point order
// (both kernels leave the parameters alone when the stream gave too few normals: the host then draws a
// longer one, and otherwise never waits between the draws and their use)
__global__ void k_perturb_points(double* __restrict__ pt, const int* __restrict__ pt_orig, int np,
                                 const double* __restrict__ normals, double sigma, const int* __restrict__ got, int need) {
    const int ip = blockIdx.x * blockDim.x + threadIdx.x;
    if (ip >= np || *got < need) return;
    const int64_t o = 3 * (int64_t)pt_orig[ip];
    for (int j = 0; j < 3; ++j) pt[4 * (int64_t)ip + j] += normals[o + j] * sigma;
}

// cameras: angle-axis += n * rs with the centre held, t recomputed, then t += n * ts
__global__ void k_perturb_cams(double* __restrict__ cam, int nc, const double* __restrict__ normals, int64_t first,
                               double rs, double ts, const int* __restrict__ got, int need) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc || (need > 0 && *got < need)) return;
    const int per = (rs > 0.0 ? 3 : 0) + (ts > 0.0 ? 3 : 0);
    int64_t k = first + (int64_t)per * c;
    double aa[3], t[3], center[3];
    for (int i = 0; i < 3; ++i) {
        aa[i] = cam[(size_t)i * nc + c];
        t[i] = cam[(size_t)(3 + i) * nc + c];
    }
    camera_center(aa, t, center);
    if (rs > 0.0) {
        for (int i = 0; i < 3; ++i) aa[i] += normals[k + i] * rs;
        k += 3;
    }
    center_translation(aa, center, t);
    if (ts > 0.0)
        for (int i = 0; i < 3; ++i) t[i] += normals[k + i] * ts;
    for (int i = 0; i < 3; ++i) {
        cam[(size_t)i * nc + c] = aa[i];
        cam[(size_t)(3 + i) * nc + c] = t[i];
    }
}

// ---------------------------------------------------------------------------------------------
// Upper median (nth_element at n/2, BALProblem.cpp:71-76) by radix selection over the IEEE bit
// patterns mapped to order-preserving keys, from the top.  Selection k: 0..2 a point axis, 3 the L1
// distances.  Histograms of 11 bits over all keys (every block picks the digit found last from the previous
// counts itself, so a pass is one launch), then the keys that share the digits so far are collected and one
// block finishes on them.  Two histograms leave a thousandth of the range around the median, a few hundred of
// 100,000 points in general position; bound by launches, 5 us each, both selections take 60 us with the wait
// for them (eight passes of eight bits, with a launch each to pick the digit: 113).  But a map may lie in a
// plane or far from the origin: most keys share 22 bits then, and the one block has them all.  At 100,000 points it
// takes 65 us so for a plane and 122 for a map a thousand extents away; what it takes grows with the points,
// so beyond kSelSpread four more histograms, which return at once when at most kSelCap keys are left, take the
// digits down to the last over the whole chip: a million points in a plane 152 us, in general position 118
// (eight passes 190 and 173; with all keys left to a block of 256 threads 4,900, and 446 for the plane of 100,000).
constexpr int kSelBits = 11;
constexpr int kSelBins = 1 << kSelBits;
constexpr int kSelPasses = 6;            // digits of a key: five of kSelBits, one of the last nine bits
constexpr int kSelSpread = 1 << 17;
constexpr unsigned int kSelCap = 1 << 14;
constexpr int kFinishBlock = 1024;
constexpr int kFinishList = 4096;        // keys the last block keeps in LDS

// A selection with its first `bits` bits found: they are the prefix's, `count` keys share them and the one looked
// for has rank `rank` among these.
struct SelState {
    unsigned long long prefix, rank;
    unsigned int count, bits;
};

__device__ __forceinline__ unsigned long long order_key(double x) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(x);
    return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}

__device__ __forceinline__ double key_value(unsigned long long k) {
    const unsigned long long u = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __longlong_as_double((long long)u);
}

// hist: [pass][selection][kSelBins], n words in all; count: collected keys per selection, range: the smallest and
// the largest of them
__global__ void __launch_bounds__(256) k_sel_init(unsigned int* __restrict__ hist, int n, unsigned int* __restrict__ count,
                                                  unsigned long long* __restrict__ range) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) hist[i] = 0;
    if (i < 4) count[i] = 0;
    if (i < 8) range[i] = i & 1 ? 0 : ~0ull;
}

// The bin of counts h (kSelBins of them) that holds rank *rank, by a block of NT threads: its number is returned
// in every thread, *rank becomes the rank inside it and *count its count.
template <int NT>
__device__ __forceinline__ unsigned int sel_pick(const unsigned int* __restrict__ h, unsigned long long* rank, unsigned int* count) {
    constexpr int per = kSelBins / NT, waves = NT / 64;
    __shared__ unsigned long long wsum[waves], rank_in;
    __shared__ unsigned int digit, count_in;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    unsigned int v[per];
    unsigned long long x = 0;
#pragma unroll
    for (int i = 0; i < per; ++i) {
        v[i] = h[per * t + i];
        x += v[i];
    }
    const unsigned long long own = x;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    __syncthreads();  // the shared words of an earlier pick have been read
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    unsigned long long excl = x - own;
    for (int w = 0; w < wave; ++w) excl += wsum[w];
    if (excl <= *rank && *rank < excl + own) {
        unsigned long long left = *rank - excl;
        int i = 0;
        while (i + 1 < per && left >= v[i]) left -= v[i++];
        digit = per * t + i;
        count_in = v[i];
        rank_in = left;
    }
    __syncthreads();
    *rank = rank_in;
    *count = count_in;
    return digit;
}

// Few enough keys are left for one block (the first two digits are always taken by the whole chip).
__device__ __forceinline__ bool sel_small(const SelState& s) { return s.bits >= 2 * kSelBits && s.count <= kSelCap; }

// Selection k as pass `pass` finds it: the state its predecessor left, with the digit that one counted.
// Block 0 leaves it for the next pass.
__device__ __forceinline__ SelState sel_state(SelState* __restrict__ states, const unsigned int* __restrict__ hist, int k, int pass,
                                              int np, bool first_block) {
    SelState s{0, (unsigned long long)(np / 2), (unsigned int)np, 0};
    if (pass > 1) s = states[(kSelPasses + 1) * k + pass - 1];
    if (pass > 0 && !sel_small(s)) {
        const unsigned int digit = sel_pick<kSelBlock>(hist + (size_t)(4 * (pass - 1) + k) * kSelBins, &s.rank, &s.count);
        s.bits = min(64u, s.bits + kSelBits);
        s.prefix |= (unsigned long long)digit << (64 - s.bits);
    }
    if (pass > 0 && first_block && threadIdx.x == 0) states[(kSelPasses + 1) * k + pass] = s;
    return s;
}

// BALProblem.cpp:274-281: L1 distance of a point to the per-axis medians
__device__ __forceinline__ double norm_dist(const double* __restrict__ p, const double m[3]) {
    return fabs(p[0] - m[0]) + fabs(p[1] - m[1]) + fabs(p[2] - m[2]);
}

// The key of point i in selection k: its coordinate on axis k, or its distance to the medians m.
__device__ __forceinline__ unsigned long long sel_key(const double* __restrict__ pt, int i, int k, const double m[3]) {
    const double* p = pt + 4 * (int64_t)i;
    return order_key(k < 3 ? p[k] : norm_dist(p, m));
}

// A round of kSelRound keys of a block: thread t has those of points i0 + t, i0 + kSelBlock + t, ... below np, all
// loads in flight together (past the last point its key again).
constexpr int kSelUnroll = 8;
constexpr int kSelRound = kSelUnroll * kSelBlock;
__device__ __forceinline__ void sel_round(const double* __restrict__ pt, int64_t i0, int np, int k, const double m[3],
                                          unsigned long long (&key)[kSelUnroll]) {
#pragma unroll
    for (int u = 0; u < kSelUnroll; ++u)
        key[u] = sel_key(pt, (int)min(i0 + u * kSelBlock + (int)threadIdx.x, (int64_t)np - 1), k, m);
}

// Counts of digit `pass` of selections first .. first + gridDim.y - 1.  Selection 3 forms the distances from
// the points and the medians, the found keys 0..2.
__global__ void __launch_bounds__(kSelBlock) k_sel_hist(const double* __restrict__ pt, int np, int first, int pass,
                                                        const unsigned long long* __restrict__ found, SelState* __restrict__ states,
                                                        unsigned int* __restrict__ hist) {
    __shared__ unsigned int h[kSelBins];
    const int k = first + (int)blockIdx.y, t = threadIdx.x;
    const SelState s = sel_state(states, hist, k, pass, np, blockIdx.x == 0);
    if (sel_small(s)) return;  // the same in every thread
    double m[3] = {0.0, 0.0, 0.0};
    if (k == 3)
        for (int j = 0; j < 3; ++j) m[j] = key_value(found[j]);
    for (int i = t; i < kSelBins; i += kSelBlock) h[i] = 0;
    __syncthreads();
    const int top = 64 - (int)s.bits, shift = max(0, top - kSelBits);  // bits [shift, top) of the keys
    const unsigned int mask = (1u << (top - shift)) - 1;
    for (int64_t i0 = (int64_t)blockIdx.x * kSelRound; i0 < np; i0 += (int64_t)gridDim.x * kSelRound) {
        unsigned long long key[kSelUnroll];
        sel_round(pt, i0, np, k, m, key);
#pragma unroll
        for (int u = 0; u < kSelUnroll; ++u)
            if (i0 + u * kSelBlock + t < np && (pass == 0 || ((key[u] ^ s.prefix) >> top) == 0))
                atomicAdd(&h[(unsigned int)(key[u] >> shift) & mask], 1u);
    }
    __syncthreads();
    // integer counts: the sum does not depend on the order the blocks add in
    unsigned int* out = hist + (size_t)(4 * pass + k) * kSelBins;
    for (int i = t; i < kSelBins; i += kSelBlock)
        if (h[i]) atomicAdd(&out[i], h[i]);
}

// After `passes` histograms: the keys that share the digits so far (at most `stride`: all points, or kSelCap after
// all the passes) and their range.  None when the digits are the whole key.  A block reserves the places of a
// round's keys with one addition, as all of them may be collected.
__global__ void __launch_bounds__(kSelBlock) k_sel_collect(const double* __restrict__ pt, int np, int first, int passes,
                                                           const unsigned long long* __restrict__ found,
                                                           SelState* __restrict__ states, const unsigned int* __restrict__ hist,
                                                           unsigned int* __restrict__ count,
                                                           unsigned long long* __restrict__ range,
                                                           unsigned long long* __restrict__ keys, int stride) {
    constexpr int NW = kSelBlock / 64;
    __shared__ unsigned int wave_n[NW], base;
    const int k = first + (int)blockIdx.y, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const SelState s = sel_state(states, hist, k, passes, np, blockIdx.x == 0);
    if (s.bits == 64) return;  // the same in every thread
    double m[3] = {0.0, 0.0, 0.0};
    if (k == 3)
        for (int j = 0; j < 3; ++j) m[j] = key_value(found[j]);
    const int top = 64 - (int)s.bits;
    unsigned long long lo = ~0ull, hi = 0;
    for (int64_t i0 = (int64_t)blockIdx.x * kSelRound; i0 < np; i0 += (int64_t)gridDim.x * kSelRound) {
        unsigned long long key[kSelUnroll], here[kSelUnroll];
        sel_round(pt, i0, np, k, m, key);
        unsigned int n = 0;  // the wave's keys
#pragma unroll
        for (int u = 0; u < kSelUnroll; ++u) {
            here[u] = __ballot(i0 + u * kSelBlock + t < np && ((key[u] ^ s.prefix) >> top) == 0);
            n += (unsigned int)__popcll(here[u]);
        }
        if (lane == 0) wave_n[wave] = n;
        __syncthreads();
        if (t == 0) {
            unsigned int all = 0;
            for (int w = 0; w < NW; ++w) all += wave_n[w];
            base = all ? atomicAdd(&count[k], all) : 0;
        }
        __syncthreads();
        unsigned int at = base;
        for (int w = 0; w < wave; ++w) at += wave_n[w];
        if (n)
#pragma unroll
            for (int u = 0; u < kSelUnroll; ++u) {
                if ((here[u] >> lane) & 1) {
                    keys[(size_t)(k % 3) * stride + at + __popcll(here[u] & ((1ull << lane) - 1))] = key[u];
                    lo = min(lo, key[u]);
                    hi = max(hi, key[u]);
                }
                at += (unsigned int)__popcll(here[u]);
            }
        __syncthreads();  // wave_n and base have been read
    }
    if (__ballot(lo <= hi) == 0) return;  // most waves have none
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        lo = min(lo, __shfl_xor(lo, d, 64));
        hi = max(hi, __shfl_xor(hi, d, 64));
    }
    if (lane == 0) {
        atomicMin(&range[2 * k], lo);
        atomicMax(&range[2 * k + 1], hi);
    }
}

// The key of rank `rank` of the n collected ones at `mine`, which lie in [lo, hi], lo < hi, by NT threads.  From the
// first bit they differ in, a histogram of kSelBits bits, and again on the keys of its bin, which are kept in
// `list` once they are few; ended when they are one value.
template <int NT>
__device__ __forceinline__ unsigned long long sel_last_bits(const unsigned long long* __restrict__ mine, int n, unsigned long long rank,
                                                            unsigned long long lo, unsigned long long hi, unsigned int* h,
                                                            unsigned long long* list) {
    constexpr int U = 8, NW = NT / 64;
    __shared__ unsigned int listed;
    __shared__ unsigned long long and_w[NW], or_w[NW];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int top = 64 - __clzll((long long)(lo ^ hi));  // at most 42: the keys share the passes' digits
    unsigned long long prefix = lo >> top << top;
    bool in_lds = false;
    // f(key without the prefix) for every key that has it
    auto each_key = [&](auto f) {
        if (in_lds) {
            for (int i = t; i < n; i += NT) {
                const unsigned long long x = list[i] ^ prefix;
                if (x < 1ull << top) f(x);
            }
            return;
        }
        for (int i0 = 0; i0 < n; i0 += U * NT) {
            unsigned long long x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) x[u] = mine[min(i0 + u * NT + t, n - 1)] ^ prefix;
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (i0 + u * NT + t < n && x[u] < 1ull << top) f(x[u]);
        }
    };
    for (unsigned int left = (unsigned int)n;;) {
        for (int i = t; i < kSelBins; i += NT) h[i] = 0;
        if (!in_lds && left <= kFinishList) {
            if (t == 0) listed = 0;
            __syncthreads();
            each_key([&](unsigned long long x) {
                const unsigned long long here = __ballot(1);
                const int leader = __ffsll(here) - 1;
                unsigned int at = 0;
                if (lane == leader) at = atomicAdd(&listed, (unsigned int)__popcll(here));
                list[__shfl(at, leader, 64) + __popcll(here & ((1ull << lane) - 1))] = x ^ prefix;
            });
            in_lds = true;
            n = (int)left;
        }
        __syncthreads();
        const int shift = max(0, top - kSelBits);
        unsigned long long all_and = ~0ull, all_or = 0;
        each_key([&](unsigned long long x) {
            all_and &= x;
            all_or |= x;
            const unsigned int bin = (unsigned int)(x >> shift), bin0 = __builtin_amdgcn_readfirstlane(bin);
            const unsigned long long same = __ballot(bin == bin0);
            if (bin != bin0)
                atomicAdd(&h[bin], 1u);
            else if (lane == __ffsll(same) - 1)
                atomicAdd(&h[bin], (unsigned int)__popcll(same));
        });
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            all_and &= __shfl_xor(all_and, d, 64);
            all_or |= __shfl_xor(all_or, d, 64);
        }
        if (lane == 0) {
            and_w[wave] = all_and;
            or_w[wave] = all_or;
        }
        __syncthreads();
        for (int w = 0; w < NW; ++w) {
            all_and &= and_w[w];
            all_or |= or_w[w];
        }
        if (all_and == all_or) return prefix | all_or;  // one value; the same in every thread
        prefix |= (unsigned long long)sel_pick<NT>(h, &rank, &left) << shift;
        top = shift;
        if (top == 0) return prefix;
        __syncthreads();
    }
}

// The remaining bits over the collected keys, one block per selection; their order does not matter.  A few hundred
// keys are work for four waves, whose barriers cost less than sixteen's.  With all of 100,000 keys collected it
// is bound by one CU's instructions, hence all its threads, eight loads a thread in flight, and the lanes of a
// wave whose key falls into its first lane's bin, often all of them, counted by one addition: 60 us (340 with a quarter
// of the threads, a load at a time and an addition a key).
__global__ void __launch_bounds__(kFinishBlock) k_sel_finish(int first, int passes, const SelState* __restrict__ states,
                                                             const unsigned int* __restrict__ count,
                                                             const unsigned long long* __restrict__ range,
                                                             const unsigned long long* __restrict__ keys, int stride,
                                                             unsigned long long* __restrict__ found) {
    __shared__ unsigned int h[kSelBins];
    __shared__ unsigned long long list[kFinishList];
    const int k = first + (int)blockIdx.x;
    const SelState s = states[(kSelPasses + 1) * k + passes];
    const int n = (int)count[k];
    const unsigned long long lo = range[2 * k], hi = range[2 * k + 1];
    const unsigned long long* mine = keys + (size_t)(k % 3) * stride;
    unsigned long long key;
    if (s.bits == 64) {
        key = s.prefix;
    } else if (lo == hi) {
        key = lo;
    } else if (n <= kFinishList) {
        if (threadIdx.x >= kSelBlock) return;
        key = sel_last_bits<kSelBlock>(mine, n, s.rank, lo, hi, h, list);
    } else {
        key = sel_last_bits<kFinishBlock>(mine, n, s.rank, lo, hi, h, list);
    }
    if (threadIdx.x == 0) found[k] = key;
}

// BALProblem.cpp:283-302: X <- s (X - m), camera centres likewise, s = 100 / MAD
__global__ void k_norm_apply(double* __restrict__ pt, int np, double* __restrict__ cam, int nc,
                             const unsigned long long* __restrict__ found) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const double m[3] = {key_value(found[0]), key_value(found[1]), key_value(found[2])};
    const double scale = 100.0 / key_value(found[3]);
    if (i < np)
        for (int j = 0; j < 3; ++j) pt[4 * (int64_t)i + j] = scale * (pt[4 * (int64_t)i + j] - m[j]);
    if (i < nc) {
        double aa[3], t[3], center[3];
        for (int j = 0; j < 3; ++j) {
            aa[j] = cam[(size_t)j * nc + i];
            t[j] = cam[(size_t)(3 + j) * nc + i];
        }
        camera_center(aa, t, center);
        for (int j = 0; j < 3; ++j) center[j] = scale * (center[j] - m[j]);
        center_translation(aa, center, t);
        for (int j = 0; j < 3; ++j) cam[(size_t)(3 + j) * nc + i] = t[j];
    }
}

template <typename T>
int ensure(DevBuf<T>& b, size_t n) {
    return b.n >= n ? BA_OK : b.alloc(n);
}

}  // namespace

int64_t first_pairs(int64_t n_normals);
int draw_normals(int64_t n_normals, int64_t n_pairs, uint32_t seed, PrepScratch* w, hipStream_t s);

int device_normalize(const DeviceParams& p, PrepScratch* w, hipStream_t s) {
    if (p.np == 0) return BA_OK;  // BALProblem.cpp:263-303 leaves an empty problem as it is
    const int np = p.np;
    const int nblocks = std::max(1, std::min(256, div_up(np, kSelBlock * 8)));
    const int passes = np > kSelSpread ? kSelPasses : 2;
    const int words = 4 * passes * kSelBins, stride = np > kSelSpread ? (int)kSelCap : np;
    constexpr int kStateWords = sizeof(SelState) / sizeof(unsigned long long) * 4 * (kSelPasses + 1);
    BA_TRY(ensure(w->sel_state, kStateWords + 12));
    BA_TRY(ensure(w->hist, (size_t)words + 4));
    BA_TRY(ensure(w->keys, 3 * (size_t)stride));
    unsigned int* count = w->hist.p + words;
    SelState* states = reinterpret_cast<SelState*>(w->sel_state.p);
    unsigned long long *found = w->sel_state.p + kStateWords, *range = found + 4;
    hipLaunchKernelGGL(k_sel_init, dim3(words / 256), dim3(256), 0, s, w->hist.p, words, count, range);
    for (int first : {0, 3}) {  // the axes together, then the distances to their medians
        const int n = first == 0 ? 3 : 1;
        for (int pass = 0; pass < passes; ++pass)
            hipLaunchKernelGGL(k_sel_hist, dim3(nblocks, n), dim3(kSelBlock), 0, s, p.pt, np, first, pass,
                               (const unsigned long long*)found, states, w->hist.p);
        hipLaunchKernelGGL(k_sel_collect, dim3(nblocks, n), dim3(kSelBlock), 0, s, p.pt, np, first, passes,
                           (const unsigned long long*)found, states, (const unsigned int*)w->hist.p, count, range, w->keys.p,
                           stride);
        hipLaunchKernelGGL(k_sel_finish, dim3(n), dim3(kFinishBlock), 0, s, first, passes, (const SelState*)states,
                           (const unsigned int*)count, (const unsigned long long*)range, (const unsigned long long*)w->keys.p, stride,
                           found);
    }
    hipLaunchKernelGGL(k_norm_apply, dim3(div_up(std::max(np, p.nc), 256)), dim3(256), 0, s, p.pt, np, p.cam, p.nc,
                       (const unsigned long long*)found);
    BA_HIP(hipGetLastError());
    return BA_OK;
}

int device_perturb(const DeviceParams& p, uint32_t seed, double rs, double ts, double ps, PrepScratch* w,
                   hipStream_t s) {
    const int64_t n_pt = ps > 0.0 ? 3 * (int64_t)p.np : 0;
    const int64_t n_normals = n_pt + (int64_t)p.nc * ((rs > 0.0 ? 3 : 0) + (ts > 0.0 ? 3 : 0));
    if (n_normals > (int64_t)1 << 30) return fail(BA_ERR_CAPACITY, "perturbation needs %lld normals (limit 2^30)",
                                                   (long long)n_normals);
    int64_t n_pairs = first_pairs(n_normals);
    BA_TRY(ensure(w->total, 1));
    for (;;) {
        if (n_normals > 0) BA_TRY(draw_normals(n_normals, n_pairs, seed, w, s));
        if (ps > 0.0 && p.np > 0)
            hipLaunchKernelGGL(k_perturb_points, dim3(div_up(p.np, 256)), dim3(256), 0, s, p.pt, p.pt_orig, p.np,
                               (const double*)w->normals.p, ps, (const int*)w->total.p, (int)n_normals);
        // every camera goes through centre and back, as in the reference, also with both sigmas 0
        if (p.nc > 0)
            hipLaunchKernelGGL(k_perturb_cams, dim3(div_up(p.nc, 64)), dim3(64), 0, s, p.cam, p.nc,
                               (const double*)w->normals.p, n_pt, rs, ts, (const int*)w->total.p, (int)n_normals);
        BA_HIP(hipGetLastError());
        if (n_normals == 0) return BA_OK;
        int got = 0;
        BA_HIP(hipMemcpyAsync(&got, w->total.p, sizeof(int), hipMemcpyDeviceToHost, s));
        BA_HIP(hipStreamSynchronize(s));
        if (got >= n_normals) return BA_OK;
        n_pairs += n_pairs / 2;
    }
}

// Pairs to draw for n normals: the acceptance rate is pi/4, so 1.3 per normal leaves a margin of many
// standard deviations; a shortfall (read back by the caller) draws again with more.
int64_t first_pairs(int64_t n_normals) { return n_normals + n_normals * 3 / 10 + 4096; }

// Normals 0..n_normals-1 of the stream glibc's rand() gives after srand(seed), from n_pairs pairs of draws,
// into w->normals; the number of accepted pairs into w->total.
int draw_normals(int64_t n_normals, int64_t n_pairs, uint32_t seed, PrepScratch* w, hipStream_t s) {
    const std::vector<uint32_t>& tables = jump_tables();
    if (!w->table_chunks) {
        BA_TRY(w->tables.upload(tables.data(), tables.size(), s));
        w->table_chunks = 1;
    }
    const RandState start = glibc_seed_state(seed);
    const int64_t n_draws = 2 * n_pairs;
    const int n_chunks = div_up(n_draws, kChunk);
    if (n_chunks >= (1 << kJumps)) return fail(BA_ERR_CAPACITY, "random stream too long");
    const int nb = div_up(n_pairs, kPairsPerBlock);
    BA_TRY(ensure(w->total, 1));
    BA_TRY(ensure(w->draws, (size_t)n_draws));
    BA_TRY(ensure(w->counts, (size_t)nb));
    BA_TRY(ensure(w->normals, (size_t)n_normals));
    hipLaunchKernelGGL(k_rand_generate, dim3(div_up(n_chunks, kBlockChunks)), dim3(256), 0, s, start, w->tables.p, n_draws,
                       w->draws.p);
    hipLaunchKernelGGL(k_pairs_count, dim3(nb), dim3(kPairBlock), 0, s, w->draws.p, n_pairs, (int*)w->counts.p);
    hipLaunchKernelGGL(k_pairs_scan, dim3(1), dim3(kPairBlock), 0, s, (int*)w->counts.p, nb, w->total.p);
    hipLaunchKernelGGL(k_pairs_emit, dim3(nb), dim3(kPairBlock), 0, s, w->draws.p, n_pairs, (const int*)w->counts.p,
                       (int)n_normals, w->normals.p);
    BA_HIP(hipGetLastError());
    return BA_OK;
}

}  // namespace mba
