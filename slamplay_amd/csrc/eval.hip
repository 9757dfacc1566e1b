// eval.hip -- per-observation Snavely residual + Jacobian on the GPU (the parity entry point that
// replaces one AutoDiffCostFunction<SnavelyReprojectionError,2,9,3> evaluation per residual block,
// utils/camera/SnavelyReprojectionError.h:42-92), and the FP64 cost 1/2 sum rho(|r|^2).
//
// Layout: observations in caller order; cameras AoS (9 doubles) as in BALProblem.  One thread per
// observation.  The Jacobian entry's camera preps are computed once per camera by k_camera_prep_aos; the cost
// has eleven terms per camera of its own (CostCam).
#include <algorithm>
#include <map>
#include <mutex>

#include "common.h"
#include "lm_kernels.h"
#include "snavely.h"

namespace mba {

template <typename Real>
__global__ void k_camera_prep_aos(const double* __restrict__ cams, int nc, CameraPrep<Real>* __restrict__ prep) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    double cam[9];
    for (int i = 0; i < 9; ++i) cam[i] = cams[9 * (size_t)c + i];
    CameraPrep<Real> P;
    camera_prep<Real>(cam, P);
    prep[c] = P;
}

template <typename Real>
__global__ void k_eval_obs(int no, const int* __restrict__ ci, const int* __restrict__ pi,
                           const double* __restrict__ obs, const double* __restrict__ pts,
                           const CameraPrep<Real>* __restrict__ prep, double* __restrict__ r_out,
                           double* __restrict__ jc_out, double* __restrict__ jp_out) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= no) return;
    const CameraPrep<Real> P = prep[ci[k]];
    const int p = pi[k];
    const double X[3] = {pts[3 * (size_t)p], pts[3 * (size_t)p + 1], pts[3 * (size_t)p + 2]};
    Real r[2], Jc[18], Jp[6];
    snavely_residual_jacobian<Real>(P, X, (Real)obs[2 * (size_t)k], (Real)obs[2 * (size_t)k + 1], r, Jc, Jp);
    r_out[2 * (size_t)k] = (double)r[0];
    r_out[2 * (size_t)k + 1] = (double)r[1];
    if (jc_out)
        for (int i = 0; i < 18; ++i) jc_out[18 * (size_t)k + i] = (double)Jc[i];
    if (jp_out)
        for (int i = 0; i < 6; ++i) jp_out[6 * (size_t)k + i] = (double)Jp[i];
}

// ---------------------------------------------------------------------------------------------
// FP64 cost 1/2 sum rho(|r|^2): per-block partial sums, then k_sum_partials, both in a fixed order.
//
// Observations come in the caller's order (BAL files list them by point), so every observation gathers
// another camera.  Of a camera's terms the residual needs eleven doubles (below); the 368-byte
// CameraPrep spread them over three cache lines, and gathering those bound the kernel (32 us for 1.2M
// observations of 1,500 cameras, 783 GB/s of inputs).  How a block gets at them:
//   kCostPrep   up to 256 cameras: every block computes them into its LDS, one camera per thread, and no
//               launch of its own is needed;
//   kCostGather beyond: computed once by k_cost_cameras, gathered from memory, 88 contiguous bytes each.
// 1.2M observations of 1,500 cameras: 40 -> 22 us a call on inputs that the caches still hold, 49.5 -> 28.6 on
// twelve sets of them in turn, 430 MB (a copy of the whole table in every CU's LDS, 132 KB, instead of the
// gather: 1 us more); 14.9k observations of 16 cameras: 12.7 -> 9.7 us, the rate the host issues two launches at.
struct CostCam {
    double u[3], c, s;   // R X = X c + (u x X) s + u (u.X)(1 - c)
    double t[3], f, k1, k2;
};
static_assert(sizeof(CostCam) == 88, "eleven doubles per camera");
enum { kCostPrep = 0, kCostGather = 1 };
constexpr int kCostPrepCams = 256;

__device__ __forceinline__ CostCam cost_camera(const double* __restrict__ cam) {
    CameraPrep<double> P;
    double a[9];
    for (int i = 0; i < 9; ++i) a[i] = cam[i];
    camera_prep<double>(a, P);
    CostCam q;
    for (int i = 0; i < 3; ++i) {
        q.u[i] = P.u[i];
        q.t[i] = P.t[i];
    }
    q.c = P.c;
    // the first-order branch R X = X + w x X is the same expression with c = 1 and s = 1
    q.s = P.taylor ? 1.0 : P.s;
    q.f = P.f;
    q.k1 = P.k1;
    q.k2 = P.k2;
    return q;
}

__global__ void k_cost_cameras(const double* __restrict__ cams, int nc, CostCam* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < nc) out[c] = cost_camera(cams + 9 * (size_t)c);
}

// snavely_residual with a CostCam (the same operations in the same order).
__device__ __forceinline__ double cost_term(const CostCam& q, const double X[3], double ox, double oy, int loss, double a) {
    const double wx[3] = {q.u[1] * X[2] - q.u[2] * X[1], q.u[2] * X[0] - q.u[0] * X[2], q.u[0] * X[1] - q.u[1] * X[0]};
    const double tmp = (q.u[0] * X[0] + q.u[1] * X[1] + q.u[2] * X[2]) * (1.0 - q.c);
    double p[3];
    for (int i = 0; i < 3; ++i) p[i] = X[i] * q.c + wx[i] * q.s + q.u[i] * tmp + q.t[i];
    const double ginv = 1.0 / p[2];
    const double xp = -p[0] * ginv, yp = -p[1] * ginv;
    const double r2 = xp * xp + yp * yp;
    const double fd = q.f * (1.0 + r2 * (q.k1 + q.k2 * r2));
    const double r0 = fd * xp - ox, r1 = fd * yp - oy;
    return half_rho(r0 * r0 + r1 * r1, loss, a);
}

// Indices are checked on the device (an observation whose camera or point index is out of range
// contributes NaN, so the cost is NaN): callers with host arrays have had them validated already, those
// with device arrays have not.
template <int MODE>
__global__ void __launch_bounds__(256) k_cost_obs(int no, int nc, int np, const int* __restrict__ ci, const int* __restrict__ pi,
                                                 const double* __restrict__ obs, const double* __restrict__ pts,
                                                 const double* __restrict__ cams, const CostCam* __restrict__ prep, int loss,
                                                 double a, double* __restrict__ partial) {
    constexpr int NT = 256;
    __shared__ CostCam tab[MODE == kCostPrep ? kCostPrepCams : 1];
    __shared__ double red[NT / 64];
    if (MODE == kCostPrep) {
        if ((int)threadIdx.x < nc) tab[threadIdx.x] = cost_camera(cams + 9 * (size_t)threadIdx.x);
        __syncthreads();
    }
    double acc = 0.0;
    const int stride = gridDim.x * NT;
    for (int64_t k = (int64_t)blockIdx.x * NT + threadIdx.x; k < no; k += stride) {
        const int cam = ci[k], p = pi[k];
        const double ox = obs[2 * (size_t)k], oy = obs[2 * (size_t)k + 1];
        if (cam < 0 || cam >= nc || p < 0 || p >= np) {
            acc = __builtin_nan("");
            continue;
        }
        const double X[3] = {pts[3 * (size_t)p], pts[3 * (size_t)p + 1], pts[3 * (size_t)p + 2]};
        const CostCam q = MODE == kCostGather ? prep[cam] : tab[cam];
        acc += cost_term(q, X, ox, oy, loss, a);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    acc = wave_sum(acc);
    if (lane == 0) red[wave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = red[0];
        for (int w = 1; w < NT / 64; ++w) s += red[w];
        partial[blockIdx.x] = s;
    }
}

__global__ void k_sum_partials(const double* __restrict__ partial, int n, double* __restrict__ out) {
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += partial[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0];
}

// Blocks of a cost evaluation, one partial sum each: enough for eight waves per SIMD, observations
// beyond them in a grid-stride loop.
constexpr int kCostMaxBlocks = 8 * kCUs;

// Enqueues the evaluation: prep holds nc CostCam (unused up to kCostPrepCams cameras), partial
// kCostMaxBlocks doubles.
inline void enqueue_cost(int no, int nc, int np, const int* ci, const int* pi, const double* obs, const double* pts,
                         const double* cams, CostCam* prep, double* partial, int loss, double a, double* cost, hipStream_t s) {
    const int blocks = std::max(1, std::min(div_up(no, 256), kCostMaxBlocks));
    if (nc <= kCostPrepCams) {
        hipLaunchKernelGGL(k_cost_obs<kCostPrep>, dim3(blocks), dim3(256), 0, s, no, nc, np, ci, pi, obs, pts, cams,
                           (const CostCam*)nullptr, loss, a, partial);
    } else {
        hipLaunchKernelGGL(k_cost_cameras, dim3(div_up(nc, 64)), dim3(64), 0, s, cams, nc, prep);
        hipLaunchKernelGGL(k_cost_obs<kCostGather>, dim3(blocks), dim3(256), 0, s, no, nc, np, ci, pi, obs, pts, cams,
                           (const CostCam*)prep, loss, a, partial);
    }
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, s, (const double*)partial, blocks, cost);
}

// ---------------------------------------------------------------------------------------------
// Allocation-free cost evaluation (ba_eval_cost_noalloc): the kernels of ba_eval_cost with their
// work space (camera preps, per-block partial sums) in a file-scope device array instead of memory
// the library allocates.  Each GPU holds its own copy until the process ends; host code uses the
// address hipGetSymbolAddress returns for the current device, never the array's name.
constexpr int kNoAllocMaxCameras = 4096;
constexpr int kNoAllocMaxObservations = 1 << 24;
constexpr size_t kNoAllocPrepBytes = sizeof(CostCam) * (size_t)kNoAllocMaxCameras;
constexpr size_t kNoAllocPartials = kCostMaxBlocks;
constexpr size_t kNoAllocScratchBytes = kNoAllocPrepBytes + kNoAllocPartials * sizeof(double);
static_assert(kNoAllocPrepBytes % 256 == 0, "partial sums start 256-byte aligned");

__device__ __align__(256) char scratch[kNoAllocScratchBytes];

namespace {

// Device address of `scratch` on the current device, looked up once per device.
int noalloc_scratch(char** out) {
    static std::mutex mu;
    static std::map<int, char*> addr;  // device -> address of its copy of scratch
    int dev = 0;
    BA_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    auto it = addr.find(dev);
    if (it == addr.end()) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return fail(BA_ERR_HIP, "scratch buffer address on device %d: %s", dev, hipGetErrorString(e));
        it = addr.emplace(dev, static_cast<char*>(ptr)).first;
    }
    *out = it->second;
    return BA_OK;
}

struct EvalUpload {
    DevBuf<int> ci, pi;
    DevBuf<double> obs, cams, pts;
    int upload(const ba_problem_view* v, hipStream_t s) {
        BA_TRY(ci.upload(v->camera_index, (size_t)v->num_observations, s));
        BA_TRY(pi.upload(v->point_index, (size_t)v->num_observations, s));
        BA_TRY(obs.upload(v->observations, 2 * (size_t)v->num_observations, s));
        BA_TRY(cams.upload(v->cameras, 9 * (size_t)v->num_cameras, s));
        BA_TRY(pts.upload(v->points, 3 * (size_t)v->num_points, s));
        return BA_OK;
    }
};

struct StreamGuard {
    hipStream_t s = nullptr;
    ~StreamGuard() {
        if (s) (void)hipStreamDestroy(s);
    }
};

template <typename Real>
int eval_impl(const ba_problem_view* v, double* residuals, double* jc, double* jp, hipStream_t s) {
    EvalUpload u;
    BA_TRY(u.upload(v, s));
    const int no = v->num_observations, nc = v->num_cameras;
    DevBuf<CameraPrep<Real>> prep;
    DevBuf<double> r, Jc, Jp;
    BA_TRY(prep.alloc(nc));
    BA_TRY(r.alloc(2 * (size_t)no));
    if (jc) BA_TRY(Jc.alloc(18 * (size_t)no));
    if (jp) BA_TRY(Jp.alloc(6 * (size_t)no));
    hipLaunchKernelGGL(k_camera_prep_aos<Real>, dim3(div_up(nc, 64)), dim3(64), 0, s, u.cams.p, nc, prep.p);
    BA_HIP(hipGetLastError());
    if (no > 0) {
        hipLaunchKernelGGL(k_eval_obs<Real>, dim3(div_up(no, 256)), dim3(256), 0, s, no, u.ci.p, u.pi.p, u.obs.p,
                           u.pts.p, prep.p, r.p, jc ? Jc.p : nullptr, jp ? Jp.p : nullptr);
        BA_HIP(hipGetLastError());
    }
    BA_HIP(hipMemcpyAsync(residuals, r.p, 2 * (size_t)no * sizeof(double), hipMemcpyDeviceToHost, s));
    if (jc) BA_HIP(hipMemcpyAsync(jc, Jc.p, 18 * (size_t)no * sizeof(double), hipMemcpyDeviceToHost, s));
    if (jp) BA_HIP(hipMemcpyAsync(jp, Jp.p, 6 * (size_t)no * sizeof(double), hipMemcpyDeviceToHost, s));
    BA_HIP(hipStreamSynchronize(s));
    return BA_OK;
}

}  // namespace
}  // namespace mba

using namespace mba;

extern "C" int ba_eval_residual_jacobian(const ba_problem_view* v, int32_t precision, double* residuals,
                                         double* jac_camera, double* jac_point) {
    clear_error();
    BA_TRY(validate_view(v, true));
    if (!residuals) return fail(BA_ERR_INVALID_ARGUMENT, "residuals output is NULL");
    if (precision != BA_PRECISION_FP64 && precision != BA_PRECISION_MIXED)
        return fail(BA_ERR_INVALID_ARGUMENT, "unknown precision %d", precision);
    BA_TRY(use_device(0));
    StreamGuard g;
    BA_HIP(hipStreamCreateWithFlags(&g.s, hipStreamNonBlocking));
    if (precision == BA_PRECISION_FP64) return eval_impl<double>(v, residuals, jac_camera, jac_point, g.s);
    return eval_impl<float>(v, residuals, jac_camera, jac_point, g.s);
}

extern "C" int ba_eval_cost(const ba_problem_view* v, int32_t loss, double loss_scale, double* cost) {
    clear_error();
    BA_TRY(validate_view(v, true));
    if (!cost) return fail(BA_ERR_INVALID_ARGUMENT, "cost output is NULL");
    BA_TRY(use_device(0));
    StreamGuard g;
    BA_HIP(hipStreamCreateWithFlags(&g.s, hipStreamNonBlocking));
    EvalUpload u;
    BA_TRY(u.upload(v, g.s));
    const int no = v->num_observations, nc = v->num_cameras;
    if (nc == 0) return fail(BA_ERR_INVALID_ARGUMENT, "no cameras");
    DevBuf<CostCam> prep;
    BA_TRY(prep.alloc(nc));
    DevBuf<double> partial, out;
    BA_TRY(partial.alloc(kCostMaxBlocks));
    BA_TRY(out.alloc(1));
    enqueue_cost(no, nc, v->num_points, u.ci.p, u.pi.p, u.obs.p, u.pts.p, u.cams.p, prep.p, partial.p, loss, loss_scale, out.p,
                 g.s);
    BA_HIP(hipGetLastError());
    BA_HIP(hipMemcpyAsync(cost, out.p, sizeof(double), hipMemcpyDeviceToHost, g.s));
    BA_HIP(hipStreamSynchronize(g.s));
    return BA_OK;
}

extern "C" int ba_eval_cost_noalloc(const ba_problem_view* v, int32_t loss, double loss_scale, double* cost,
                                    void* stream) {
    clear_error();
    if (!v || !cost) return fail(BA_ERR_INVALID_ARGUMENT, "NULL argument");
    if (v->camera_block_size != 9) return fail(BA_ERR_INVALID_ARGUMENT, "camera_block_size must be 9");
    const int no = v->num_observations, nc = v->num_cameras, np = v->num_points;
    if (no < 0 || nc < 0 || np < 0) return fail(BA_ERR_INVALID_ARGUMENT, "negative problem size");
    if (nc > kNoAllocMaxCameras || no > kNoAllocMaxObservations)
        return fail(BA_ERR_CAPACITY, "ba_eval_cost_noalloc holds at most %d cameras and %d observations (got %d, %d)",
                    kNoAllocMaxCameras, kNoAllocMaxObservations, nc, no);
    if (no > 0 && (!v->camera_index || !v->point_index || !v->observations || !v->points))
        return fail(BA_ERR_INVALID_ARGUMENT, "observation or point arrays are NULL");
    if (nc > 0 && !v->cameras) return fail(BA_ERR_INVALID_ARGUMENT, "camera array is NULL");
    char* base = nullptr;
    BA_TRY(noalloc_scratch(&base));
    hipStream_t s = static_cast<hipStream_t>(stream);
    enqueue_cost(no, nc, np, v->camera_index, v->point_index, v->observations, v->points, v->cameras,
                 reinterpret_cast<CostCam*>(base), reinterpret_cast<double*>(base + kNoAllocPrepBytes), loss, loss_scale, cost, s);
    BA_HIP(hipGetLastError());
    return BA_OK;
}
