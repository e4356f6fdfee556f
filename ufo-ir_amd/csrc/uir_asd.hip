// uir_asd.hip -- the per-slice steps of batched ASD-POCS (ufo-ir-asdpocs-task.c:411-509)
// between the projections: positivity, the image distances, the TV steps
// and the FP64 reductions that set the TV step length and the data-constraint
// test, all on the device so that one iteration replays as a hipGraph.
//
// Every kernel runs over a grid (blocks per slice, slices): block (c, s)
// handles elements [c * kChunk, (c + 1) * kChunk) of slice s and writes one
// FP64 partial sum; uirk_asd_finish adds a slice's partials in a fixed order
// and applies the step's scalar logic to the slice's state.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "uir_device.h"

namespace {

constexpr int kThreads = 256;
constexpr uint32_t kChunk = UIRK_ASD_CHUNK;
constexpr int kPer = kChunk / kThreads;

__device__ __forceinline__ float ld(const float *p, uint32_t i) { return p[i]; }
__device__ __forceinline__ float ld(const __half *p, uint32_t i) { return __half2float(p[i]); }
__device__ __forceinline__ float ld(const __hip_bfloat16 *p, uint32_t i) { return __bfloat162float(p[i]); }
__device__ __forceinline__ void st(float *p, uint32_t i, float v) { p[i] = v; }
__device__ __forceinline__ void st(__half *p, uint32_t i, float v) { p[i] = __float2half(v); }
__device__ __forceinline__ void st(__hip_bfloat16 *p, uint32_t i, float v) { p[i] = __float2bfloat16(v); }

// Block sum of one double per thread; thread 0 writes it to *out.
__device__ __forceinline__ void block_sum(double v, double *out)
{
    __shared__ double red[kThreads / 64];
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0;
        for (int w = 0; w < kThreads / 64; ++w)
            s += red[w];
        *out = s;
    }
}

__device__ __forceinline__ double measure(float d, int l2) { return l2 ? (double)d * (double)d : fabs((double)d); }

// mode 0: x = 0 (the reference restarts its df-minimizer from zero,
// ufo-ir-sart-task.c:205-207); 1: x_prev = x (textbook: warm start, dp
// measured from the image before the data step); 2: x = x_prev (the
// reference's output, the image before the TV steps, :468); 3: x = g read as
// image-dtype data (the SART step's second buffer).
template <typename TI>
__global__ __launch_bounds__(kThreads) void k_asd_begin(const uirk_asd_slice *__restrict__ sl, int mode)
{
    const uirk_asd_slice S = sl[blockIdx.y];
    const uint32_t nv = S.n * S.n, base = blockIdx.x * kChunk;
    if (base >= nv)
        return;
    TI *x = (TI *)S.x, *xp = (TI *)S.x_prev;
    for (int k = 0; k < kPer; ++k) {
        const uint32_t i = base + k * kThreads + threadIdx.x;
        if (i < nv) {
            if (mode == 1)
                xp[i] = x[i];
            else if (mode == 2)
                x[i] = xp[i];
            else if (mode == 3)
                x[i] = ((const TI *)S.g)[i];
            else
                st(x, i, 0.0f);
        }
    }
}

// After the data step: x = POSC(x) (ufo-ir-asdpocs-task.c:463-465), partial of
// |x - x_prev| (dp, :481-483), then x_prev = x (:490).
template <typename TI>
__global__ __launch_bounds__(kThreads) void k_asd_posc_dp(const uirk_asd_slice *__restrict__ sl, int posc, int l2,
                                                          double *__restrict__ partials, int nblk)
{
    const uirk_asd_slice S = sl[blockIdx.y];
    const uint32_t nv = S.n * S.n, base = blockIdx.x * kChunk;
    double acc = 0;
    if (base < nv) {
        TI *x = (TI *)S.x, *xp = (TI *)S.x_prev;
        for (int k = 0; k < kPer; ++k) {
            const uint32_t i = base + k * kThreads + threadIdx.x;
            if (i < nv) {
                float v = ld(x, i);
                if (posc && !(v > 0.0f)) {
                    v = 0.0f;
                    st(x, i, v);
                }
                acc += measure(v - ld(xp, i), l2);
                st(xp, i, v);
            }
        }
    }
    block_sum(acc, &partials[(size_t)blockIdx.y * nblk + blockIdx.x]);
}

// Partial of |x - x_prev| (dg, :496-497).
template <typename TI>
__global__ __launch_bounds__(kThreads) void k_asd_diff(const uirk_asd_slice *__restrict__ sl, int l2,
                                                       double *__restrict__ partials, int nblk)
{
    const uirk_asd_slice S = sl[blockIdx.y];
    const uint32_t nv = S.n * S.n, base = blockIdx.x * kChunk;
    double acc = 0;
    if (base < nv) {
        const TI *x = (const TI *)S.x, *xp = (const TI *)S.x_prev;
        for (int k = 0; k < kPer; ++k) {
            const uint32_t i = base + k * kThreads + threadIdx.x;
            if (i < nv)
                acc += measure(ld(x, i) - ld(xp, i), l2);
        }
    }
    block_sum(acc, &partials[(size_t)blockIdx.y * nblk + blockIdx.x]);
}

// Partial of |r| over the residual sinogram b - A x (dd, :471-478).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_asd_sino(const uirk_asd_slice *__restrict__ sl, int l2,
                                                       double *__restrict__ partials, int nblk)
{
    const uirk_asd_slice S = sl[blockIdx.y];
    const uint32_t ns = S.n_sino;
    double acc = 0;
    for (uint32_t base = blockIdx.x * kChunk; base < ns; base += (uint32_t)nblk * kChunk) {
        const T *r = (const T *)S.r;
        for (int k = 0; k < kPer; ++k) {
            const uint32_t i = base + k * kThreads + threadIdx.x;
            if (i < ns)
                acc += measure(ld(r, i), l2);
        }
    }
    block_sum(acc, &partials[(size_t)blockIdx.y * nblk + blockIdx.x]);
}

// The smoothed TV gradient of one pixel (ufo-math-tvstd-method.cl:5-57, eps
// 1e-3).  The three quotients v / sqrt(w) are formed as v * rsqrt(w) (hardware
// reciprocal square root, ~1 ulp, a quarter of the rate of other operations);
// the second is the first of the pixel to the right, bit for bit, and comes from
// its lane.  (The third is the first of the pixel above but for the order of two
// additions, which the TV steps amplify: it stays its own.)
constexpr float kTvEps = 0.001f;
__device__ __forceinline__ float tv_root(float f, float left, float below)
{
    return __builtin_amdgcn_rsqf(kTvEps + (f - left) * (f - left) + (f - below) * (f - below));
}
__device__ __forceinline__ float tv_df(float f, float left, float right, float above, float above_left, float below,
                                       float root, float root_right)
{
    const float w2 = kTvEps + (above - f) * (above - f) + (above - above_left) * (above - above_left);
    return (2.0f * f - left - below) * root - (right - f) * root_right -
           (above - f) * __builtin_amdgcn_rsqf(w2);
}

// The value of the next lower / higher lane (column x - 1 / x + 1).
__device__ __forceinline__ float lane_below(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, false)); // wave_shr:1
}
__device__ __forceinline__ float lane_above(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, false)); // wave_shl:1
}

// v as the image's storage holds it
__device__ __forceinline__ float stored(const float *, float v) { return v; }
__device__ __forceinline__ float stored(const __half *, float v) { return __half2float(__float2half(v)); }
__device__ __forceinline__ float stored(const __hip_bfloat16 *, float v)
{
    return __bfloat162float(__float2bfloat16(v));
}

// One TV step and the gradient norm the next one needs, in one pass: x1 = x -
// factor g(x) (operation_deduction2, ufo-ir-basic-ops.cl:104-125, factor = dtgv /
// |g| from the slice's state), from one of the slice's two buffers (S.x, S.g) to
// the other, and the partial of |g(x1)|.  step 0: x1 = x, not written (the norm
// before the first step); norm 0: no partial (the last step).  A slice whose TV
// steps have ended keeps its image.
// A wave owns 60 columns x kTvRows rows and walks down them with the rows in
// registers: lane i holds column base - 2 + i, its neighbours' values come by
// DPP shifts, g(x) is right on lanes 1 .. 62 and g(x1) on lanes 2 .. 61.  So a
// step reads and writes the image once (8 bytes a pixel in FP32); a gradient
// kernel and a step kernel moved 20: 307 us a step over 64 slices of 1024 x
// 1024, this takes 166 (3.1 TB/s).
constexpr int kTvRows = UIRK_ASD_TV_ROWS;
constexpr int kTvCols = UIRK_ASD_TV_COLS;

template <typename TI>
__global__ __launch_bounds__(kThreads) void k_asd_tv(const uirk_asd_slice *__restrict__ sl,
                                                     const uirk_asd_state *__restrict__ state, int from_g, int step,
                                                     int norm, int l2, double *__restrict__ partials, int nblk)
{
    const uirk_asd_slice S = sl[blockIdx.y];
    const int n = (int)S.n;
    const int lane = threadIdx.x & 63;
    const int strips = (n + kTvCols - 1) / kTvCols, bands = (n + kTvRows - 1) / kTvRows;
    const int w = (int)blockIdx.x * (kThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool stop = state[blockIdx.y].stop != 0;
    double acc = 0;
    if (w < strips * bands && (step || !stop)) {
        const TI *in = from_g ? (const TI *)S.g : (const TI *)S.x;
        TI *out = from_g ? (TI *)S.x : (TI *)S.g;
        const float factor = state[blockIdx.y].factor;
        const int c = (w % strips) * kTvCols - 2 + lane;
        const bool cin = c >= 0 && c < n, own = cin && lane >= 2 && lane < 2 + kTvCols;
        const int y0 = (w / strips) * kTvRows, y1 = min(y0 + kTvRows, n);
        auto load = [&](int y) { // 0 outside the image
            return cin && y >= 0 && y < n ? ld(in, (uint32_t)y * (uint32_t)n + (uint32_t)c) : 0.0f;
        };
        constexpr int kAhead = 4; // rows loaded ahead
        float next[kAhead];
        float a = load(y0 - 2), b = load(y0 - 1);
#pragma unroll
        for (int k = 0; k < kAhead; ++k)
            next[k] = load(y0 + k);
        float al = lane_below(a), bl = lane_below(b), br = lane_above(b);
        // x1 of the rows above the current one, and their neighbours
        float p2 = 0, p2l = 0, p1 = 0, p1l = 0, p1r = 0;
        for (int r0 = y0 - 1; r0 <= y1; r0 += kAhead) {
            float cur[kAhead];
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {
                cur[k] = next[k];
                next[k] = load(r0 + 1 + kAhead + k);
            }
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {
                const int r = r0 + k; // x rows r - 1 (a), r (b), r + 1 (d)
                if (r > y1)
                    break;
                const float d = cur[k];
                float v = b;
                if (step && !stop) {
                    const float root = tv_root(b, bl, d);
                    v = stored(in, b - factor * tv_df(b, bl, br, a, al, d, root, lane_above(root)));
                    v = cin && r >= 0 && r < n ? v : 0.0f;
                }
                if (step && own && r >= y0 && r < y1)
                    st(out, (uint32_t)r * (uint32_t)n + (uint32_t)c, v);
                if (norm && !stop && r > y0) {
                    const float root = tv_root(p1, p1l, v);
                    const float df = tv_df(p1, p1l, p1r, p2, p2l, v, root, lane_above(root));
                    acc += own ? measure(df, l2) : 0.0;
                }
                p2 = p1;
                p2l = p1l;
                p1 = v;
                p1l = lane_below(v);
                p1r = lane_above(v);
                a = b;
                al = bl;
                b = d;
                bl = lane_below(d);
                br = lane_above(d);
            }
        }
    }
    if (norm)
        block_sum(acc, &partials[(size_t)blockIdx.y * nblk + blockIdx.x]);
}

// One block per slice: the slice's partials added in a fixed order, then the
// step's scalar update (ufo-ir-asdpocs-task.c:478-503, tvstd :573-579).
__global__ __launch_bounds__(kThreads) void k_asd_finish(uirk_asd_state *__restrict__ state,
                                                         const double *__restrict__ partials, int nblk, int what,
                                                         uirk_asd_params p, float *__restrict__ diag, int n_slices,
                                                         int max_iters)
{
    const int s = blockIdx.x;
    double v = 0;
    for (int c = threadIdx.x; c < nblk; c += kThreads)
        v += partials[(size_t)s * nblk + c];
    __shared__ double total;
    block_sum(v, &total);
    __syncthreads();
    if (threadIdx.x != 0)
        return;
    const double norm = p.textbook ? sqrt(total) : total;
    uirk_asd_state &S = state[s];
    switch (what) {
    case UIRK_ASD_DD:
        S.dd = (float)norm;
        break;
    case UIRK_ASD_DP:
        S.dp = (float)norm;
        if (S.it == 0) // :485-487
            S.dtgv = p.alpha * S.dp;
        S.stop = 0;
        break;
    case UIRK_ASD_G:
        if (S.stop)
            break;
        if (p.textbook && !(norm > 0)) { // a zero gradient ends the steps
            S.stop = 1;
            break;
        }
        S.factor = S.dtgv / (float)norm;
        break;
    default: { // UIRK_ASD_DG: end of the iteration
        S.dg = (float)norm;
        if (S.it < max_iters) {
            float *d = diag + ((size_t)S.it * n_slices + s) * 4;
            d[0] = S.dd;
            d[1] = S.dp;
            d[2] = S.dg;
            d[3] = S.dtgv;
        }
        S.beta *= p.beta_red;                         // :498
        if (S.dg > p.r_max * S.dp && S.dd > 0.001f)  // :495, 501-503
            S.dtgv *= p.alpha_red;
        if (S.beta >= 0.0f && S.beta <= 1.0f)        // :459, a [0, 1] property
            S.relax = S.beta;
        S.it += 1;
        S.stop = 0;
    }
    }
}

template <typename TI>
int launch_image(int kind, const uirk_asd_slice *sl, int n_slices, int nblk, int flag, int l2, double *partials,
                 hipStream_t stm)
{
    const dim3 grid(nblk, n_slices);
    switch (kind) {
    case 0: hipLaunchKernelGGL(k_asd_begin<TI>, grid, dim3(kThreads), 0, stm, sl, flag); break;
    case 1: hipLaunchKernelGGL(k_asd_posc_dp<TI>, grid, dim3(kThreads), 0, stm, sl, flag, l2, partials, nblk); break;
    default: hipLaunchKernelGGL(k_asd_diff<TI>, grid, dim3(kThreads), 0, stm, sl, l2, partials, nblk); break;
    }
    return (int)hipGetLastError();
}

} // namespace

extern "C" {

int uirk_asd_image(int kind, int img_dtype, const uirk_asd_slice *d_sl, int n_slices, int nblk, int flag, int l2,
                   double *d_partials, void *stream)
{
    if (n_slices <= 0 || nblk <= 0 || n_slices > 65535)
        return n_slices == 0 ? 0 : (int)hipErrorInvalidValue;
    hipStream_t stm = (hipStream_t)stream;
    switch (img_dtype) {
    case UIR_DTYPE_F32: return launch_image<float>(kind, d_sl, n_slices, nblk, flag, l2, d_partials, stm);
    case UIR_DTYPE_F16: return launch_image<__half>(kind, d_sl, n_slices, nblk, flag, l2, d_partials, stm);
    case UIR_DTYPE_BF16:
        return launch_image<__hip_bfloat16>(kind, d_sl, n_slices, nblk, flag, l2, d_partials, stm);
    default: return (int)hipErrorInvalidValue;
    }
}

int uirk_asd_tv(int img_dtype, const uirk_asd_slice *d_sl, int n_slices, int max_n, int nblk,
                const uirk_asd_state *d_state, int from_g, int step, int norm, int l2, double *d_partials, void *stream)
{
    if (n_slices <= 0 || nblk <= 0 || n_slices > 65535)
        return n_slices == 0 ? 0 : (int)hipErrorInvalidValue;
    const int waves = ((max_n + kTvCols - 1) / kTvCols) * ((max_n + kTvRows - 1) / kTvRows);
    const int blocks = (waves + kThreads / 64 - 1) / (kThreads / 64);
    if (blocks > nblk)
        return (int)hipErrorInvalidValue;
    const dim3 grid(norm ? nblk : blocks, n_slices); // every partial of a norm is written
    hipStream_t stm = (hipStream_t)stream;
    switch (img_dtype) {
    case UIR_DTYPE_F32:
        hipLaunchKernelGGL(k_asd_tv<float>, grid, dim3(kThreads), 0, stm, d_sl, d_state, from_g, step, norm, l2,
                           d_partials, nblk);
        break;
    case UIR_DTYPE_F16:
        hipLaunchKernelGGL(k_asd_tv<__half>, grid, dim3(kThreads), 0, stm, d_sl, d_state, from_g, step, norm, l2,
                           d_partials, nblk);
        break;
    case UIR_DTYPE_BF16:
        hipLaunchKernelGGL(k_asd_tv<__hip_bfloat16>, grid, dim3(kThreads), 0, stm, d_sl, d_state, from_g, step, norm,
                           l2, d_partials, nblk);
        break;
    default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

int uirk_asd_sino_norm(int dtype, const uirk_asd_slice *d_sl, int n_slices, int nblk, int l2, double *d_partials,
                       void *stream)
{
    if (n_slices <= 0 || nblk <= 0 || n_slices > 65535)
        return n_slices == 0 ? 0 : (int)hipErrorInvalidValue;
    const dim3 grid(nblk, n_slices);
    hipStream_t stm = (hipStream_t)stream;
    switch (dtype) {
    case UIR_DTYPE_F32:
        hipLaunchKernelGGL(k_asd_sino<float>, grid, dim3(kThreads), 0, stm, d_sl, l2, d_partials, nblk);
        break;
    case UIR_DTYPE_F16:
        hipLaunchKernelGGL(k_asd_sino<__half>, grid, dim3(kThreads), 0, stm, d_sl, l2, d_partials, nblk);
        break;
    case UIR_DTYPE_BF16:
        hipLaunchKernelGGL(k_asd_sino<__hip_bfloat16>, grid, dim3(kThreads), 0, stm, d_sl, l2, d_partials, nblk);
        break;
    default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

int uirk_asd_finish(uirk_asd_state *d_state, const double *d_partials, int n_slices, int nblk, int what,
                    const uirk_asd_params *p, float *d_diag, int max_iters, void *stream)
{
    if (n_slices <= 0)
        return 0;
    hipLaunchKernelGGL(k_asd_finish, dim3(n_slices), dim3(kThreads), 0, (hipStream_t)stream, d_state, d_partials, nblk,
                       what, *p, d_diag, n_slices, max_iters);
    return (int)hipGetLastError();
}

} // extern "C"
