// uir_kernels.hip -- reference-compatible gfx950 kernels of libuir: the Joseph
// forward projector and backprojector, the elementwise kernels of
// ufo-ir-basic-ops.cl, finite differences, the smoothed-TV gradient and the
// reductions that ufo-ir ran as host loops.
//
// Built with -ffp-contract=off: every float operation rounds where the
// reference source rounds, so these kernels reproduce the reference's
// arithmetic operation for operation (sum order included).  The fast
// reduced-precision batched kernels live in uir_fast.hip.
#include <hip/hip_runtime.h>

#include <cstring>
#include <type_traits>

#include "uir_device.h"

namespace {

constexpr int kBlockSamples = 64; // projector-parallel-joseph.cl:4

// A raw buffer load whose byte offset lies at or beyond the resource's size
// returns zero and touches no memory (negative offsets are large unsigned
// ones): the zero border of a row.  The offset has to be whole in the vector
// register, as the check does not see a wrap by an immediate one (opaque).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const float *base, uint32_t elems)
{
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, (int)(elems * 4u), 0x00020000);
}
__device__ __forceinline__ float row_load(__amdgpu_buffer_rsrc_t r, int i)
{
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (uint32_t)i * 4u, 0, 0));
}
__device__ __forceinline__ int opaque(int i)
{
    asm("" : "+v"(i));
    return i;
}

// --------------------------------------------------------------------------
// Joseph forward projection, one thread per ray (detector s, angle).
// --------------------------------------------------------------------------
struct FpRefArgs {
    const float *vol;
    const float *r_sino;
    float *w_sino;
    const float *ray_w;
    const float *sin_lut;
    const float *cos_lut;
    int n, n_dets, ang0, n_ang, dir;
    float axis, corr;
};

// Per-ray set-up of projector-parallel-joseph.cl:51-75 / :112-136: returns
// false for an inactive detector; else the start coordinate along the ray's
// interpolation axis (a double expression rounded to float, :73 / :134), the
// per-line step and the family (0 = FP_hor, 1 = FP_vert).
__device__ __forceinline__ bool fp_ray_setup(int s, int ang, int N, int D, float axis, const float *sin_lut,
                                             const float *cos_lut, int dir_in, float &pos, float &step, int &dir)
{
    const float required_width = axis * 2;
    const float diff = (float)D - required_width;
    if ((diff < 0 && (float)s < fabsf(diff)) || (diff > 0 && (float)s > required_width))
        return false;
    const float rot = diff / 2.0f;
    const float origin_shift = (float)N / 2.0f;
    const float st = sin_lut[ang], ct = cos_lut[ang];
    dir = dir_in >= 0 ? dir_in : (fabsf(st) <= fabsf(ct));
    const double t = ((0.5 + (double)rot) + (double)s) - (double)(0.5f * (float)D);
    if (dir == 0) {
        const float det_step = -1.0f / st;
        step = ct / st;
        pos = (float)(t * (double)det_step + (double)((-origin_shift) * step) + (double)(0.5f * (float)N));
    } else {
        const float det_step = 1.0f / ct;
        step = st / ct;
        pos = (float)(t * (double)det_step + (double)((-origin_shift) * step) + (double)(0.5f * (float)N));
    }
    return true;
}

// One block sum of :82-90: samples i in [b0, bend) of the ray, pos advanced
// by step per sample (the incremental float stepping of the reference).
// FP_hor walks column i linear in y; FP_vert walks row i linear in x.  Samples
// past the image edge read the zero border and do not change the sum.
// Samples are taken in batches of kFpBatch: the batch's coordinates follow
// the same sequential float additions, all its taps are loaded (clamped,
// always-valid addresses, zero where the reference reads the border), and
// only then are the samples added to the block sum in order -- the
// arithmetic and its order are the reference's, the loads overlap.
constexpr int kFpBatch = 8;

__device__ __forceinline__ float fp_block_sum(const float *img, int N, int dir, int b0, int bend, float &pos, float step)
{
    float inner = 0.0f;
    for (int i0 = b0; i0 < bend; i0 += kFpBatch) {
        float w[kFpBatch], va[kFpBatch], vb[kFpBatch];
        int c0[kFpBatch];
#pragma unroll
        for (int k = 0; k < kFpBatch; ++k) {
            const int i = min(i0 + k, bend - 1); // lanes past bend load a valid address, unused
            const float v = pos - 0.5f;
            const float fv = floorf(v);
            c0[k] = (int)fv;
            w[k] = v - fv;
            const int ca = min(max(c0[k], 0), N - 1), cb = min(max(c0[k] + 1, 0), N - 1);
            // FP_hor walks column i linear in y; FP_vert walks row i linear in x
            const size_t oa = dir == 0 ? (size_t)ca * N + i : (size_t)i * N + ca;
            const size_t ob = dir == 0 ? (size_t)cb * N + i : (size_t)i * N + cb;
            va[k] = img[oa];
            vb[k] = img[ob];
            if (i0 + k < bend)
                pos += step;
        }
        // An empty statement that takes the loaded registers: every load of the
        // batch is issued before the first one is waited for (otherwise the
        // compiler moves a load whose value is only used under the bounds test
        // into a branch and waits on it there).
#pragma unroll
        for (int k = 0; k < kFpBatch; ++k)
            asm volatile("" : "+v"(va[k]), "+v"(vb[k]));
#pragma unroll
        for (int k = 0; k < kFpBatch; ++k) {
            if (i0 + k < bend) {
                const float t0 = (c0[k] >= 0 && c0[k] < N) ? va[k] : 0.0f;
                const float t1 = (c0[k] + 1 >= 0 && c0[k] + 1 < N) ? vb[k] : 0.0f;
                const float omw = 1.0f - w[k];
                inner += omw * t0 + w[k] * t1;
            }
        }
    }
    return inner;
}

// Inactive detector (:63-66): the reference kernel returns and the (aliased)
// sinogram keeps r; the SIRT / SART form then multiplies by the ray weight.
__device__ __forceinline__ void fp_inactive(const FpRefArgs &p, size_t o)
{
    if (p.ray_w)
        p.w_sino[o] = p.r_sino[o] * p.ray_w[o];
    else if (p.w_sino != p.r_sino)
        p.w_sino[o] = p.r_sino[o];
}

__device__ __forceinline__ void fp_epilogue(const FpRefArgs &p, size_t o, float acc)
{
    float w = p.r_sino[o] + acc * p.corr; // :92-94
    if (p.ray_w)
        w = w * p.ray_w[o];
    p.w_sino[o] = w;
}

__global__ __launch_bounds__(256) void k_fp_ref(FpRefArgs p)
{
    const int s = blockIdx.x * 64 + threadIdx.x;
    const int k = blockIdx.y * 4 + threadIdx.y;
    if (s >= p.n_dets || k >= p.n_ang)
        return;
    const int ang = p.ang0 + k;
    const int N = p.n;
    const size_t o = (size_t)ang * p.n_dets + s;
    float pos, step;
    int dir;
    if (!fp_ray_setup(s, ang, N, p.n_dets, p.axis, p.sin_lut, p.cos_lut, p.dir, pos, step, dir)) {
        fp_inactive(p, o);
        return;
    }
    float acc = 0.0f;
    for (int b0 = 0; b0 < N; b0 += kBlockSamples)
        acc += fp_block_sum(p.vol, N, dir, b0, min(N, b0 + kBlockSamples), pos, step);
    fp_epilogue(p, o, acc);
}

// The same projection with each ray split over 16 threads: thread slot q
// takes blocks q, q + 16, ...; it reaches a block's start coordinate by
// replaying the reference's float additions (no memory traffic), so every
// sample sees the coordinate the sequential walk would see.  The block sums
// meet in LDS and are added in block order, as the reference adds them.
// Used where few rays are projected at once (kernel-level subsets of up to 4
// angles).
constexpr int kSplitRays = 16, kSplitSlots = 16, kMaxBlocks = 16384 / kBlockSamples;

__global__ __launch_bounds__(256) void k_fp_ref_split(FpRefArgs p)
{
    __shared__ float sums[kSplitRays][kMaxBlocks];
    const int r = threadIdx.x % kSplitRays, q = threadIdx.x / kSplitRays;
    const int s = blockIdx.x * kSplitRays + r;
    const int ang = p.ang0 + blockIdx.y;
    const int N = p.n;
    const int n_blocks = (N + kBlockSamples - 1) / kBlockSamples;
    float pos = 0.0f, step = 0.0f;
    int dir = 0;
    const bool live = s < p.n_dets &&
                      fp_ray_setup(s, ang, N, p.n_dets, p.axis, p.sin_lut, p.cos_lut, p.dir, pos, step, dir);
    if (live) {
        int at = 0; // blocks already stepped over (every block before the last is whole)
        for (int j = q; j < n_blocks; j += kSplitSlots) {
            for (; at < j; ++at) {
#pragma unroll
                for (int k = 0; k < kBlockSamples; ++k)
                    pos += step;
            }
            const int b0 = j * kBlockSamples;
            sums[r][j] = fp_block_sum(p.vol, N, dir, b0, min(N, b0 + kBlockSamples), pos, step);
            at = j + 1;
        }
    }
    __syncthreads();
    if (q != 0 || s >= p.n_dets)
        return;
    const size_t o = (size_t)ang * p.n_dets + s;
    if (!live) {
        fp_inactive(p, o);
        return;
    }
    float acc = 0.0f;
    for (int j = 0; j < n_blocks; ++j)
        acc += sums[r][j];
    fp_epilogue(p, o, acc);
}

// --------------------------------------------------------------------------
// The same projection with one wave per 64-sample block of 64 rays, from the
// image and its transpose.
// --------------------------------------------------------------------------
// A workgroup owns 64 detectors of one angle, a wave one of the rays' blocks
// (waves past 16 blocks take further ones): it replays the reference's float
// additions to the block's start, and its samples walk the lines of the image
// (FP_vert) or of the transposed image (FP_hor), so that the 64 rays' taps are
// neighbours on one line and the line's ends read as zero.  The block sums
// meet in LDS and are added in block order.  For images whose LDS-staged work
// table (k_fp_ref_tab) would leave most of the chip idle.
constexpr int kBlkWaves = 16;

// kFpBatch samples (or n of them) of a block from line l on, added in order.
template <int n> __device__ __forceinline__ float fp_lines(const float *img, int N, int l, float &pos, float step, float inner)
{
    float w[n], va[n], vb[n];
#pragma unroll
    for (int k = 0; k < n; ++k) {
        const float v = pos - 0.5f;
        const float fv = floorf(v);
        const int c0 = (int)fv;
        w[k] = v - fv;
        const __amdgpu_buffer_rsrc_t r = row_rsrc(img + (size_t)(l + k) * N, (uint32_t)N);
        va[k] = row_load(r, c0);
        vb[k] = row_load(r, opaque(c0 + 1));
        pos += step;
    }
#pragma unroll
    for (int k = 0; k < n; ++k) {
        const float omw = 1.0f - w[k];
        inner += omw * va[k] + w[k] * vb[k];
    }
    return inner;
}

__global__ __launch_bounds__(64 * kBlkWaves) void k_fp_blocks(FpRefArgs p, const float *__restrict__ vol_t)
{
    __shared__ float sums[kBlkWaves][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_waves = blockDim.x >> 6;
    const int s = blockIdx.x * 64 + lane, ang = p.ang0 + blockIdx.y;
    const int N = p.n, n_blocks = (N + kBlockSamples - 1) / kBlockSamples;
    const size_t o = (size_t)ang * p.n_dets + s;
    float pos = 0.0f, step = 0.0f;
    int dir = 0;
    const bool live = s < p.n_dets &&
                      fp_ray_setup(s, ang, N, p.n_dets, p.axis, p.sin_lut, p.cos_lut, p.dir, pos, step, dir);
    const bool vertical = p.dir >= 0 ? p.dir != 0 : fabsf(p.sin_lut[ang]) <= fabsf(p.cos_lut[ang]); // uniform
    const float *img = vertical ? p.vol : vol_t;
    float acc = 0.0f;
    int at = 0; // blocks already stepped over
    for (int j0 = 0; j0 < n_blocks; j0 += n_waves) {
        const int j = j0 + wave;
        if (j < n_blocks) {
            for (; at < j; ++at) {
#pragma unroll
                for (int k = 0; k < kBlockSamples; ++k)
                    pos += step;
            }
            const int bend = min(N, (j + 1) * kBlockSamples);
            float inner = 0.0f;
            int l = j * kBlockSamples;
            for (; l + kFpBatch <= bend; l += kFpBatch)
                inner = fp_lines<kFpBatch>(img, N, l, pos, step, inner);
            for (; l < bend; ++l)
                inner = fp_lines<1>(img, N, l, pos, step, inner);
            at = j + 1;
            sums[wave][lane] = inner;
        }
        __syncthreads();
        if (wave == 0)
            for (int k = 0; k < n_waves && j0 + k < n_blocks; ++k) // :89
                acc += sums[k][lane];
        __syncthreads();
    }
    if (wave != 0 || s >= p.n_dets)
        return;
    if (live)
        fp_epilogue(p, o, acc);
    else
        fp_inactive(p, o);
}

// out = in^T of an n x n image, 64 x 64 tiles through LDS.
__global__ __launch_bounds__(256) void k_transpose(const float *__restrict__ in, float *__restrict__ out, int n)
{
    __shared__ float t[64][65];
    const int lx = threadIdx.x & 63, ly = threadIdx.x >> 6;
    const int x = blockIdx.x * 64 + lx, y0 = blockIdx.y * 64;
#pragma unroll
    for (int k = 0; k < 64; k += 4)
        if (x < n && y0 + ly + k < n)
            t[ly + k][lx] = in[(size_t)(y0 + ly + k) * n + x];
    __syncthreads();
    const int xo = y0 + lx, yo = blockIdx.x * 64;
#pragma unroll
    for (int k = 0; k < 64; k += 4)
        if (xo < n && yo + ly + k < n)
            out[(size_t)(yo + ly + k) * n + xo] = t[lx][ly + k];
}

// --------------------------------------------------------------------------
// Backprojection, R pixels per thread, per-run accumulation.
// --------------------------------------------------------------------------
struct BpRefArgs {
    const float *r_vol;
    float *w_vol;
    const float *sino;
    const float *pix_w;
    const float *sin_lut;
    const float *cos_lut;
    int n, n_dets, n_angles, posc;
    float axis, relax;
    uirk_runs runs;
};

// The taps are gathered straight from the sinogram rows: neighbouring pixels
// read neighbouring bins, so a wave's 64 taps lie in three cache lines that the
// workgroup's other rows read too, and nothing is staged or waited for at a
// barrier.  A thread keeps R pixels (rows) and takes kBpU angles at a time, all
// their taps in flight before the first is used.  What bounds it is the VALU:
// about 13 operations a sample, three of them at half rate.  Against LDS-staged
// 64 x 64 tiles (a wave a SIMD at 1024 x 1024, 16 workgroups at 256 x 256) it
// took 197 us instead of 425 at 1024 / 720 / 1448 and 15 instead of 109 at
// 256 / 180 / 367.
constexpr int kBpU = 8;

// floor(x) converted to int in one instruction (no memory access).
__device__ __forceinline__ int cvt_flr(float x)
{
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// CLAMP 2: any axis and any LUT.  1: 0.5 <= edge0 <= edge1 <= n_dets - 0.5 (an
// axis with active detectors), so that the clamp is one median and every lower
// tap lies in the row.  0: no pixel reaches an edge either, no clamp.  3: as 1
// for any LUT: a NaN coordinate stays one, which the median would drop.
template <int R, int CLAMP> __global__ __launch_bounds__(256) void k_bp_gather(BpRefArgs p)
{
    const int N = p.n, D = p.n_dets;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int px = blockIdx.x * 64 + lane;
    const int py0 = (blockIdx.y * 4 + wave) * R;

    // projector-parallel-joseph.cl:174-190 (detector quantities use n_dets)
    const float required_width = p.axis * 2;
    const float diff = (float)D - required_width;
    const float half_active = diff < 0 ? (float)D - p.axis : p.axis;
    const float edge0 = p.axis - half_active + 0.5f;
    const float edge1 = p.axis + half_active - 0.5f;
    const float rot = diff / 2.0f;
    const float det_shift = (float)D / 2.0f;
    const float origin_shift = (float)N / 2.0f;
    const float shift = det_shift - rot;
    const float fX = (float)px + 0.5f - origin_shift;
    float fY[R], out[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
        fY[q] = (float)(py0 + q) + 0.5f - origin_shift;
        out[q] = (!p.pix_w && px < N && py0 + q < N) ? p.r_vol[(size_t)(py0 + q) * N + px] : 0.0f;
    }
    for (int r = 0; r < p.runs.count; ++r) {
        const int off = (int)p.runs.offset[r], cnt = (int)p.runs.n[r];
        float value[R];
#pragma unroll
        for (int q = 0; q < R; ++q)
            value[q] = 0.0f;
        // :196-214, kBpU angles at a time: their taps are all in flight before
        // the first is used
        auto angles = [&](int k, auto n_) {
            constexpr int n = decltype(n_)::value;
            float t0[n][R], t1[n][R], a[n][R];
#pragma unroll
            for (int e = 0; e < n; ++e) {
                const int ang = off + k + e;
                const float st = p.sin_lut[ang], ct = p.cos_lut[ang];
                const float *row = p.sino + (size_t)ang * D;
                const __amdgpu_buffer_rsrc_t r0 = row_rsrc(row, (uint32_t)D), r1 = row_rsrc(row + 1, (uint32_t)D - 1u);
                const float fXc = fX * ct;
#pragma unroll
                for (int q = 0; q < R; ++q) {
                    float u = fXc - fY[q] * st + shift;
                    if (CLAMP == 1) {
                        u = __builtin_amdgcn_fmed3f(u, edge0, edge1);
                    } else if (CLAMP == 3) {
                        u = u != u ? u : __builtin_amdgcn_fmed3f(u, edge0, edge1);
                    } else if (CLAMP == 2) {
                        if (u > edge1)
                            u = edge1;
                        else if (u < edge0)
                            u = edge0;
                    }
                    const float w = u - 0.5f;
                    const int i0 = cvt_flr(w);
                    a[e][q] = CLAMP != 2 ? __builtin_amdgcn_fractf(w) : w - floorf(w); // the same for w >= 0
                    t0[e][q] = row_load(r0, i0);
                    t1[e][q] = CLAMP != 2 ? row_load(r1, i0) : row_load(r0, opaque(i0 + 1));
                }
            }
#pragma unroll
            for (int e = 0; e < n; ++e) {
#pragma unroll
                for (int q = 0; q < R; ++q) {
                    const float oma = 1.0f - a[e][q];
                    value[q] += oma * t0[e][q] + a[e][q] * t1[e][q];
                }
            }
        };
        int k = 0;
        for (; k + kBpU <= cnt; k += kBpU)
            angles(k, std::integral_constant<int, kBpU>{});
        for (; k < cnt; ++k)
            angles(k, std::integral_constant<int, 1>{});
#pragma unroll
        for (int q = 0; q < R; ++q)
            out[q] = out[q] + p.relax * value[q]; // :216
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
        if (px >= N || py0 + q >= N)
            continue;
        const size_t o = (size_t)(py0 + q) * N + px;
        float v = out[q];
        if (p.pix_w) {
            v = v * p.pix_w[o];
            v = v + p.r_vol[o];
            if (p.posc)
                v = v > 0 ? v : 0.0f;
        }
        p.w_vol[o] = v;
    }
}

template <int R> void launch_bp_gather(const BpRefArgs &a, bool unit_lut, hipStream_t st)
{
    const float half = (float)a.n_dets - a.axis * 2 < 0 ? (float)a.n_dets - a.axis : a.axis;
    const float edge0 = a.axis - half + 0.5f, edge1 = a.axis + half - 0.5f;
    const bool window = edge0 >= 0.5f && edge0 <= edge1 && edge1 <= (float)a.n_dets - 0.5f;
    // u - shift is at most the distance of a corner pixel's centre from the
    // image centre, plus the rounding of three float operations
    const float rot = ((float)a.n_dets - a.axis * 2) / 2.0f, shift = (float)a.n_dets / 2.0f - rot;
    const double reach = 0.7071067811865476 * (a.n - 1) * (1.0 + 1e-5) + 1e-3;
    const bool inside = window && shift - reach > edge0 && shift + reach < edge1;
    const dim3 grid((a.n + 63) / 64, (a.n + 4 * R - 1) / (4 * R));
    // a caller's LUT may hold anything, as pairs longer than 1, which reach past
    // the corners' distance
    if (!unit_lut && window)
        hipLaunchKernelGGL((k_bp_gather<R, 3>), grid, dim3(256), 0, st, a);
    else if (inside)
        hipLaunchKernelGGL((k_bp_gather<R, 0>), grid, dim3(256), 0, st, a);
    else if (window)
        hipLaunchKernelGGL((k_bp_gather<R, 1>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((k_bp_gather<R, 2>), grid, dim3(256), 0, st, a);
}

// --------------------------------------------------------------------------
// SART: the BP of one angle and the FP of the next in one launch
// --------------------------------------------------------------------------
// SART alternates the FP of one angle and the BP of its weighted residual into
// the image, so each launch waits for the one before and is short: what bounds
// a sweep is the chain of launches and, within each, of dependent loads and of
// instruction fetches (a launch starts with cold instruction caches, and a
// kilobyte of straight code costs about 0.6 us).  So one launch here applies
// the BP of angle bp_ang to the image, from x_in to the other buffer x_out, and
// takes the block sums of the FP of angle fp_ang of that updated image, which
// it forms on the fly from x_in, and many short waves of little code do it.
// Two kinds of workgroups share the launch and nothing else:
//   FP: 64 detectors (lanes) x one 64-sample block, kSeg samples to each wave.
//       A wave replays at most 56 additions of the step from the block's start,
//       its taps are neighbours on a line, and every tap gets its BP update by
//       the operations the BP workgroups use; the samples meet in LDS and one
//       wave adds them in order (:82-90).  The block sum goes to
//       part_out[block][detector].
//   BP: a tile of 64 x 64 pixels, kSeg per thread, x_out = x_in + relax BP (:196-216).
// Both first form the residuals of the bins they need in LDS: the previous
// launch's block sums added in block order, then (b + corr sum) R (:89-94).
// The image is held transposed while the angles are horizontal (FP_hor), so
// that rays always walk its rows.  Every operation and its order is the
// reference's: bit-identical to k_fp_ref and k_bp_gather angle by angle.
// A separate FP and BP per angle, the FP gathering along columns for half of
// the angles, took 11.8 + 7.1 us an angle at 1024 x 1024 / 1448 bins, this
// takes 7.3 (of them 1.6 for an empty launch, 1.8 to fetch the image, 2.4 for
// the updates); 5.1 + 2.4 and 4.5 at 128 x 128.
// Bins a workgroup touches: an FP's 64 rays cover at most 63 sqrt(2) + 63 = 153
// positions of 64 lines, and its region takes a margin on each side that covers
// the drift of the float stepping (N additions, each off by at most N 2^-24
// inside the image), 66 positions for the largest image of 4 GiB: 285 positions
// x 64 lines are 292 bins apart.  A BP tile needs 90.
constexpr int kSartBins = 320;
constexpr int kSeg = 8; // samples or pixels per thread (4 and 16 are slower by up to 0.3 and 1.3 us)
constexpr int kSartThreads = 4096 / kSeg, kSartWaves = kSartThreads / 64;

struct SartStepArgs {
    const float *x_in;
    float *x_out;
    const float *b, *ray_w;  // rows of angle bp_ang
    const float *starts;     // of angle fp_ang, [block][detector], or NULL: replay the stepping
    const float *part_in;
    float *part_out;         // [block][detector]
    int n, n_dets;
    int bp;                  // apply the BP
    int n_fp, n_bp;          // FP and BP workgroups per band of 64 lines
    int n_xcd;
    float axis, corr, relax;
    float kp, kl;            // BP: u = (fP kp - fL kl) + shift at position P of line L
    float det_step, step;    // FP
};

// The coordinate at the start of every 64-sample block of every ray of angles
// [0, n_angles), [angle][block][detector], by the reference's sequential walk
// (:82-90), which does not depend on the image; inactive rays get 0.
__global__ __launch_bounds__(256) void k_fp_block_starts(FpRefArgs p, float *__restrict__ starts)
{
    const int s = blockIdx.x * 256 + threadIdx.x;
    const int ang = p.ang0 + blockIdx.y;
    if (s >= p.n_dets)
        return;
    const int N = p.n, n_blocks = (N + kBlockSamples - 1) / kBlockSamples;
    float pos = 0.0f, step = 0.0f;
    int dir = 0;
    float *out = starts + (size_t)ang * n_blocks * p.n_dets + s;
    const bool live = fp_ray_setup(s, ang, N, p.n_dets, p.axis, p.sin_lut, p.cos_lut, p.dir, pos, step, dir);
    for (int j = 0; j < n_blocks; ++j) {
        out[(size_t)j * p.n_dets] = live ? pos : 0.0f;
#pragma unroll
        for (int k = 0; k < kBlockSamples; ++k)
            pos += step;
    }
}

// WINDOW: edge0 <= edge1 (an axis with active detectors): the clamp is a median.
// TURN: the BP writes its tiles transposed, through LDS, for an FP of the other
// direction in the next launch.  A transpose between the launches reads and
// writes the image once more and waits for both: 14 angles 1.94 rad apart, the
// direction changing 10 times, took 10.2 us an angle at 128 x 128 and 32.6 at
// 2048 x 2048 with it, 6.3 and 26.5 without.
template <bool WINDOW, bool TURN> __global__ __launch_bounds__(kSartThreads) void k_sart_ref_step(SartStepArgs p)
{
    __shared__ float row[kSartBins];
    __shared__ float samples[kBlockSamples][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int N = p.n, D = p.n_dets;
    const int n_blocks = (N + kBlockSamples - 1) / kBlockSamples;
    // a band's workgroups, FP and BP, run on one XCD (workgroup g on XCD g mod
    // n_xcd), in this launch and the next: its L2 holds the band's pixels
    const uint32_t turn = blockIdx.x / (uint32_t)p.n_xcd, per_band = (uint32_t)(p.n_fp + p.n_bp);
    const int band = (int)((blockIdx.x - turn * (uint32_t)p.n_xcd) + (turn / per_band) * (uint32_t)p.n_xcd);
    const int item = (int)(turn % per_band);
    if (band * 64 >= p.n)
        return;
    const bool fp = item < p.n_fp; // uniform
    const int at = fp ? item : item - p.n_fp;

    // projector-parallel-joseph.cl:174-190 (detector quantities use n_dets)
    const float required_width = p.axis * 2;
    const float diff = (float)D - required_width;
    const float half_active = diff < 0 ? (float)D - p.axis : p.axis;
    const float edge0 = p.axis - half_active + 0.5f;
    const float edge1 = p.axis + half_active - 0.5f;
    const float rot = diff / 2.0f;
    const float origin_shift = (float)N / 2.0f;
    const float shift = (float)D / 2.0f - rot;

    // this workgroup's lines [l0, l1) and positions [c_lo, c_hi] of the image
    const int l0 = band * 64, l1 = min(N, l0 + 64);
    float c_lo = (float)(at * 64), c_hi = fminf(c_lo + 63.0f, (float)(N - 1));

    // the image values first: their loads overlap the residuals' below
    float va[kSeg], vb[kSeg], fv[kSeg], w[kSeg];
    const int s = at * 64 + lane;                                    // FP: this lane's ray; BP: its position
    const int i0 = fp ? l0 + kSeg * wave : l0 + wave;         // this wave's first line
    bool live = false;
    if (fp) {
        live = s < D && !((diff < 0 && (float)s < fabsf(diff)) || (diff > 0 && (float)s > required_width)); // :63-66
        float pos = 0.0f;
        const float step = p.step;
        if (p.starts) {
            if (live)
                pos = p.starts[(size_t)band * D + s];
        } else {
            const double t = ((0.5 + (double)rot) + (double)s) - (double)(0.5f * (float)D); // :73, :134
            pos = (float)(t * (double)p.det_step + (double)((-origin_shift) * step) + (double)(0.5f * (float)N));
#pragma unroll 8
            for (int k = 0; k < l0; ++k)
                pos += step;
        }
        // the region: the positions of the first and last ray on the first and
        // last line, and a margin
        const float pa = ((float)(at * 64) + 0.5f - p.axis) * p.det_step + (0.5f * (float)N + ((float)l0 - 0.5f * (float)N) * step);
        const float pb = pa + 63.0f * p.det_step, dl = 63.0f * step;
        const float margin = 2.0f + ceilf((float)N * (float)N * 0x1p-24f);
        c_lo = fminf(fmaxf(floorf(fminf(pa, pb) + fminf(dl, 0.0f)) - margin, 0.0f), (float)(N - 1));
        c_hi = fmaxf(fminf(floorf(fmaxf(pa, pb) + fmaxf(dl, 0.0f)) + margin, (float)(N - 1)), c_lo);
#pragma unroll 1
        for (int r = 0; r < wave; ++r) {
#pragma unroll
            for (int k = 0; k < kSeg; ++k)
                pos += step;
        }
#pragma unroll
        for (int k = 0; k < kSeg; ++k) {
            const float v = pos - 0.5f;
            fv[k] = floorf(v);
            w[k] = v - fv[k];
            const int line = i0 + k, c = (int)fv[k];
            const __amdgpu_buffer_rsrc_t r = row_rsrc(p.x_in + (size_t)line * N, line < N ? (uint32_t)N : 0u);
            va[k] = row_load(r, c);
            vb[k] = row_load(r, opaque(c + 1));
            pos += step;
        }
    } else {
#pragma unroll
        for (int k = 0; k < kSeg; ++k) {
            const int line = i0 + kSartWaves * k;
            va[k] = row_load(row_rsrc(p.x_in + (size_t)line * N, line < N ? (uint32_t)N : 0u), s);
        }
    }

    // residuals of the bins under the region
    int umin = 0;
    if (p.bp) {
        const float cx0 = (c_lo + 0.5f - origin_shift) * p.kp, cx1 = (c_hi + 0.5f - origin_shift) * p.kp;
        const float cy0 = ((float)l0 + 0.5f - origin_shift) * p.kl, cy1 = ((float)(l1 - 1) + 0.5f - origin_shift) * p.kl;
        float umn = (fminf(cx0, cx1) - fmaxf(cy0, cy1)) + shift, umx = (fmaxf(cx0, cx1) - fminf(cy0, cy1)) + shift;
        const float e_lo = fminf(edge0, edge1), e_hi = fmaxf(edge0, edge1);
        umn = fminf(fmaxf(umn, e_lo), e_hi);
        umx = WINDOW ? fminf(fmaxf(umx, e_lo), e_hi) : e_hi;
        if (!WINDOW)
            umn = e_lo;
        umin = (int)floorf(umn - 0.5f) - 2;
        const int width = min((int)(umx - umn) + 6, kSartBins);
        for (int e0 = threadIdx.x; e0 < width; e0 += kSartThreads) {
            const int bin = umin + e0;
            float r = 0.0f;
            if (bin >= 0 && bin < D) {
                r = p.b[bin];
                const float rw = p.ray_w[bin];
                float acc = 0.0f;
#pragma unroll 1
                for (int j = 0; j < n_blocks; j += 8) {
                    float v[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        v[e] = j + e < n_blocks ? p.part_in[(size_t)(j + e) * D + bin] : 0.0f;
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        acc = acc + v[e]; // :89 (the sum is never -0: adding 0 past the last block keeps it)
                }
                if (!((diff < 0 && (float)bin < fabsf(diff)) || (diff > 0 && (float)bin > required_width)))
                    r = r + acc * p.corr; // :92-94
                r = r * rw;
            }
            row[e0] = r;
        }
        __syncthreads();
    }
    auto update = [&](float x, float fP, float lineterm) { // :196-216
        float u = (fP * p.kp - lineterm) + shift;
        if (WINDOW) {
            u = __builtin_amdgcn_fmed3f(u, edge0, edge1);
        } else {
            if (u > edge1)
                u = edge1;
            else if (u < edge0)
                u = edge0;
        }
        const float v = u - 0.5f;
        const float f = floorf(v);
        // a tap outside the region is not used: any entry of the row
        const int b0 = (int)min((uint32_t)((int)f - umin), (uint32_t)(kSartBins - 2));
        const float a = v - f;
        const float oma = 1.0f - a;
        // (the reference adds the sample to 0 first, which only turns a -0 into
        // +0: no difference to x, which is never -0)
        return x + p.relax * (oma * row[b0] + a * row[b0 + 1]);
    };

    if (!fp) {
        const float fP = (float)s + 0.5f - origin_shift;
#pragma unroll
        for (int k = 0; k < kSeg; ++k) {
            const int line = i0 + kSartWaves * k;
            if (TURN) { // column lane ^ row: both ways without bank conflicts
                const float v = update(va[k], fP, ((float)line + 0.5f - origin_shift) * p.kl);
                samples[line - l0][lane ^ (line - l0)] = v;
            } else if (s < N && line < N)
                p.x_out[(size_t)line * N + s] = update(va[k], fP, ((float)line + 0.5f - origin_shift) * p.kl);
        }
        if (TURN) {
            __syncthreads();
#pragma unroll
            for (int k = 0; k < kSeg; ++k) {
                const int r = wave + kSartWaves * k, P = at * 64 + r;
                if (P < N && l0 + lane < N)
                    p.x_out[(size_t)P * N + l0 + lane] = samples[lane][r ^ lane];
            }
        }
        return;
    }

#pragma unroll
    for (int k = 0; k < kSeg; ++k) {
        float t0 = va[k], t1 = vb[k];
        if (p.bp) {
            const float lt = ((float)(i0 + k) + 0.5f - origin_shift) * p.kl;
            const float fP = fv[k] + (0.5f - origin_shift); // half-integers: exact in any order
            const float ta = update(t0, fP, lt);
            const float tb = update(t1, fP + 1.0f, lt);
            t0 = fv[k] >= 0.0f && fv[k] < (float)N ? ta : 0.0f;
            t1 = fv[k] >= -1.0f && fv[k] < (float)(N - 1) ? tb : 0.0f;
        }
        const float omw = 1.0f - w[k];
        samples[kSeg * wave + k][lane] = omw * t0 + w[k] * t1;
    }
    __syncthreads();
    if (wave != 0)
        return;
    float run = 0.0f;
    int k = 0;
    for (; k + 8 <= l1 - l0; k += 8) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            run = run + samples[k + e][lane];
    }
    for (; k < l1 - l0; ++k)
        run = run + samples[k][lane];
    if (s < D)
        p.part_out[(size_t)band * D + s] = live ? run : 0.0f;
}

// --------------------------------------------------------------------------
// Elementwise
// --------------------------------------------------------------------------
inline unsigned grid1d(size_t n, unsigned block = 256)
{
    size_t g = (n + block - 1) / block;
    if (g > 65536u * 16u)
        g = 65536u * 16u;
    return (unsigned)(g ? g : 1);
}

__global__ void k_set(float *out, size_t n, float v)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = v;
}

__global__ void k_copy(float *dst, const float *src, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

__global__ void k_inv(const float *in, float *out, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float v = in[i];
        out[i] = (v != 0) ? 1.0f / v : 0.0f; // ufo-ir-basic-ops.cl:34
    }
}

// Ray weights with a floor: rays whose FP(1) is below vmin are treated as
// missing the image (weight 0).
__global__ void k_inv_min(const float *in, float *out, size_t n, float vmin)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float v = in[i];
        out[i] = (v != 0 && v >= vmin) ? 1.0f / v : 0.0f;
    }
}

__global__ void k_binary(int op, const float *a, const float *b, float m, float *out, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float x = a[i], y = b[i];
        float r;
        switch (op) {
        case UIRK_MUL: r = x * y; break;
        case UIRK_ADD: r = x + y; break;
        case UIRK_SUB: r = x - y; break;
        case UIRK_SUB_SCALED: r = x - m * y; break;
        case UIRK_ADD_SCALED: r = x + m * y; break;
        case UIRK_MAX: r = fmaxf(x, y); break;
        default: r = x / y; break;
        }
        out[i] = r;
    }
}

__global__ void k_unary(int op, const float *in, float *out, size_t n, float m)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float x = in[i];
        float r;
        switch (op) {
        case UIRK_POSC: r = x > 0 ? x : 0.0f; break;
        case UIRK_SQRT: r = sqrtf(x); break;
        default: r = x * m; break;
        }
        out[i] = r;
    }
}

__global__ void k_mul_rows(const float *a, const float *b, float *out, uint32_t width, uint32_t offset, uint32_t rows)
{
    const size_t total = (size_t)width * rows;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t idx = (size_t)offset * width + i;
        out[idx] = a[idx] * b[idx];
    }
}

// --------------------------------------------------------------------------
// Reductions (deterministic: fixed grid, fixed tree order)
// --------------------------------------------------------------------------
constexpr int kRedBlock = 256;
constexpr unsigned kRedMaxBlocks = 1024;

inline unsigned red_blocks(size_t n)
{
    size_t g = (n + kRedBlock * 4 - 1) / (kRedBlock * 4);
    if (g > kRedMaxBlocks)
        g = kRedMaxBlocks;
    return (unsigned)(g ? g : 1);
}

template <typename T>
__device__ T block_sum(T v, T *sh)
{
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int w = kRedBlock / 2; w > 0; w >>= 1) {
        if (t < w)
            sh[t] = sh[t] + sh[t + w];
        __syncthreads();
    }
    return sh[0];
}

template <int KIND> // 0: sum |a|, 1: sum a*b
__global__ __launch_bounds__(kRedBlock) void k_red_f64(const float *a, const float *b, size_t n, double *ws)
{
    __shared__ double sh[kRedBlock];
    double acc = 0.0;
    for (size_t i = blockIdx.x * (size_t)kRedBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kRedBlock) {
        if (KIND == 0)
            acc += fabs((double)a[i]);
        else
            acc += (double)a[i] * (double)b[i];
    }
    const double s = block_sum(acc, sh);
    if (threadIdx.x == 0)
        ws[blockIdx.x] = s;
}

__global__ __launch_bounds__(kRedBlock) void k_red_final_f64(const double *ws, unsigned nb, double *result)
{
    __shared__ double sh[kRedBlock];
    double acc = 0.0;
    for (unsigned i = threadIdx.x; i < nb; i += kRedBlock)
        acc += ws[i];
    const double s = block_sum(acc, sh);
    if (threadIdx.x == 0)
        *result = s;
}

// Sum of lds[0, n) added to acc one after another in index order, as the
// reference's sequential float loop adds them (n a multiple of 4 is read in
// 16-byte pieces, the rest one by one).
__device__ __forceinline__ float add_in_order(const float *lds, uint32_t n, float acc)
{
    uint32_t k = 0;
    for (; k + 16 <= n; k += 16) {
        float4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            v[j] = *(const float4 *)(lds + k + 4 * j);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc += v[j].x;
            acc += v[j].y;
            acc += v[j].z;
            acc += v[j].w;
        }
    }
    for (; k < n; ++k)
        acc += lds[k];
    return acc;
}

// ufo-ir-basic-ops-processor.c:181-193: part p sums a[p*i] * b[p*i] for
// i < part_len in float, in order.  One wave per part: its lanes load and
// multiply kDotChunk elements at a time (all loads in flight, those of the next
// chunk issued before the current one is summed), and lane 0 adds the products
// in order from LDS.  What remains serial is the additions; a thread per part
// that also loaded serially was bound by the latency of its strided loads: a
// 256 x 256 dot took 79 us in its two kernels, this takes about 10.
constexpr int kDotLane = 8;              // elements per lane and chunk
constexpr int kDotChunk = 64 * kDotLane;
constexpr int kDotParts = 4;             // parts (waves) per workgroup

__global__ __launch_bounds__(64 * kDotParts) void k_dot_compat_parts(const float *__restrict__ a,
                                                                     const float *__restrict__ b, uint32_t parts,
                                                                     uint32_t part_len, float *__restrict__ ws)
{
    __shared__ __align__(16) float prod[kDotParts][kDotChunk];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t p = blockIdx.x * kDotParts + wave;
    const uint32_t len = p < parts ? part_len : 0;
    float va[kDotLane], vb[kDotLane];
    auto load = [&](uint32_t i0) {
#pragma unroll
        for (int k = 0; k < kDotLane; ++k) {
            const uint32_t i = i0 + lane + 64u * k;
            const size_t idx = i < len ? (size_t)p * i : 0; // past the end: a valid address, unused
            va[k] = a[idx];
            vb[k] = b[idx];
        }
    };
    float part = 0.0f;
    if (part_len)
        load(0);
    for (uint32_t i0 = 0; i0 < part_len; i0 += kDotChunk) { // same trip count for every wave
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kDotLane; ++k)
            prod[wave][lane + 64 * k] = va[k] * vb[k];
        __syncthreads();
        if (i0 + kDotChunk < part_len)
            load(i0 + kDotChunk);
        if (lane == 0 && i0 < len)
            part = add_in_order(prod[wave], len - i0 < kDotChunk ? len - i0 : kDotChunk, part);
    }
    if (lane == 0 && p < parts)
        ws[p] = part;
}

// The parts added in order: one workgroup stages them through LDS, its first
// lane adds.
__global__ __launch_bounds__(256) void k_dot_compat_final(const float *__restrict__ ws, uint32_t parts,
                                                          float *__restrict__ result)
{
    constexpr uint32_t kStage = 1024;
    __shared__ __align__(16) float buf[kStage];
    float norm = 0.0f;
    for (uint32_t p0 = 0; p0 < parts; p0 += kStage) {
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < kStage && p0 + k < parts; k += 256)
            buf[k] = ws[p0 + k];
        __syncthreads();
        if (threadIdx.x == 0)
            norm = add_in_order(buf, parts - p0 < kStage ? parts - p0 : kStage, norm);
    }
    if (threadIdx.x == 0)
        *result = norm;
}

void launch_dot_compat(const float *a, const float *b, uint32_t parts, uint32_t part_len, float *ws, float *result,
                       hipStream_t st)
{
    hipLaunchKernelGGL(k_dot_compat_parts, dim3((parts + kDotParts - 1) / kDotParts), dim3(64 * kDotParts), 0, st, a,
                       b, parts, part_len, ws);
    hipLaunchKernelGGL(k_dot_compat_final, dim3(1), dim3(256), 0, st, ws, parts, result);
}

__global__ __launch_bounds__(kRedBlock) void k_minmax(const float *v, size_t n, float *ws)
{
    __shared__ float smx[kRedBlock], smn[kRedBlock];
    float mx = -3.40282347e+38f, mn = 3.40282347e+38f;
    for (size_t i = blockIdx.x * (size_t)kRedBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kRedBlock) {
        mx = fmaxf(v[i], mx);
        mn = fminf(v[i], mn);
    }
    const int t = threadIdx.x;
    smx[t] = mx;
    smn[t] = mn;
    __syncthreads();
    for (int w = kRedBlock / 2; w > 0; w >>= 1) {
        if (t < w) {
            smx[t] = fmaxf(smx[t], smx[t + w]);
            smn[t] = fminf(smn[t], smn[t + w]);
        }
        __syncthreads();
    }
    if (t == 0) {
        ws[2 * blockIdx.x] = smn[0];
        ws[2 * blockIdx.x + 1] = smx[0];
    }
}

__global__ void k_minmax_final(const float *ws, unsigned nb, float *minmax)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        float mn = 3.40282347e+38f, mx = -3.40282347e+38f;
        for (unsigned i = 0; i < nb; ++i) {
            mn = fminf(ws[2 * i], mn);
            mx = fmaxf(ws[2 * i + 1], mx);
        }
        minmax[0] = mn;
        minmax[1] = mx;
    }
}

// ufo-ir-basic-ops-processor.c:362-366
__global__ void k_normalize_apply(float *v, size_t n, const float *minmax)
{
    const float mn = minmax[0], mx = minmax[1];
    const float delta = 1 / (mx - mn);
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        v[i] = delta * v[i] - mn * delta;
}

// --------------------------------------------------------------------------
// Finite differences and TV gradient
// --------------------------------------------------------------------------
__global__ void k_diff(int kind, const float *in, float *out, int w, int h)
{
    const int x = blockIdx.x * 64 + threadIdx.x;
    const int y = blockIdx.y * 4 + threadIdx.y;
    if (x >= w || y >= h)
        return;
    const int idx = y * w + x;
    const int last = w * h;
    float r;
    switch (kind) {
    case UIRK_DX: r = in[idx] - in[idx - 1 + (x == 0 ? w : 0)]; break;            // Dx :1-11
    case UIRK_DXT: r = in[idx] - in[idx + 1 - (x == w - 1 ? w : 0)]; break;       // Dxt :13-24
    case UIRK_DY: r = in[idx] - in[idx - w + (y == 0 ? last : 0)]; break;         // Dy :26-37
    default: r = in[idx] - in[idx + w - (y == h - 1 ? last : 0)]; break;          // Dyt :39-51
    }
    out[idx] = r;
}

__device__ inline float nb_read(const float *img, int w, int h, int x, int y)
{
    return (x >= 0 && x < w && y >= 0 && y < h) ? img[(size_t)y * w + x] : 0.0f;
}

// ufo-math-tvstd-method.cl:5-57
__global__ void k_l1_grad(const float *in, float *out, int w, int h)
{
    const int x = blockIdx.x * 64 + threadIdx.x;
    const int y = blockIdx.y * 4 + threadIdx.y;
    if (x >= w || y >= h)
        return;
    const float eps = 0.001f;
    const float f3 = nb_read(in, w, h, x, y);
    const float f1 = nb_read(in, w, h, x, y - 1);
    const float f0 = nb_read(in, w, h, x - 1, y - 1);
    const float f2 = nb_read(in, w, h, x - 1, y);
    const float f4 = nb_read(in, w, h, x + 1, y);
    const float f6 = nb_read(in, w, h, x + 1, y + 1);
    const float f5 = nb_read(in, w, h, x, y + 1);
    const float df = (2.0f * f3 - f2 - f5) / sqrtf(eps + (f3 - f2) * (f3 - f2) + (f3 - f5) * (f3 - f5))
                   - (f4 - f3) / sqrtf(eps + (f4 - f3) * (f4 - f3) + (f4 - f6) * (f4 - f6))
                   - (f1 - f3) / sqrtf(eps + (f1 - f3) * (f1 - f3) + (f1 - f0) * (f1 - f0));
    out[(size_t)y * w + x] = df;
}

} // namespace

// ==========================================================================
// Launchers (C ABI, see uir_device.h)
// ==========================================================================
extern "C" {

int uirk_fp_ref(const float *vol, const float *r_sino, float *w_sino, const float *ray_w,
                const float *sin_lut, const float *cos_lut, int n, int n_dets, float axis,
                float corr, int ang0, int n_ang, int dir, void *stream)
{
    if (n_ang <= 0 || n_dets <= 0)
        return 0;
    FpRefArgs a{vol, r_sino, w_sino, ray_w, sin_lut, cos_lut, n, n_dets, ang0, n_ang, dir, axis, corr};
    dim3 block(64, 4), grid((n_dets + 63) / 64, (n_ang + 3) / 4);
    hipLaunchKernelGGL(k_fp_ref, grid, block, 0, (hipStream_t)stream, a);
    return (int)hipGetLastError();
}

int uirk_fp_ref_split(const float *vol, const float *r_sino, float *w_sino, const float *ray_w,
                      const float *sin_lut, const float *cos_lut, int n, int n_dets, float axis,
                      float corr, int ang0, int n_ang, int dir, void *stream)
{
    if (n_ang <= 0 || n_dets <= 0)
        return 0;
    if (n > 16384)
        return (int)hipErrorInvalidValue;
    FpRefArgs a{vol, r_sino, w_sino, ray_w, sin_lut, cos_lut, n, n_dets, ang0, n_ang, dir, axis, corr};
    dim3 grid((n_dets + kSplitRays - 1) / kSplitRays, n_ang);
    hipLaunchKernelGGL(k_fp_ref_split, grid, dim3(256), 0, (hipStream_t)stream, a);
    return (int)hipGetLastError();
}

int uirk_transpose(const float *in, float *out, int n, void *stream)
{
    if (n <= 0)
        return 0;
    const unsigned t = (n + 63) / 64;
    hipLaunchKernelGGL(k_transpose, dim3(t, t), dim3(256), 0, (hipStream_t)stream, in, out, n);
    return (int)hipGetLastError();
}

int uirk_fp_blocks(const float *vol, const float *vol_t, const float *r_sino, float *w_sino, const float *ray_w,
                   const float *sin_lut, const float *cos_lut, int n, int n_dets, float axis, float corr, int ang0,
                   int n_ang, void *stream)
{
    if (n_ang <= 0 || n_dets <= 0)
        return 0;
    if (n_ang > 65535)
        return (int)hipErrorInvalidValue;
    FpRefArgs a{vol, r_sino, w_sino, ray_w, sin_lut, cos_lut, n, n_dets, ang0, n_ang, -1, axis, corr};
    const int n_blocks = (n + kBlockSamples - 1) / kBlockSamples;
    const unsigned waves = n_blocks < 1 ? 1 : (n_blocks < kBlkWaves ? n_blocks : kBlkWaves);
    hipLaunchKernelGGL(k_fp_blocks, dim3((n_dets + 63) / 64, n_ang), dim3(64 * waves), 0, (hipStream_t)stream, a,
                       vol_t);
    return (int)hipGetLastError();
}

int uirk_fp_block_starts(const float *sin_lut, const float *cos_lut, int n, int n_dets, float axis, int n_angles,
                         int dir, float *starts, void *stream)
{
    if (n_angles <= 0 || n_dets <= 0 || n <= 0)
        return 0;
    FpRefArgs a{nullptr, nullptr, nullptr, nullptr, sin_lut, cos_lut, n, n_dets, 0, n_angles, dir, axis, 0.0f};
    dim3 grid((n_dets + 255) / 256, n_angles);
    hipLaunchKernelGGL(k_fp_block_starts, grid, dim3(256), 0, (hipStream_t)stream, a, starts);
    return (int)hipGetLastError();
}

int uirk_sart_ref_step(const float *x_in, float *x_out, const float *b, const float *ray_w, const float *starts,
                       const float *part_in, float *part_out, const float *sin_h, const float *cos_h, int n,
                       int n_dets, float axis, float corr, float relax, int bp_ang, int fp_ang, int trans, int turn,
                       int n_xcd, void *stream)
{
    if (n <= 0 || n_dets <= 0)
        return 0;
    const int nt = (n + 63) / 64; // blocks and tiles are both 64 lines
    SartStepArgs a{};
    a.x_in = x_in;
    a.x_out = x_out;
    a.part_in = part_in;
    a.part_out = part_out;
    a.n = n;
    a.n_dets = n_dets;
    a.bp = bp_ang >= 0;
    a.n_bp = bp_ang >= 0 ? nt : 0;
    a.n_xcd = n_xcd > 0 ? n_xcd : 1;
    a.axis = axis;
    a.corr = corr;
    a.relax = relax;
    if (bp_ang >= 0) {
        a.b = b + (size_t)bp_ang * n_dets;
        a.ray_w = ray_w + (size_t)bp_ang * n_dets;
        // X cos - Y sin with X, Y = P, L or, transposed, L, P (the signs go with the factors)
        a.kp = trans ? -sin_h[bp_ang] : cos_h[bp_ang];
        a.kl = trans ? -cos_h[bp_ang] : sin_h[bp_ang];
    }
    if (fp_ang >= 0) {
        const float st = sin_h[fp_ang], ct = cos_h[fp_ang];
        a.starts = starts ? starts + (size_t)fp_ang * nt * n_dets : nullptr;
        a.det_step = trans ? -1.0f / st : 1.0f / ct; // :51-75 / :112-136
        a.step = trans ? ct / st : st / ct;
        a.n_fp = (n_dets + 63) / 64;
    }
    const int grid = a.n_xcd * ((nt + a.n_xcd - 1) / a.n_xcd) * (a.n_fp + a.n_bp);
    if (grid <= 0)
        return 0;
    const float half = (float)n_dets - axis * 2 < 0 ? (float)n_dets - axis : axis;
    const bool window = axis - half + 0.5f <= axis + half - 0.5f;
    const auto kernel = window ? (turn ? k_sart_ref_step<true, true> : k_sart_ref_step<true, false>)
                               : (turn ? k_sart_ref_step<false, true> : k_sart_ref_step<false, false>);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kSartThreads), 0, (hipStream_t)stream, a);
    return (int)hipGetLastError();
}

int uirk_bp_ref(const float *r_vol, float *w_vol, const float *sino, int n_angles,
                const float *sin_lut, const float *cos_lut, int n, int n_dets, float axis,
                float relax, const uirk_runs *runs, int unit_lut, const float *pix_w, int posc, void *stream)
{
    if (n <= 0)
        return 0;
    BpRefArgs a;
    a.r_vol = r_vol;
    a.w_vol = w_vol;
    a.sino = sino;
    a.pix_w = pix_w;
    a.sin_lut = sin_lut;
    a.cos_lut = cos_lut;
    a.n = n;
    a.n_dets = n_dets;
    a.n_angles = n_angles;
    a.posc = posc;
    a.axis = axis;
    a.relax = relax;
    a.runs = *runs;
    // Two pixels a thread from 512 x 512 on (2 waves a SIMD are left): the
    // per-angle scalar work is shared.  Below, one: 15 us against 22 at 256 /
    // 180 / 367; at 512 / 400 / 725 both take 46 - 51 us, at 1024 / 720 / 1448
    // two take 197 us and one 269.
    if (n < 512)
        launch_bp_gather<1>(a, unit_lut != 0, (hipStream_t)stream);
    else
        launch_bp_gather<2>(a, unit_lut != 0, (hipStream_t)stream);
    return (int)hipGetLastError();
}

int uirk_set(float *out, size_t n, float v, void *stream)
{
    if (!n)
        return 0;
    hipLaunchKernelGGL(k_set, dim3(grid1d(n)), dim3(256), 0, (hipStream_t)stream, out, n, v);
    return (int)hipGetLastError();
}

int uirk_copy(float *dst, const float *src, size_t n, void *stream)
{
    if (!n)
        return 0;
    hipLaunchKernelGGL(k_copy, dim3(grid1d(n)), dim3(256), 0, (hipStream_t)stream, dst, src, n);
    return (int)hipGetLastError();
}

int uirk_inv_min(const float *in, float *out, size_t n, float vmin, void *stream)
{
    if (!n)
        return 0;
    hipLaunchKernelGGL(k_inv_min, dim3(grid1d(n)), dim3(256), 0, (hipStream_t)stream, in, out, n, vmin);
    return (int)hipGetLastError();
}

int uirk_inv(const float *in, float *out, size_t n, void *stream)
{
    if (!n)
        return 0;
    hipLaunchKernelGGL(k_inv, dim3(grid1d(n)), dim3(256), 0, (hipStream_t)stream, in, out, n);
    return (int)hipGetLastError();
}

int uirk_binary(int op, const float *a, const float *b, float m, float *out, size_t n, void *stream)
{
    if (!n)
        return 0;
    hipLaunchKernelGGL(k_binary, dim3(grid1d(n)), dim3(256), 0, (hipStream_t)stream, op, a, b, m, out, n);
    return (int)hipGetLastError();
}

int uirk_unary(int op, const float *in, float *out, size_t n, float m, void *stream)
{
    if (!n)
        return 0;
    hipLaunchKernelGGL(k_unary, dim3(grid1d(n)), dim3(256), 0, (hipStream_t)stream, op, in, out, n, m);
    return (int)hipGetLastError();
}

int uirk_mul_rows(const float *a, const float *b, float *out, uint32_t width, uint32_t offset,
                  uint32_t rows, void *stream)
{
    const size_t n = (size_t)width * rows;
    if (!n)
        return 0;
    hipLaunchKernelGGL(k_mul_rows, dim3(grid1d(n)), dim3(256), 0, (hipStream_t)stream, a, b, out, width, offset, rows);
    return (int)hipGetLastError();
}

size_t uirk_reduce_ws_bytes(size_t n)
{
    // f64 partials (kRedMaxBlocks), minmax pairs, compat parts (<= n)
    size_t a = kRedMaxBlocks * sizeof(double) * 2;
    size_t b = n * sizeof(float) + 64;
    return a > b ? a : b;
}

int uirk_l1_f64(const float *v, size_t n, double *ws, double *result_dev, void *stream)
{
    const unsigned nb = red_blocks(n);
    hipLaunchKernelGGL(k_red_f64<0>, dim3(nb), dim3(kRedBlock), 0, (hipStream_t)stream, v, v, n, ws);
    hipLaunchKernelGGL(k_red_final_f64, dim3(1), dim3(kRedBlock), 0, (hipStream_t)stream, ws, nb, result_dev);
    return (int)hipGetLastError();
}

int uirk_dot_f64(const float *a, const float *b, size_t n, double *ws, double *result_dev, void *stream)
{
    const unsigned nb = red_blocks(n);
    hipLaunchKernelGGL(k_red_f64<1>, dim3(nb), dim3(kRedBlock), 0, (hipStream_t)stream, a, b, n, ws);
    hipLaunchKernelGGL(k_red_final_f64, dim3(1), dim3(kRedBlock), 0, (hipStream_t)stream, ws, nb, result_dev);
    return (int)hipGetLastError();
}

int uirk_dot_compat(const float *a, const float *b, uint32_t w, uint32_t h, float *ws,
                    float *result_dev, void *stream)
{
    if (h == 0)
        return (int)hipErrorInvalidValue;
    const uint32_t part_len = (uint32_t)(((size_t)w * h) / h);
    launch_dot_compat(a, b, h, part_len, ws, result_dev, (hipStream_t)stream);
    return (int)hipGetLastError();
}

int uirk_minmax(const float *v, size_t n, float *ws, float *minmax_dev, void *stream)
{
    const unsigned nb = red_blocks(n);
    hipLaunchKernelGGL(k_minmax, dim3(nb), dim3(kRedBlock), 0, (hipStream_t)stream, v, n, ws);
    hipLaunchKernelGGL(k_minmax_final, dim3(1), dim3(64), 0, (hipStream_t)stream, ws, nb, minmax_dev);
    return (int)hipGetLastError();
}

int uirk_normalize_apply(float *v, size_t n, const float *minmax_dev, void *stream)
{
    if (!n)
        return 0;
    hipLaunchKernelGGL(k_normalize_apply, dim3(grid1d(n)), dim3(256), 0, (hipStream_t)stream, v, n, minmax_dev);
    return (int)hipGetLastError();
}

int uirk_diff(int kind, const float *in, float *out, uint32_t w, uint32_t h, void *stream)
{
    if (!w || !h)
        return 0;
    dim3 block(64, 4), grid((w + 63) / 64, (h + 3) / 4);
    hipLaunchKernelGGL(k_diff, grid, block, 0, (hipStream_t)stream, kind, in, out, (int)w, (int)h);
    return (int)hipGetLastError();
}

int uirk_l1_grad(const float *in, float *out, uint32_t w, uint32_t h, void *stream)
{
    if (!w || !h)
        return 0;
    dim3 block(64, 4), grid((w + 63) / 64, (h + 3) / 4);
    hipLaunchKernelGGL(k_l1_grad, grid, block, 0, (hipStream_t)stream, in, out, (int)w, (int)h);
    return (int)hipGetLastError();
}

} // extern "C"

// ==========================================================================
// Allocation-free strided "dot" (uir_op_dot_compat_noalloc)
// ==========================================================================
// The same two kernels as uir_op_dot_compat (one float partial per row, then
// the partials added in row order), with the row partials in this file-scope
// device array instead of a workspace the library allocates, and the result
// written to the caller's device memory without a host synchronisation.  Each
// device holds its own copy of the array for the life of the process.  Every
// partial the final kernel reads is written by the same call's first kernel,
// so nothing needs clearing between calls; calls that overlap on one device
// race on the array.
constexpr uint32_t kNoAllocMaxRows = 65536; // 256 KiB of FP32 partials
static __device__ __align__(256) float scratch[kNoAllocMaxRows];

#include "uir_internal.h"

namespace {
constexpr int kMaxDevices = 64;
float *g_scratch_dev[kMaxDevices]; // the array's device address, per device
pthread_mutex_t g_scratch_lock = PTHREAD_MUTEX_INITIALIZER;

// The device address of `scratch` on the current device, looked up once per
// device (the host-side name is not a device address).
uir_status scratch_address(float **out)
{
    int dev = -1;
    uir_status s = uir_check_hip(hipGetDevice(&dev), "hipGetDevice");
    if (s != UIR_OK)
        return s;
    if (dev < 0 || dev >= kMaxDevices)
        return uir_set_error(UIR_ERR_UNSUPPORTED, "device %d: at most %d devices", dev, kMaxDevices);
    pthread_mutex_lock(&g_scratch_lock);
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        s = uir_check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
        if (s == UIR_OK && !p)
            s = uir_set_error(UIR_ERR_DEVICE, "hipGetSymbolAddress(scratch) gave NULL");
        if (s == UIR_OK)
            g_scratch_dev[dev] = (float *)p;
    }
    *out = g_scratch_dev[dev];
    pthread_mutex_unlock(&g_scratch_lock);
    return s;
}
} // namespace

extern "C" uir_status uir_op_dot_compat_noalloc(const float *a, const float *b, uint32_t width, uint32_t height,
                                                float *d_result, void *stream)
{
    if (!a || !b || !d_result)
        return uir_set_error(UIR_ERR_INVALID_ARGUMENT, "NULL pointer");
    if (height == 0)
        return uir_set_error(UIR_ERR_INVALID_ARGUMENT, "height is 0");
    if (height > kNoAllocMaxRows)
        return uir_set_error(UIR_ERR_INVALID_ARGUMENT,
                             "height %u exceeds the %u rows the allocation-free dot holds (uir_op_dot_compat "
                             "takes any height)", height, kNoAllocMaxRows);
    float *ws = nullptr;
    uir_status s = scratch_address(&ws);
    if (s != UIR_OK)
        return s;
    const uint32_t part_len = (uint32_t)(((size_t)width * height) / height); // ufo-ir-basic-ops-processor.c:181-183
    launch_dot_compat(a, b, height, part_len, ws, d_result, (hipStream_t)stream);
    return uir_check_hip(hipGetLastError(), "dot_compat launch");
}
