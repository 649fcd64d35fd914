// Adaptive raw-data filtering (Kachelriess-Kalender style), reference
// src/preprocessing.cu:31-156 and include/preprocessing.cuh:32-285.
//
// The reference runs one thread per view for every step (a serial loop over
// the 23 552 samples of a view in filter_projections).  Here each step is
// parallelised to its natural width while keeping the reference's float
// arithmetic in the same order (including the fused multiply-adds nvcc forms
// for "acc += a*b"), so results are bit-identical to a sequential FP32
// restatement:
//   1. view maximum         one workgroup per view, tree max (order-free); the
//      stage copies the pull on the way
//   2. 18-degree smoothing  one thread per view, sequential fmaf sum
//   3. 180-degree min/max + eccentricity, and
//   4. threshold bisection  one wavefront per view: the view's window is
//      held in registers (min and max taken on the way, order-free), then
//      exact integer counts over it
//   5. 5x5x5 triangle smoothing of samples above threshold: a wave takes 64
//      channels x 8 rows of a view, or of several views of few rows
// A fixed-threshold mode (no counterpart in the reference) skips steps 1-4
// and smooths the samples above one given line-integral threshold, e.g.
// ln(I0 / N) for a noise threshold of N photons at I0 incident photons.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"

// Only the explicit fmaf calls may fuse: every other multiply-add rounds
// twice, as in the sequential FP32 statement of the algorithm.
#pragma clang fp contract(off)

namespace ctbb {

namespace {

__device__ __forceinline__ float wave_max(float v) {
    for (int s = 32; s > 0; s >>= 1) v = fmaxf(v, __shfl_xor(v, s, 64));
    return v;
}

__device__ __forceinline__ float wave_min(float v) {
    for (int s = 32; s > 0; s >>= 1) v = fminf(v, __shfl_xor(v, s, 64));
    return v;
}

// View maximum, one workgroup per view (max is order-free, so any reduction
// order gives the reference's value), gridDim.x workgroups looping over the
// n_proj views.  frame % 4 == 0 is checked on the host.  kCopy: the frame is
// also copied to out (16-byte stores), so that the apply step only rewrites
// the views the filter changes instead of reading the whole pull again:
// bound by HBM, 8448 views of 32 x 736 in 304 us (5.2 TB/s) against 163 us for the
// maximum and 261 us for an apply step over every view.
template <bool kCopy>
__global__ __launch_bounds__(256) void af_sup(const float *raw, float *sup, float *out, size_t frame, int n_proj) {
    __shared__ float red[4];
    for (int p = blockIdx.x; p < n_proj; p += gridDim.x) {
        const float4 *f = reinterpret_cast<const float4 *>(raw + static_cast<size_t>(p) * frame);
        float4 *o = reinterpret_cast<float4 *>(out + static_cast<size_t>(p) * frame);
        float m = 0.0f;   // reference starts from 0.0f (preprocessing.cuh:75)
        for (size_t i = threadIdx.x; i < frame / 4; i += 256) {
            const float4 v = f[i];
            m = fmaxf(fmaxf(m, fmaxf(v.x, v.y)), fmaxf(v.z, v.w));
            if (kCopy) o[i] = v;
        }
        m = wave_max(m);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
        __syncthreads();
        if (threadIdx.x == 0) sup[p] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        __syncthreads();                        // red is rewritten for the next view
    }
}

// reference preprocessing.cuh:87-113.  64 views per workgroup, their window
// of maxima (edge indices clamped) in LDS, kSmoothPart values of a view's sum at a
// time: the n_avg dependent fused multiply-adds then wait for LDS instead of
// memory (8448 views, n_avg 231: 5.3 against 23 us).
constexpr int kSmoothViews = 64, kSmoothPart = 1024;

__global__ __launch_bounds__(kSmoothViews) void af_smooth(const float *sup, float *sm, int n_proj, int n_avg) {
    __shared__ float w[kSmoothViews + kSmoothPart];
    const int p0 = blockIdx.x * kSmoothViews, off = n_avg / 2, max_idx = n_proj - 1;
    const float inv = 1.0f / static_cast<float>(n_avg);
    float acc = 0.0f;
    for (int i0 = 0; i0 < n_avg; i0 += kSmoothPart) {
        const int n = min(n_avg - i0, kSmoothPart);
        if (i0 > 0) __syncthreads();
        for (int i = threadIdx.x; i < kSmoothViews + n; i += kSmoothViews) {
            int idx = p0 - off + i0 + i;
            idx = idx < 0 ? 0 : (idx > max_idx ? max_idx : idx);
            w[i] = sup[idx];
        }
        __syncthreads();
#pragma unroll 8
        for (int i = 0; i < n; i++) acc = fmaf(inv, w[threadIdx.x + i], acc);
    }
    if (p0 + static_cast<int>(threadIdx.x) < n_proj) sm[p0 + threadIdx.x] = acc;
}

// The counting window of reference preprocessing.cuh:32-62 (clipped to the
// pull), fixed for a view while the bisection moves T.
__device__ __forceinline__ void af_window(int &start_idx, int &numel_range, int max_idx) {
    const int diff = start_idx + (numel_range - 1);
    if (diff < numel_range - 1) {
        numel_range += start_idx;
        start_idx = 0;
    }
    if (diff > max_idx) numel_range -= (diff - max_idx);
}

// reference preprocessing.cuh:115-206; one wavefront per view.  The view's
// window stays in registers (kVals per lane, lane l the values l, l + 64,
// ...; kVals = 0: windows over 64 * 44 values are read from memory at every
// step), its minimum and maximum taken on the way (the reference's 180-degree
// range, preprocessing.cuh:115-163: the same views as the counting window,
// its clamped edge indices repeat values inside it).  A bisection step counts
// the values above T exactly with one compare per register and scalar
// population counts; once the counts at both ends of the interval agree no
// value lies between them, every later count is the same and only T moves.
// Bound by instruction issue: 8448 views with 2305 values 51 us against
// 111 us with the window in LDS, shuffles and a count at every step (four
// waves per view, which repeat the scalar steps: 61 us).
template <int kVals>
__global__ __launch_bounds__(64) void af_thresh(const float *sm, float *thr, int n_proj, int n_range, int n_proj_ffs,
                                                float strength) {
    const int p = blockIdx.x, lane = threadIdx.x;
    const int max_idx = n_proj - 1;
    int start = p - n_range / 2, numel = n_range;
    af_window(start, numel, max_idx);
    const float *win = sm + start;
    float v[kVals > 0 ? kVals : 1];
    float hi = 0.0f, lo = 10000.0f;     // the reference's starting values
    if (kVals > 0) {
#pragma unroll
        for (int q = 0; q < kVals; q++) {
            const float x = win[min(64 * q + lane, numel - 1)];     // (unconditional: all loads in flight)
            hi = fmaxf(hi, x);
            lo = fminf(lo, x);
            v[q] = 64 * q + lane < numel ? x : -1.0f;               // (never above T >= 0)
        }
    } else {
        for (int i = lane; i < numel; i += 64) {
            hi = fmaxf(hi, win[i]);
            lo = fminf(lo, win[i]);
        }
    }
    hi = wave_max(hi);
    lo = wave_min(lo);
    float e = 1 - lo / hi;
    e = (e - 0.3f) / (0.5f - 0.3f);
    const float ecc = e > 1 ? 1.0f : (e < 0 ? 0.0f : e);
    const float inv_pi = 1.0f / 3.1415368979f;
    const float inv_npf = 1.0f / static_cast<float>(n_proj_ffs);
    float lower = lo, upper = hi;
    float T = (hi + lo) / 2.0f;
    const float lhs = 0.03f * strength * ecc;
    auto count = [&](float t) {
        int cnt = 0;
        if (kVals > 0) {
#pragma unroll
            for (int q = 0; q < kVals; q++) cnt += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v[q] > t));
        } else {
            for (int i0 = 0; i0 < numel; i0 += 64)
                cnt += __builtin_popcountll(__builtin_amdgcn_ballot_w64(i0 + lane < numel && win[i0 + lane] > t));
        }
        return cnt;
    };
    // rhs of reference preprocessing.cuh:32-62: the exact count of values
    // above T, then the reference's float products
    int cnt = count(T), cnt_lower = -1, cnt_upper = 0;  // (above the maximum: none)
    float rhs = inv_pi * static_cast<float>(cnt) * inv_npf;
    int iter = 0;
    while (static_cast<double>(fabsf(lhs - rhs) / lhs) > 0.01) {
        if (iter >= 20) break;
        iter += 1;
        if (rhs > lhs) {
            lower = T;
            cnt_lower = cnt;
        } else if (rhs < lhs) {
            upper = T;
            cnt_upper = cnt;
        } else {
            break;
        }
        T = (lower + upper) / 2.0f;
        if (cnt_lower == cnt_upper) {
            // rhs, and with it the test and the side taken, stays
            for (; iter < 20; iter++) {
                if (rhs > lhs) lower = T;
                else upper = T;
                T = (lower + upper) / 2.0f;
            }
            break;
        }
        cnt = count(T);
        rhs = inv_pi * static_cast<float>(cnt) * inv_npf;
    }
    if (lane == 0) thr[p] = T;
}

// Apply step, reference preprocessing.cuh:208-285 (3D branch, __FILTER_3D__
// defined): a sample x <= T is kept, one above it becomes the 5x5x5 weighted
// mean of its neighbourhood, weights triangle_3d(5, ii, jj, kk) with
// ceil(5/2) = 3 (peak at offset +1), summed over channel, row, view in this
// order, each sum one chain of fused multiply-adds.
//
// One wave takes 64 channels x kRows rows of one view, a lane one channel.
// A wave with no sample above T copies its rows.  Otherwise the lane walks
// the channels ii (rolled) and rows of its neighbourhood, loads the row's 5
// views once and feeds them to every output row they belong to: 60 loads per
// channel for 8 output rows, 37.5 per output instead of 125, with 125 fused
// multiply-adds.  Neighbours outside the pull contribute nothing: they read
// as zeros through the buffer descriptors (one per view, of the frame's size
// and of size 0 for a view outside the pull; a row or channel outside the
// frame gives an offset past its end), and a zero leaves the sum as it is.
// The sums keep the order and so the bits of the one-sample form.
// Bound by the VALU where samples are smoothed and by HBM elsewhere; views
// are dealt to the XCDs in contiguous bands so that the 5 frames around a
// view are read from one L2.  4096 views of 32 x 672 samples with a fixed
// threshold of 1.204: 4.52 ms with one thread per four samples and 125
// guarded loads each, 0.36 ms here (with no sample above T, 8448 views of
// 32 x 736: 0.26 ms, 6.1 TB/s).
constexpr int kRows = 8;

__device__ __forceinline__ constexpr int af_tri(int i) { return 3 - (i < 3 ? 3 - i : i - 3); }

// kGroup rows are loaded at a time: with smoothed samples everywhere the other
// waves cover the loads and one row at a time needs the fewest registers (0.36
// against 0.39 ms for two); where few waves smooth, each waits for memory at
// every group.
// kFew: rows outside the frame are passed over.
template <int kGroup, bool kFew>
__device__ __forceinline__ void af_smooth_rows(const float *raw, float (&acc)[kRows], int i, int j0, int p, int n_proj,
                                               int n_rows_raw, int nch, size_t ps) {
    __amdgpu_buffer_rsrc_t rs[5];
#pragma unroll
    for (int kk = 0; kk < 5; kk++) {
        const int fp = p + kk - 2;
        const bool in = fp >= 0 && fp < n_proj;
        rs[kk] = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(raw + ps * (in ? fp : p)), static_cast<short>(0),
                                                   in ? static_cast<int>(ps * sizeof(float)) : 0, 0x00020000);
    }
#pragma unroll
    for (int r = 0; r < kRows; r++) acc[r] = 0.0f;
    const int row_b = nch * 4;
#pragma unroll 1
    for (int ii = 0; ii < 5; ii++) {
        const int c = i + ii - 2;
        const float ta = static_cast<float>(3 - abs(ii - 3));
        // byte offset of (row j0 - 2, channel c); a channel outside the frame
        // stays past the end of every frame (< 2 GiB) for all kRows + 4 rows
        int off = c >= 0 && c < nch ? (j0 - 2) * row_b + c * 4 : static_cast<int>(0x80000000u);
        const bool c_in = off != static_cast<int>(0x80000000u);
        static_assert((kRows + 4) % kGroup == 0, "whole groups of rows");
#pragma unroll
        for (int q0 = 0; q0 < kRows + 4; q0 += kGroup) {
            if (kFew && (j0 - 2 + q0 + kGroup <= 0 || j0 - 2 + q0 >= n_rows_raw)) {
                off = c_in ? off + kGroup * row_b : off;
                continue;
            }
            float v[kGroup][5];
#pragma unroll
            for (int g = 0; g < kGroup; g++) {          // row j0 - 2 + q0 + g
#pragma unroll
                for (int kk = 0; kk < 5; kk++)
                    v[g][kk] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs[kk], off, 0, 0));
                off = c_in ? off + row_b : off;
            }
            if (kGroup > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < kGroup; g++)
#pragma unroll
                for (int r = 0; r < kRows; r++) {
                    const int jj = q0 + g - r;          // output row j0 + r sees it as row offset jj - 2
                    if (jj < 0 || jj > 4) continue;
#pragma unroll
                    for (int kk = 0; kk < 5; kk++)
                        acc[r] = fmaf(v[g][kk], ta + static_cast<float>(af_tri(jj) + af_tri(kk) + 1), acc[r]);
                }
        }
    }
}

// Sum of the weights of the neighbours inside the pull (whole numbers below
// 2^24: exact in any order).
__device__ __forceinline__ float af_norm(int i, int j, int p, int n_proj, int n_rows_raw, int nch) {
    auto axis = [](int at, int n, int &count, int &sum) {
        count = sum = 0;
#pragma unroll
        for (int o = 0; o < 5; o++)
            if (at + o - 2 >= 0 && at + o - 2 < n) {
                count += 1;
                sum += af_tri(o);
            }
    };
    int ni, nj, nk, si, sj, sk;
    axis(i, nch, ni, si);
    axis(j, n_rows_raw, nj, sj);
    axis(p, n_proj, nk, sk);
    return static_cast<float>(si * nj * nk + sj * ni * nk + sk * ni * nj + ni * nj * nk);
}

// Rows j0 .. j0 + kRows - 1 of channels i (one per lane) of view p; kCopied:
// out already holds the raw samples, only waves that smooth some are written.
template <bool kCopied, int kGroup, bool kFew>
__device__ __forceinline__ void af_apply_rows(const float *raw, float T, float *out, int i, int j0, int p, int n_proj,
                                              int n_rows_raw, int nch, size_t ps) {
    const size_t base = ps * p + static_cast<size_t>(j0) * nch + i;
    float x[kRows];
    bool hot = false;
#pragma unroll
    for (int r = 0; r < kRows; r++) {
        x[r] = i < nch && j0 + r < n_rows_raw ? raw[base + static_cast<size_t>(r) * nch] : 0.0f;
        hot |= i < nch && j0 + r < n_rows_raw && x[r] > T;
    }
    if (__builtin_amdgcn_ballot_w64(hot)) {
        float acc[kRows];
        af_smooth_rows<kGroup, kFew>(raw, acc, i, j0, p, n_proj, n_rows_raw, nch, ps);
#pragma unroll
        for (int r = 0; r < kRows; r++)
            if (x[r] > T) x[r] = (1.0f / af_norm(i, j0 + r, p, n_proj, n_rows_raw, nch)) * acc[r];
    } else if (kCopied) {
        return;
    }
#pragma unroll
    for (int r = 0; r < kRows; r++)
        if (i < nch && j0 + r < n_rows_raw) out[base + static_cast<size_t>(r) * nch] = x[r];
}

// Waves (64 channels x kRows rows) of a view.
__host__ __device__ __forceinline__ int af_view_waves(int n_rows_raw, int nch) {
    return ((nch + 63) / 64) * ((n_rows_raw + kRows - 1) / kRows);
}

// bpv workgroups of 4 waves per view, XCD x the x-th eighth of the views.
enum ApplyMode {
    kAllViews,      // every view
    kHotFlagged,    // only the views the filter changes (view p is unchanged where its maximum, af_sup from 0, is at or
                    // below its threshold); hot[p] flags them, a reader takes the others from the raw pull
    kHotCopied      // only those views, and of them only the samples it changes: out holds a copy of the pull
};

// (kHotFlagged takes 56 VGPRs: beside a backprojection's four waves of 112 one
// of it fits.)
template <int kMode>
__global__ __launch_bounds__(256) void af_apply(const float *raw, const float *sup, const float *thr, float *out,
                                                unsigned char *hot, int n_proj, int n_rows_raw, int nch, int bpv) {
    const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3, band = (n_proj + 7) / 8;
    const int pv = idx / bpv, p = xcd * band + pv, part = idx - pv * bpv;
    if (pv >= band || p >= n_proj) return;
    const float T = thr[p];
    if (kMode != kAllViews) {
        const bool h = sup[p] > T;
        if (kMode == kHotFlagged && part == 0 && threadIdx.x == 0) hot[p] = h ? 1 : 0;
        if (!h) return;
    }
    const int tiles = (nch + 63) / 64, waves = af_view_waves(n_rows_raw, nch);
#pragma unroll 1
    for (int w = part * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); w < waves; w += 4 * bpv) {
        const int g = w / tiles;
        af_apply_rows<kMode == kHotCopied, kMode == kAllViews ? 1 : 2, false>(
            raw, T, out, (w - g * tiles) * 64 + (threadIdx.x & 63), g * kRows, p, n_proj, n_rows_raw, nch,
            static_cast<size_t>(nch) * n_rows_raw);
    }
}

// Every view of a detector of few rows: a wave takes the kRows / n_rows_raw views
// that fill its rows, copies those without a sample above their threshold and
// smooths the others one by one.  XCD x takes the x-th `band` of these groups of
// views.  With 8 rows of one view per wave most of a wave were rows outside the
// frame: 46592 views of 672 channels in one row, all smoothed / a thousandth of
// the samples above the threshold, 348 / 102 against 1216 / 324 us (one thread per
// four samples: 1178 / 134), 24192 views of two rows 265 / 112 against 660 / 217
// (1967 / 217).
__global__ __launch_bounds__(256) void af_apply_few(const float *raw, const float *thr, float *out, int n_proj,
                                                    int n_rows_raw, int nch, int band) {
    const int xcd = blockIdx.x & 7, tiles = (nch + 63) / 64, n_v = kRows / n_rows_raw;
    const int w = static_cast<int>(blockIdx.x >> 3) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int group = w / tiles, i = (w - group * tiles) * 64 + (threadIdx.x & 63);
    const int p0 = (xcd * band + group) * n_v;
    if (group >= band || p0 >= n_proj) return;
    const size_t ps = static_cast<size_t>(nch) * n_rows_raw;
    // rows of the group's views, one after the other in memory
    const int rows = min(n_v, n_proj - p0) * n_rows_raw;
    const size_t base = ps * p0 + i;
    float x[kRows];
    unsigned hot = 0;               // views with a sample above their threshold
#pragma unroll
    for (int r = 0; r < kRows; r++) x[r] = r < rows && i < nch ? raw[base + static_cast<size_t>(r) * nch] : 0.0f;
#pragma unroll
    for (int r = 0; r < kRows; r++) {
        const int v = r / n_rows_raw;
        if (r < rows && __builtin_amdgcn_ballot_w64(i < nch && x[r] > thr[p0 + v])) hot |= 1u << v;
    }
#pragma unroll
    for (int r = 0; r < kRows; r++)
        if (r < rows && i < nch && !(hot >> (r / n_rows_raw) & 1u)) out[base + static_cast<size_t>(r) * nch] = x[r];
#pragma unroll 1
    for (int v = 0; hot >> v; v++)
        if (hot >> v & 1u)
            af_apply_rows<false, 1, true>(raw, thr[p0 + v], out, i, 0, p0 + v, n_proj, n_rows_raw, nch, ps);
}

// Fixed-threshold mode: every view's threshold is the same constant.
__global__ __launch_bounds__(256) void af_const(float *thr, int n_proj, float T) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n_proj) thr[p] = T;
}

int odd_window(float frac, int n_proj_ffs) {
    int n = static_cast<int>(ceilf(frac * static_cast<float>(n_proj_ffs)));
    return n + (1 - n % 2);
}

}  // namespace

int launch_adaptive(const AdaptiveArgs &a, hipStream_t stream) {
    if (!a.raw || !a.out || !a.work || a.raw == a.out) return CTBB_ERR_ARG;
    if (a.n_proj <= 0 || a.n_rows_raw <= 0 || a.nch <= 0 || a.n_proj_ffs <= 0) return CTBB_ERR_SHAPE;
    if (a.n_proj > 65535 || a.n_rows_raw > 65535) return CTBB_ERR_SHAPE;  // grid.z / grid.y limits
    if ((static_cast<size_t>(a.n_rows_raw) * a.nch) % 4 != 0) return CTBB_ERR_SHAPE;  // float4 frames
    const size_t np = static_cast<size_t>(a.n_proj);
    // work: [sup][sm][3 unused][thr], n_proj floats each
    float *sup = a.work, *sm = sup + np, *thr = sm + 4 * np;
    const size_t frame = static_cast<size_t>(a.n_rows_raw) * a.nch;
    const int n_avg = odd_window(18.0f / 360.0f, a.n_proj_ffs);
    const int n_range = odd_window(180.0f / 360.0f, a.n_proj_ffs);
    const unsigned g1 = static_cast<unsigned>((a.n_proj + 255) / 256);
    if (a.max_groups < 0) return CTBB_ERR_SHAPE;
    const unsigned gsup = static_cast<unsigned>(a.max_groups > 0 && a.max_groups < a.n_proj ? a.max_groups : a.n_proj);
    // A per-view threshold leaves most views unchanged (it is placed so that
    // few of the view maxima exceed it), so out of place the pull is copied
    // while its maxima are taken and only the changed views are visited again;
    // a fixed threshold has no maxima to take and reads the pull once.
    const bool aligned = (reinterpret_cast<uintptr_t>(a.raw) & 15u) == 0 && (reinterpret_cast<uintptr_t>(a.out) & 15u) == 0;
    const bool fixed = a.fixed_threshold > 0.0f;
    const bool copied = !a.hot_only && !fixed && aligned;
    if (fixed) {
        if (!(a.fixed_threshold < 3.0e38f)) return CTBB_ERR_ARG;
        hipLaunchKernelGGL(af_const, dim3(g1), dim3(256), 0, stream, thr, a.n_proj, a.fixed_threshold);
    }
    // (with a fixed threshold the view maxima decide which views hot_only writes)
    if (copied)
        hipLaunchKernelGGL(af_sup<true>, dim3(gsup), dim3(256), 0, stream, a.raw, sup, a.out, frame, a.n_proj);
    else if (!fixed || a.hot_only)
        hipLaunchKernelGGL(af_sup<false>, dim3(gsup), dim3(256), 0, stream, a.raw, sup, a.out, frame, a.n_proj);
    if (!fixed) {
        hipLaunchKernelGGL(af_smooth, dim3(static_cast<unsigned>((a.n_proj + kSmoothViews - 1) / kSmoothViews)),
                           dim3(kSmoothViews), 0, stream, sup, sm, a.n_proj, n_avg);
        if (n_range <= 64 * 16)
            hipLaunchKernelGGL(af_thresh<16>, dim3(a.n_proj), dim3(64), 0, stream, sm, thr, a.n_proj, n_range,
                               a.n_proj_ffs, a.strength);
        else if (n_range <= 64 * 44)
            hipLaunchKernelGGL(af_thresh<44>, dim3(a.n_proj), dim3(64), 0, stream, sm, thr, a.n_proj, n_range,
                               a.n_proj_ffs, a.strength);
        else
            hipLaunchKernelGGL(af_thresh<0>, dim3(a.n_proj), dim3(64), 0, stream, sm, thr, a.n_proj, n_range,
                               a.n_proj_ffs, a.strength);
    }
    // (a form that visits few views gives a workgroup up to 16 of a view's
    // waves: most of its workgroups only find their view unchanged)
    const bool few = a.hot_only || copied;
    const int bpv = (af_view_waves(a.n_rows_raw, a.nch) + (few ? 15 : 3)) / (few ? 16 : 4);
    const unsigned long long grid = 8ull * static_cast<unsigned long long>((a.n_proj + 7) / 8) * bpv;
    if (grid > 0x7fffffffull) return CTBB_ERR_SHAPE;
    // (bands of groups of views, af_apply_few)
    const int few_views = kRows / std::min(a.n_rows_raw, kRows), few_band = ((a.n_proj + few_views - 1) / few_views + 7) / 8;
    unsigned char *hot = adaptive_hot_flags(a.work, a.n_proj);
    const dim3 g(static_cast<unsigned>(grid));
    if (a.hot_only)
        hipLaunchKernelGGL(af_apply<kHotFlagged>, g, dim3(256), 0, stream, a.raw, sup, thr, a.out, hot, a.n_proj,
                           a.n_rows_raw, a.nch, bpv);
    else if (copied)
        hipLaunchKernelGGL(af_apply<kHotCopied>, g, dim3(256), 0, stream, a.raw, sup, thr, a.out, hot, a.n_proj,
                           a.n_rows_raw, a.nch, bpv);
    else if (2 * a.n_rows_raw <= kRows)
        hipLaunchKernelGGL(af_apply_few, dim3(8 * ((few_band * ((a.nch + 63) / 64) + 3) / 4)), dim3(256), 0, stream,
                           a.raw, thr, a.out, a.n_proj, a.n_rows_raw, a.nch, few_band);
    else
        hipLaunchKernelGGL(af_apply<kAllViews>, g, dim3(256), 0, stream, a.raw, sup, thr, a.out, hot, a.n_proj,
                           a.n_rows_raw, a.nch, bpv);
    return hipGetLastError() == hipSuccess ? CTBB_OK : CTBB_ERR_HIP;
}

}  // namespace ctbb
