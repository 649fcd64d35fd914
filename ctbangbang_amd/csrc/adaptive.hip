// Adaptive raw-data filtering (Kachelriess-Kalender style), reference
// src/preprocessing.cu:31-156 and include/preprocessing.cuh:32-285.
//
// The reference runs one thread per view for every step (a serial loop over
// the 23 552 samples of a view in filter_projections).  Here each step is
// parallelised to its natural width while keeping the reference's float
// arithmetic in the same order (including the fused multiply-adds nvcc forms
// for "acc += a*b"), so results are bit-identical to a sequential FP32
// restatement:
//   1. view maximum         one workgroup per view, tree max (order-free)
//   2. 18-degree smoothing  one thread per view, sequential fmaf sum
//   3. 180-degree min/max + eccentricity, and
//   4. threshold bisection  one wavefront per view: the view's window is
//      copied once to LDS (min and max taken on the way, order-free), then
//      exact integer counts over it
//   5. 5x5x5 triangle smoothing of samples above threshold: one thread per
//      sample (coalesced along channels)
// A fixed-threshold mode (no counterpart in the reference) skips steps 1-4
// and smooths the samples above one given line-integral threshold, e.g.
// ln(I0 / N) for a noise threshold of N photons at I0 incident photons.
#include <hip/hip_runtime.h>

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
// n_proj views.  frame % 4 == 0 is checked on the host.
__global__ __launch_bounds__(256) void af_sup(const float *raw, float *sup, size_t frame, int n_proj) {
    __shared__ float red[4];
    for (int p = blockIdx.x; p < n_proj; p += gridDim.x) {
        const float4 *f = reinterpret_cast<const float4 *>(raw + static_cast<size_t>(p) * frame);
        float m = 0.0f;   // reference starts from 0.0f (preprocessing.cuh:75)
        for (size_t i = threadIdx.x; i < frame / 4; i += 256) {
            const float4 v = f[i];
            m = fmaxf(fmaxf(m, fmaxf(v.x, v.y)), fmaxf(v.z, v.w));
        }
        m = wave_max(m);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
        __syncthreads();
        if (threadIdx.x == 0) sup[p] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        __syncthreads();                        // red is rewritten for the next view
    }
}

// reference preprocessing.cuh:87-113
__global__ void af_smooth(const float *sup, float *sm, int n_proj, int n_avg) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_proj) return;
    const int off = n_avg / 2;
    const int max_idx = n_proj - 1;
    const float inv = 1.0f / static_cast<float>(n_avg);
    float acc = 0.0f;
    for (int i = 0; i < n_avg; i++) {
        int idx = p - off + i;
        idx = idx < 0 ? 0 : (idx > max_idx ? max_idx : idx);
        acc = fmaf(inv, sup[idx], acc);
    }
    sm[p] = acc;
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

// rhs of reference preprocessing.cuh:32-62 for a window of numel values:
// the exact count of values above T, then the reference's float products.
__device__ __forceinline__ float af_rhs_wave(const float *win, int numel, float T, float inv_pi_npf_a,
                                             float inv_npf) {
    int cnt = 0;
    for (int i = threadIdx.x & 63; i < numel; i += 64) cnt += win[i] > T ? 1 : 0;
    for (int s = 32; s > 0; s >>= 1) cnt += __shfl_xor(cnt, s, 64);
    return inv_pi_npf_a * static_cast<float>(cnt) * inv_npf;
}

// reference preprocessing.cuh:115-206; one wavefront per view.  The view's
// window is copied to LDS once (kLds, when it fits in the dynamic LDS the
// host gives the launch), its minimum and maximum taken on the way (the
// reference's 180-degree range, preprocessing.cuh:115-163: the same views as
// the counting window, its clamped edge indices repeat values inside it),
// and every bisection step counts from there; otherwise each step reads the
// window from memory.
template <bool kLds>
__global__ __launch_bounds__(64) void af_thresh(const float *sm, float *thr, int n_proj, int n_range, int n_proj_ffs,
                                                float strength) {
    extern __shared__ float win_lds[];
    const int p = blockIdx.x;
    const int max_idx = n_proj - 1;
    int start = p - n_range / 2, numel = n_range;
    af_window(start, numel, max_idx);
    const float *win = sm + start;
    float hi = 0.0f, lo = 10000.0f;     // the reference's starting values
    for (int i = threadIdx.x; i < numel; i += 64) {
        const float v = win[i];
        hi = fmaxf(hi, v);
        lo = fminf(lo, v);
        if (kLds) win_lds[i] = v;
    }
    hi = wave_max(hi);
    lo = wave_min(lo);
    if (kLds) {
        __syncthreads();
        win = win_lds;
    }
    float e = 1 - lo / hi;
    e = (e - 0.3f) / (0.5f - 0.3f);
    const float ecc = e > 1 ? 1.0f : (e < 0 ? 0.0f : e);
    const float inv_pi = 1.0f / 3.1415368979f;
    const float inv_npf = 1.0f / static_cast<float>(n_proj_ffs);
    float lower = lo, upper = hi;
    float T = (hi + lo) / 2.0f;
    const float lhs = 0.03f * strength * ecc;
    float rhs = af_rhs_wave(win, numel, T, inv_pi, inv_npf);
    int iter = 0;
    while (static_cast<double>(fabsf(lhs - rhs) / lhs) > 0.01) {
        if (iter >= 20) break;
        iter += 1;
        if (rhs > lhs) lower = T;
        else if (rhs < lhs) upper = T;
        else break;
        T = (lower + upper) / 2.0f;
        rhs = af_rhs_wave(win, numel, T, inv_pi, inv_npf);
    }
    if (threadIdx.x == 0) thr[p] = T;
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
#pragma unroll
        for (int q = 0; q < kRows + 4; q++) {           // row j0 - 2 + q
            float v[5];
#pragma unroll
            for (int kk = 0; kk < 5; kk++)
                v[kk] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs[kk], off, 0, 0));
            off = c_in ? off + row_b : off;
#pragma unroll
            for (int r = 0; r < kRows; r++) {
                const int jj = q - r;                   // output row j0 + r sees it as row offset jj - 2
                if (jj < 0 || jj > 4) continue;
#pragma unroll
                for (int kk = 0; kk < 5; kk++)
                    acc[r] = fmaf(v[kk], ta + static_cast<float>(af_tri(jj) + af_tri(kk) + 1), acc[r]);
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

// Rows j0 .. j0 + kRows - 1 of channels i (one per lane) of view p.
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
        af_smooth_rows(raw, acc, i, j0, p, n_proj, n_rows_raw, nch, ps);
#pragma unroll
        for (int r = 0; r < kRows; r++)
            if (x[r] > T) x[r] = (1.0f / af_norm(i, j0 + r, p, n_proj, n_rows_raw, nch)) * acc[r];
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
// kHot: only the views the filter changes (view p is unchanged where its
// maximum, af_sup from 0, is at or below its threshold); hot[p] flags them,
// and a reader takes the other views from the raw pull (C1: about 6% of the
// views are hot).  37 VGPRs: a wave of it fits beside a backprojection's four.
template <bool kHot>
__device__ __forceinline__ void af_apply_block(const float *raw, const float *sup, const float *thr, float *out,
                                               unsigned char *hot, int n_proj, int n_rows_raw, int nch, int bpv) {
    const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3, band = (n_proj + 7) / 8;
    const int pv = idx / bpv, p = xcd * band + pv, part = idx - pv * bpv;
    if (pv >= band || p >= n_proj) return;
    const float T = thr[p];
    if (kHot) {
        const bool h = sup[p] > T;
        if (part == 0 && threadIdx.x == 0) hot[p] = h ? 1 : 0;
        if (!h) return;
    }
    const int tiles = (nch + 63) / 64;
    const int w = part * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (w >= af_view_waves(n_rows_raw, nch)) return;
    const int g = w / tiles;
    af_apply_rows(raw, T, out, (w - g * tiles) * 64 + (threadIdx.x & 63), g * kRows, p, n_proj, n_rows_raw, nch,
                  static_cast<size_t>(nch) * n_rows_raw);
}

__global__ __launch_bounds__(256) void af_apply(const float *raw, const float *thr, float *out, int n_proj,
                                                int n_rows_raw, int nch, int bpv) {
    af_apply_block<false>(raw, nullptr, thr, out, nullptr, n_proj, n_rows_raw, nch, bpv);
}

__global__ __launch_bounds__(256) void af_apply_hot(
    const float *raw, const float *sup, const float *thr, float *out, unsigned char *hot, int n_proj, int n_rows_raw,
    int nch, int bpv) {
    af_apply_block<true>(raw, sup, thr, out, hot, n_proj, n_rows_raw, nch, bpv);
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
    if (a.fixed_threshold > 0.0f) {
        if (!(a.fixed_threshold < 3.0e38f)) return CTBB_ERR_ARG;
        hipLaunchKernelGGL(af_const, dim3(g1), dim3(256), 0, stream, thr, a.n_proj, a.fixed_threshold);
        // (the view maxima decide which views hot_only writes)
        if (a.hot_only) hipLaunchKernelGGL(af_sup, dim3(gsup), dim3(256), 0, stream, a.raw, sup, frame, a.n_proj);
    } else {
        hipLaunchKernelGGL(af_sup, dim3(gsup), dim3(256), 0, stream, a.raw, sup, frame, a.n_proj);
        hipLaunchKernelGGL(af_smooth, dim3(g1), dim3(256), 0, stream, sup, sm, a.n_proj, n_avg);
        // the counting window (at most n_range values) in LDS when it takes <= 16 KB
        const size_t win_bytes = static_cast<size_t>(n_range) * sizeof(float);
        if (win_bytes <= 16384)
            hipLaunchKernelGGL(af_thresh<true>, dim3(a.n_proj), dim3(64), win_bytes, stream, sm, thr, a.n_proj,
                               n_range, a.n_proj_ffs, a.strength);
        else
            hipLaunchKernelGGL(af_thresh<false>, dim3(a.n_proj), dim3(64), 0, stream, sm, thr, a.n_proj, n_range,
                               a.n_proj_ffs, a.strength);
    }
    const int bpv = (af_view_waves(a.n_rows_raw, a.nch) + 3) / 4;
    const unsigned long long grid = 8ull * static_cast<unsigned long long>((a.n_proj + 7) / 8) * bpv;
    if (grid > 0x7fffffffull) return CTBB_ERR_SHAPE;
    if (a.hot_only)
        hipLaunchKernelGGL(af_apply_hot, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, a.raw, sup, thr, a.out,
                           adaptive_hot_flags(a.work, a.n_proj), a.n_proj, a.n_rows_raw, a.nch, bpv);
    else
        hipLaunchKernelGGL(af_apply, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, a.raw, thr, a.out,
                           a.n_proj, a.n_rows_raw, a.nch, bpv);
    return hipGetLastError() == hipSuccess ? CTBB_OK : CTBB_ERR_HIP;
}

}  // namespace ctbb
