// Fan-to-parallel rebinning with flying focal spot, fused into a single pass
// per FFS mode and writing the backprojection layout directly.
//
// Reference behaviour (GPU path, clamp-addressed linear texture fetches):
//   no FFS   n1_rebin/n2_rebin    include/rebin_filter.cuh:72-96
//   z FFS    z1_rebin/z2_rebin    include/rebin_filter.cuh:186-228
//   phi FFS  p1/p2_rebin_t + p1/p2_rebin   include/rebin_filter.cuh:111-169
//   phi+z    a1..a4_rebin_t + a1/a2_rebin_b include/rebin_filter.cuh:247-350
//   + reshape_out (view trimming, [proj][row][channel] layout)
//                                 include/rebin_filter.cuh:354-366
// The reference stages the raw data through focal-spot "sheets", texture
// arrays and a full-size intermediate per pass; here each output sample is
// computed directly from the raw pull with the same clamped bilinear
// arithmetic (2 taps along the azimuthal axis of each of the 2 channel taps),
// using FP64-derived per-channel coordinate maps (geometry.cpp).
//
// Output element (v, r, c) = rebinned projection v + add_projections, row r,
// oversampled channel c.  Threads run along c (coalesced writes).  In every
// mode it interpolates linearly between two channel taps, each linear between
// the readings p and p + 1 of its focal spot, p + f = (v + add) - aoff, and
// aoff does not depend on the view: from one view to the next p moves by
// exactly one reading, the upper one becoming the lower, and f stays but for
// the rounding of the index.  A thread that walks kViews views therefore
// loads one new sample per tap and view at an address that only advances by
// a uniform step.
//
// Every raw sample the reconstruction uses reaches some rebinned sample
// (non-finite values propagate through the interpolation), so the kernels
// also report non-finite input: a wave with a non-finite output sample
// stores 1 to *nonfinite (the reference instead drops such fetches in its
// backprojection and resets h_t, include/backproject.cuh:89-95).
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace ctbb {

namespace {

// Views per thread (one more reading is loaded than views are written), and
// views whose loads are in flight together.  1934 views of 64 rows x 1472
// channels, four focal spots: 550 us (822 us with four loads per output and
// the index arithmetic per view and tap); 16 to 128 views, batches of 4 or 8
// and any occupancy from 4 waves per SIMD up stay within 545-575 us: the
// kernel is bound by the cache lines a gather touches (a wave's 64 channels
// lie on about 14 readings' rows), 90-110 cycles per CU and wave of output.
constexpr int kViews = 16;
constexpr int kBatch = 4;

// Clamp a fractional index into [0, n-1] and split it into the two taps and
// the weight of the upper tap (texture clamp addressing).
__device__ __forceinline__ void taps(float x, int n, int &i0, int &i1, float &f) {
    x = fminf(fmaxf(x, 0.0f), static_cast<float>(n - 1));
    float fl = floorf(x);
    i0 = static_cast<int>(fl);
    i1 = min(i0 + 1, n - 1);
    f = x - fl;
}

// One plain store of 1 per wave that saw a non-finite output sample (every
// writer stores the same value, so no atomic is needed).
__device__ __forceinline__ void report_nonfinite(unsigned *flag, bool bad) {
    const unsigned long long any = __builtin_amdgcn_ballot_w64(bad);
    if (any && flag && (threadIdx.x & 63) == static_cast<unsigned>(__builtin_ctzll(any)))
        *reinterpret_cast<volatile unsigned *>(flag) = 1u;
}

// Smallest value over a wave (all lanes active), in a scalar register.
__device__ __forceinline__ int wave_min(int v) {
    for (int s = 32; s > 0; s >>= 1) v = min(v, __shfl_xor(v, s, 64));
    return __builtin_amdgcn_readfirstlane(v);
}

// The (x, y, z) workgroups of the rebin's grid (x: 256 output channels, y:
// row, z: kViews views), in dispatch order, taken in a stride of gridDim.x by
// the launched one-dimensional grid (fewer workgroups than the grid has: the
// rebin then leaves room on every CU for a kernel launched beside it).
template <class F>
__device__ __forceinline__ void for_each_block(const RebinArgs &a, F f) {
    const unsigned gx = static_cast<unsigned>(a.nos + 255) / 256u, gxy = gx * static_cast<unsigned>(a.n_rows);
    const unsigned total = gxy * static_cast<unsigned>((a.n_proj_out + kViews - 1) / kViews);
    for (unsigned vb = blockIdx.x; vb < total; vb += gridDim.x) {
        const unsigned bz = vb / gxy, rem = vb - bz * gxy, br = rem / gx;
        f(rem - br * gx, br, bz);
    }
}

// kHot: frames whose flag a.hot is set come from a.raw_af (the adaptive
// filter's output where it changed the frame), the others from the pull.
template <bool kHot>
__device__ __forceinline__ void rebin_block(const RebinArgs &a, unsigned bx, unsigned br, unsigned bz, bool &bad) {
    const int cl = static_cast<int>(bx) * 256 + static_cast<int>(threadIdx.x);
    const int c = min(cl, a.nos - 1);                   // (lanes past the row repeat its last channel, unstored)
    const bool store = cl < a.nos;
    const int r = static_cast<int>(br);
    // set of the row (kinds 1 and 3 interleave rows: set 0, the -dr focal
    // spot(s), -> row 2j, set 1 -> 2j + 1, swapped with ReverseRowInterleave)
    const bool inter = (a.kind & 1) != 0;
    const int set = inter ? (r & 1) ^ (a.reverse_rows ? 1 : 0) : 0;
    const int j = inter ? r >> 1 : r;
    // the two channel taps: raw channel, focal spot and azimuthal offset of
    // each (kinds 0 and 1: neighbouring raw channels of one spot; 2 and 3:
    // neighbouring oversampled channels, alternately of the set's two spots)
    const float by = a.bidx[set * a.nos + c];
    int t0, t1, ch0, ch1, fs0, fs1;
    float fc, ao0, ao1;
    if (a.kind <= 1) {
        taps(by, a.nch, t0, t1, fc);
        ch0 = t0;
        ch1 = t1;
        fs0 = fs1 = a.kind == 1 ? set : 0;
        ao0 = ao1 = a.aoff[set * a.nos + c];
    } else {
        taps(by, a.nos, t0, t1, fc);
        ch0 = t0 >> 1;
        ch1 = t1 >> 1;
        fs0 = 2 * set + (t0 & 1);
        fs1 = 2 * set + (t1 & 1);
        ao0 = a.aoff[set * a.nos + t0];
        ao1 = a.aoff[set * a.nos + t1];
    }
    const int v0 = static_cast<int>(bz) * kViews;
    const int n_v = min(kViews, a.n_proj_out - v0);
    // reading of the lower azimuthal tap at view v0
    const float fl0 = floorf(-ao0), fl1 = floorf(-ao1);
    const int p0 = v0 + a.add + static_cast<int>(fl0), p1 = v0 + a.add + static_cast<int>(fl1);
    const size_t frame = static_cast<size_t>(a.n_rows_raw) * a.nch;
    float *out = a.out + (static_cast<size_t>(v0) * a.n_rows + r) * a.nos;
    const size_t ostep = static_cast<size_t>(a.n_rows) * a.nos;
    const size_t step = static_cast<size_t>(a.n_ffs) * frame;       // samples from one reading of a spot to the next
    const int p_lo = wave_min(min(p0, p1)), p_hi = -wave_min(-max(p0, p1)) + n_v;
    // every reading inside the pull, and all of them (and the output rows)
    // within 32-bit byte offsets
    bool plain = p_lo >= 0 && p_hi < a.n_proj &&
                 static_cast<unsigned long long>(p_hi - p_lo + 1) * step < (1ull << 29) && kViews * ostep < (1ull << 29);
    if (kHot && plain) {
        // a wave whose readings the filter left alone reads the pull
        bool h = false;
        for (int f = p_lo * a.n_ffs + static_cast<int>(threadIdx.x & 63); f < (p_hi + 1) * a.n_ffs; f += 64)
            h |= a.hot[f] != 0;
        plain = __builtin_amdgcn_ballot_w64(h) == 0;
    }
    if (plain) {
        // Buffer accesses: descriptors over the readings p_lo .. p_hi and the
        // n_v output rows, constant 32-bit lane offsets, the view's step in
        // the scalar offset.  A lane past the row has an output offset past
        // the end and stores nothing.
        const unsigned step_b = static_cast<unsigned>(step) * 4u, ostep_b = static_cast<unsigned>(ostep) * 4u;
        const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(a.raw + static_cast<size_t>(p_lo) * step), static_cast<short>(0),
            static_cast<int>(static_cast<unsigned>(p_hi - p_lo + 1) * step_b), 0x00020000);
        const __amdgpu_buffer_rsrc_t dst = __builtin_amdgcn_make_buffer_rsrc(
            out, static_cast<short>(0), static_cast<int>(static_cast<unsigned>(n_v - 1) * ostep_b + a.nos * 4u),
            0x00020000);
        const unsigned fb = static_cast<unsigned>(frame) * 4u, jb = static_cast<unsigned>(j * a.nch) * 4u;
        const int o0 = static_cast<int>(static_cast<unsigned>((p0 - p_lo) * a.n_ffs + fs0) * fb + jb + static_cast<unsigned>(ch0) * 4u);
        const int o1 = static_cast<int>(static_cast<unsigned>((p1 - p_lo) * a.n_ffs + fs1) * fb + jb + static_cast<unsigned>(ch1) * 4u);
        const int oc = store ? c * 4 : static_cast<int>(0x80000000u);
        auto load = [&](int o, unsigned so) {
            return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src, o, static_cast<int>(so), 0));
        };
        float u0 = load(o0, 0), u1 = load(o1, 0);
        unsigned so = 0, oo = 0;
        float chk = 0.0f;           // NaN once an output is not finite
        float proj = static_cast<float>(v0 + a.add);
        auto view = [&](float w0, float w1) {
            // weight of the upper reading: the FP32 index proj - aoff less the
            // lower reading's number proj + floor(-aoff) (both steps exact but
            // for the index's own rounding)
            const float fa0 = (proj - ao0) - (proj + fl0), fa1 = (proj - ao1) - (proj + fl1);
            proj += 1.0f;
            const float x0 = fmaf(fa0, w0 - u0, u0), x1 = fmaf(fa1, w1 - u1, u1);
            float y = fmaf(fc, x1 - x0, x0);
            asm volatile("" : "+v"(y));     // one view after the other: no packing of several into wider registers
            u0 = w0;
            u1 = w1;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y), dst, oc, static_cast<int>(oo), 0);
            chk = fmaf(y, 0.0f, chk);
            oo += ostep_b;
        };
        int vv = 0;
#pragma unroll 1
        for (; vv + kBatch <= n_v; vv += kBatch) {
            float w0[kBatch], w1[kBatch];
#pragma unroll
            for (int e = 0; e < kBatch; e++) {
                so += step_b;
                w0[e] = load(o0, so);
                w1[e] = load(o1, so);
            }
            __builtin_amdgcn_sched_barrier(0);      // all of the batch's loads in flight
#pragma unroll
            for (int e = 0; e < kBatch; e++) view(w0[e], w1[e]);
        }
#pragma unroll 1
        for (; vv < n_v; vv++) {
            so += step_b;
            view(load(o0, so), load(o1, so));
        }
        bad |= chk != 0.0f;         // (true for NaN)
        return;
    }
    // readings clamped into the pull, each from its own source
    auto sample = [&](int p, int fs, int ch) {
        const size_t f = static_cast<size_t>(min(max(p, 0), a.n_proj - 1)) * a.n_ffs + fs;
        const float *s = kHot && a.hot[f] ? a.raw_af : a.raw;
        return s[f * frame + static_cast<size_t>(j) * a.nch + ch];
    };
    out += c;
    float u0 = sample(p0, fs0, ch0), u1 = sample(p1, fs1, ch1);
#pragma unroll 1
    for (int vv = 0; vv < n_v; vv++) {
        const float proj = static_cast<float>(v0 + a.add + vv);
        const float fa0 = (proj - ao0) - (proj + fl0), fa1 = (proj - ao1) - (proj + fl1);
        const float w0 = sample(p0 + vv + 1, fs0, ch0), w1 = sample(p1 + vv + 1, fs1, ch1);
        const float x0 = fmaf(fa0, w0 - u0, u0), x1 = fmaf(fa1, w1 - u1, u1);
        const float y = fmaf(fc, x1 - x0, x0);
        u0 = w0;
        u1 = w1;
        if (store) *out = y;
        bad |= !__builtin_isfinite(y);
        out += ostep;
    }
}

// One workgroup per (x, y, z) block of the grid.  Few registers: waves of it
// fit in the 64 per lane a running backprojection leaves.
template <bool kHot>
__global__ __launch_bounds__(256) void rebin_kernel(RebinArgs a) {
    bool bad = false;
    rebin_block<kHot>(a, blockIdx.x, blockIdx.y, blockIdx.z, bad);
    report_nonfinite(a.nonfinite, bad);
}

// A one-dimensional grid of RebinArgs::max_groups workgroups looping over the
// blocks.
template <bool kHot>
__global__ __launch_bounds__(256) void rebin_loop_kernel(RebinArgs a) {
    bool bad = false;
    for_each_block(a, [&](unsigned bx, unsigned br, unsigned bz) { rebin_block<kHot>(a, bx, br, bz, bad); });
    report_nonfinite(a.nonfinite, bad);
}

}  // namespace

int launch_rebin(const RebinArgs &a, hipStream_t stream) {
    if (!a.raw || !a.out || !a.bidx || !a.aoff || (a.hot && !a.raw_af)) return CTBB_ERR_ARG;
    if (a.kind < 0 || a.kind > 3 || a.nch <= 1 || a.nos != 2 * a.nch || a.n_proj < 2 || a.n_proj_out <= 0)
        return CTBB_ERR_SHAPE;
    if (a.add < 0 || a.add + a.n_proj_out > a.n_proj) return CTBB_ERR_SHAPE;
    const int rows_needed = (a.kind == 1 || a.kind == 3) ? 2 * a.n_rows_raw : a.n_rows_raw;
    if (a.n_rows != rows_needed) return CTBB_ERR_SHAPE;
    const dim3 grid((a.nos + 255) / 256, a.n_rows, (a.n_proj_out + kViews - 1) / kViews);
    if (grid.z > 65535u || grid.y > 65535u || a.max_groups < 0) return CTBB_ERR_SHAPE;
    const unsigned long long blocks = static_cast<unsigned long long>(grid.x) * grid.y * grid.z;
    const bool hot = a.hot != nullptr;
    if (a.max_groups > 0 && static_cast<unsigned long long>(a.max_groups) < blocks) {
        const dim3 g1(static_cast<unsigned>(a.max_groups));
        if (hot) hipLaunchKernelGGL(rebin_loop_kernel<true>, g1, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL(rebin_loop_kernel<false>, g1, dim3(256), 0, stream, a);
    } else if (hot) {
        hipLaunchKernelGGL(rebin_kernel<true>, grid, dim3(256), 0, stream, a);
    } else {
        hipLaunchKernelGGL(rebin_kernel<false>, grid, dim3(256), 0, stream, a);
    }
    return hipGetLastError() == hipSuccess ? CTBB_OK : CTBB_ERR_HIP;
}

}  // namespace ctbb
