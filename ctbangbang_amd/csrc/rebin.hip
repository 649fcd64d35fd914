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
// and any occupancy from 4 waves per SIMD up stay within 545-575 us: bound by
// the cache lines a gather touches (a wave's 64 channels lie on the rows of 14
// readings), 90-110 cycles per CU and wave of output.
constexpr int kViews = 16;
constexpr int kBatch = 4;
// azimuthal offset that puts every view before the first reading (a whole number)
constexpr float kFirstReading = 1073741824.0f;

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

// What an output channel of a row interpolates between.
struct Lane {
    int c, set, j;              // channel (clamped into the row), set and raw row
    bool store;                 // not past the row
    int ch0, ch1, fs0, fs1;     // raw channel and focal spot of the two taps
    float fc, ao0, ao1;         // weight of the upper tap, azimuthal offsets
};

__device__ __forceinline__ Lane lane_taps(const RebinArgs &a, unsigned bx, unsigned br) {
    Lane L;
    const int cl = static_cast<int>(bx) * 256 + static_cast<int>(threadIdx.x);
    L.c = min(cl, a.nos - 1);                           // (lanes past the row repeat its last channel, unstored)
    L.store = cl < a.nos;
    const int r = static_cast<int>(br);
    // set of the row (kinds 1 and 3 interleave rows: set 0, the -dr focal
    // spot(s), -> row 2j, set 1 -> 2j + 1, swapped with ReverseRowInterleave)
    const bool inter = (a.kind & 1) != 0;
    L.set = inter ? (r & 1) ^ (a.reverse_rows ? 1 : 0) : 0;
    L.j = inter ? r >> 1 : r;
    // the two channel taps: raw channel, focal spot and azimuthal offset of
    // each (kinds 0 and 1: neighbouring raw channels of one spot; 2 and 3:
    // neighbouring oversampled channels, alternately of the set's two spots)
    const float by = a.bidx[L.set * a.nos + L.c];
    int t0, t1;
    if (a.kind <= 1) {
        taps(by, a.nch, t0, t1, L.fc);
        L.ch0 = t0;
        L.ch1 = t1;
        L.fs0 = L.fs1 = a.kind == 1 ? L.set : 0;
        L.ao0 = L.ao1 = a.aoff[L.set * a.nos + L.c];
    } else {
        taps(by, a.nos, t0, t1, L.fc);
        L.ch0 = t0 >> 1;
        L.ch1 = t1 >> 1;
        L.fs0 = 2 * L.set + (t0 & 1);
        L.fs1 = 2 * L.set + (t1 & 1);
        L.ao0 = a.aoff[L.set * a.nos + t0];
        L.ao1 = a.aoff[L.set * a.nos + t1];
    }
    // A channel that no fan ray is parallel to (more than a radian off the central
    // one) has no offset: NaN, which as an index clamps to the first reading.
    if (L.ao0 != L.ao0) L.ao0 = kFirstReading;
    if (L.ao1 != L.ao1) L.ao1 = kFirstReading;
    return L;
}

// Views v0 .. v0 + kViews - 1 (to the end of the output) of the lane.
// kHot: frames whose flag a.hot is set come from a.raw_af (the adaptive
// filter's output where it changed the frame), the others from the pull.
template <bool kHot>
__device__ __forceinline__ void rebin_views(const RebinArgs &a, const Lane &L, unsigned br, int v0, bool &bad) {
    const int c = L.c, j = L.j, ch0 = L.ch0, ch1 = L.ch1, fs0 = L.fs0, fs1 = L.fs1, r = static_cast<int>(br);
    const bool store = L.store;
    const float fc = L.fc, ao0 = L.ao0, ao1 = L.ao1;
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

template <bool kHot>
__device__ __forceinline__ void rebin_block(const RebinArgs &a, unsigned bx, unsigned br, unsigned bz, bool &bad) {
    rebin_views<kHot>(a, lane_taps(a, bx, br), br, static_cast<int>(bz) * kViews, bad);
}

// One workgroup per (x, y, z) block of the grid, for frames from two sources.
__global__ __launch_bounds__(256) void rebin_hot_kernel(RebinArgs a) {
    bool bad = false;
    rebin_block<true>(a, blockIdx.x, blockIdx.y, blockIdx.z, bad);
    report_nonfinite(a.nonfinite, bad);
}

// The rebin with the chip to itself: a wave keeps the readings that its 64
// channels are at in LDS and loads each of them once, row by row, where a gather
// from memory touches the rows of all of them for every view.  Ring of 32
// readings x 32 channels per focal spot, and four more channels of each reading
// (64 output channels take 33 or 34 raw ones); in rows of 32 the channel alone
// decides a sample's bank, so lanes on different readings do not collide.  The
// readings come in chunks of 8: 8 views need three of them, and the next chunk is
// on its way into registers meanwhile.  Each wave has its own ring and runs
// without barriers.
// 1934 views of 64 rows x 1472 channels from four focal spots: 320 us, the copy
// rate for its 1.48 GB (551 us from memory); 1862 views of 1344 channels from two
// spots: 250 us (414).
constexpr int kRing = 32, kChunk = 8;
constexpr int kRingMain = kRing * 32, kRingMore = kRing * 4;       // floats per spot

template <int kSpots>
__global__ __launch_bounds__(256) void rebin_ring_kernel(RebinArgs a, int views) {
    // [wave][spot][reading][32 channels], [wave][spot][reading][4 channels]
    __shared__ __attribute__((aligned(4 * kRingMain))) float lds[4 * kSpots * (kRingMain + kRingMore)];
    bool bad = false;
    const unsigned br = blockIdx.y;
    const Lane L = lane_taps(a, blockIdx.x, br);
    const int v0 = static_cast<int>(blockIdx.z) * views, n_v = min(views, a.n_proj_out - v0);
    const float fl0 = floorf(-L.ao0), fl1 = floorf(-L.ao1);
    const int p0 = v0 + a.add + static_cast<int>(fl0), p1 = v0 + a.add + static_cast<int>(fl1);
    const int p_lo = wave_min(min(p0, p1)), span = -wave_min(-max(p0, p1)) - p_lo;
    const int c_lo = wave_min(min(L.ch0, L.ch1)), c_n = -wave_min(-max(L.ch0, L.ch1)) - c_lo + 1;
    const size_t frame = static_cast<size_t>(a.n_rows_raw) * a.nch, step = static_cast<size_t>(a.n_ffs) * frame;
    const size_t ostep = static_cast<size_t>(a.n_rows) * a.nos;
    // readings p_lo .. p_lo + np - 1, one more than the views use if their
    // number is odd (they are loaded in pairs)
    int np = span + n_v + 1;
    np += np & 1;
    // all inside the pull and (with the output rows) within 32-bit byte
    // offsets, and three chunks hold what 8 views use
    if (p_lo < 0 || p_lo + np > a.n_proj || span >= 2 * kChunk || c_n > 36 ||
        static_cast<unsigned long long>(np) * step >= (1ull << 29) ||
        static_cast<unsigned long long>(views) * ostep >= (1ull << 29)) {
        for (int vv = 0; vv < n_v; vv += kViews) rebin_views<false>(a, L, br, v0 + vv, bad);
        report_nonfinite(a.nonfinite, bad);
        return;
    }
    const unsigned step_b = static_cast<unsigned>(step) * 4u, ostep_b = static_cast<unsigned>(ostep) * 4u;
    const unsigned fb = static_cast<unsigned>(frame) * 4u;
    const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.raw + static_cast<size_t>(p_lo) * step), static_cast<short>(0),
        static_cast<int>(static_cast<unsigned>(np) * step_b), 0x00020000);
    const __amdgpu_buffer_rsrc_t dst = __builtin_amdgcn_make_buffer_rsrc(
        a.out + (static_cast<size_t>(v0) * a.n_rows + br) * a.nos, static_cast<short>(0),
        static_cast<int>(static_cast<unsigned>(n_v - 1) * ostep_b + a.nos * 4u), 0x00020000);
    // A chunk is loaded in pairs of readings of 32 channels, and 4 channels more
    // of all its readings (channels clamped into the row; readings past the last
    // one repeat it and are not used).
    const int l = static_cast<int>(threadIdx.x & 63);
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int ls = kSpots > 1 ? l >> 5 : 0;                         // spot of the lane's further channel
    const int fs = a.kind <= 1 ? L.set : 2 * L.set;                 // first of the spots (kind 0: set 0)
    const unsigned row_b = static_cast<unsigned>(fs) * fb + static_cast<unsigned>(L.j * a.nch) * 4u;
    const int o_main = static_cast<int>(row_b + static_cast<unsigned>(l >> 5) * step_b) + 4 * min(c_lo + (l & 31), a.nch - 1);
    const int o_more = static_cast<int>(row_b + static_cast<unsigned>(ls) * fb) + 4 * min(c_lo + 32 + (l & 3), a.nch - 1);
    constexpr int kMain = kSpots * kChunk / 2;
    auto load = [&](int chunk, float (&m)[kMain + 1]) {
        auto get = [&](int o, unsigned so) {
            return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src, o, static_cast<int>(so), 0));
        };
#pragma unroll
        for (int i = 0; i < kMain; i++)
            m[i] = get(o_main, static_cast<unsigned>(min(chunk * kChunk + 2 * (i % (kChunk / 2)), np - 2)) * step_b +
                                   i / (kChunk / 2) * fb);
        m[kMain] = get(o_more + static_cast<int>(static_cast<unsigned>(min(chunk * kChunk + ((l & 31) >> 2), np - 1)) * step_b), 0);
    };
    float *const ring = lds + wave * kSpots * kRingMain + l;
    float *const rest = lds + (4 * kSpots * kRingMain + (wave * kSpots + ls) * kRingMore + (l & 31));
    auto put = [&](int chunk, const float (&m)[kMain + 1]) {
        const int h = chunk & (kRing / kChunk - 1);
#pragma unroll
        for (int i = 0; i < kMain; i++)
            ring[i / (kChunk / 2) * kRingMain + h * 32 * kChunk + 64 * (i % (kChunk / 2))] = m[i];
        rest[h * 4 * kChunk] = m[kMain];
        // (a wave's LDS accesses keep their order)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    // LDS byte address of a tap's reading: up by a row per view, round in the ring
    const unsigned lds_b = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)lds;
    struct Tap {
        unsigned at, row, mask;
    };
    auto tap = [&](int ch, int f, int p) {
        const int cc = ch - c_lo, s = kSpots > 1 ? f - fs : 0;
        Tap t;
        t.row = cc < 32 ? 128u : 16u;
        t.mask = t.row * kRing - 1;
        t.at = lds_b + 4u * static_cast<unsigned>(cc < 32 ? (wave * kSpots + s) * kRingMain + cc
                                                          : 4 * kSpots * kRingMain + (wave * kSpots + s) * kRingMore + cc - 32) +
               static_cast<unsigned>(p - p_lo) * t.row;
        return t;
    };
    auto read = [](const Tap &t) { return *(const __attribute__((address_space(3))) float *)t.at; };
    auto next = [](Tap &t) {
        const unsigned n = t.at + t.row;
        t.at = (n & t.mask) | (t.at & ~t.mask);
    };
    float m[kMain + 1];
    {
        float m1[kMain + 1], m2[kMain + 1];
        load(0, m);
        load(1, m1);
        load(2, m2);
        __builtin_amdgcn_sched_barrier(0);
        put(0, m);
        put(1, m1);
        put(2, m2);
    }
    Tap t0 = tap(L.ch0, L.fs0, p0), t1 = tap(L.ch1, L.fs1, p1);
    const int oc = L.store ? L.c * 4 : static_cast<int>(0x80000000u);
    unsigned oo = 0;
    float chk = 0.0f;           // NaN once an output is not finite
    float proj = static_cast<float>(v0 + a.add);
    float u0 = read(t0), u1 = read(t1);
    auto view = [&](float w0, float w1) {
        // weight of the upper reading: the FP32 index proj - aoff less the
        // lower reading's number proj + floor(-aoff) (both steps exact but
        // for the index's own rounding)
        const float fa0 = (proj - L.ao0) - (proj + fl0), fa1 = kSpots == 1 ? fa0 : (proj - L.ao1) - (proj + fl1);
        proj += 1.0f;
        const float x0 = fmaf(fa0, w0 - u0, u0), x1 = fmaf(fa1, w1 - u1, u1);
        const float y = fmaf(L.fc, x1 - x0, x0);
        u0 = w0;
        u1 = w1;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y), dst, oc, static_cast<int>(oo), 0);
        chk = fmaf(y, 0.0f, chk);
        oo += ostep_b;
    };
#pragma unroll 1
    for (int b = 0; b * kChunk < n_v; b++) {
        const bool more = (b + 1) * kChunk < n_v;
        if (more) load(b + 3, m);
        __builtin_amdgcn_sched_barrier(0);
        if ((b + 1) * kChunk <= n_v) {
#pragma unroll
            for (int g = 0; g < kChunk; g += kBatch) {
                float w0[kBatch], w1[kBatch];
#pragma unroll
                for (int e = 0; e < kBatch; e++) {
                    next(t0);
                    w0[e] = read(t0);
                    next(t1);
                    w1[e] = read(t1);
                }
                __builtin_amdgcn_sched_barrier(0);      // all of the reads in flight
#pragma unroll
                for (int e = 0; e < kBatch; e++) view(w0[e], w1[e]);
            }
        } else {
#pragma unroll 1
            for (int vv = b * kChunk; vv < n_v; vv++) {
                next(t0);
                next(t1);
                view(read(t0), read(t1));
            }
        }
        if (more) put(b + 3, m);
    }
    bad |= chk != 0.0f;         // (true for NaN)
    report_nonfinite(a.nonfinite, bad);
}

// A one-dimensional grid of RebinArgs::max_groups workgroups looping over the
// blocks, from memory: in such a loop the ring takes 80 registers, and with its
// LDS one workgroup per CU fits beside a backprojection.
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
    const unsigned long long row_blocks = static_cast<unsigned long long>(grid.x) * grid.y;
    if (a.max_groups > 0 && static_cast<unsigned long long>(a.max_groups) < row_blocks * grid.z) {
        const dim3 g1(static_cast<unsigned>(a.max_groups));
        if (a.hot) hipLaunchKernelGGL(rebin_loop_kernel<true>, g1, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL(rebin_loop_kernel<false>, g1, dim3(256), 0, stream, a);
    } else if (a.hot) {
        hipLaunchKernelGGL(rebin_hot_kernel, grid, dim3(256), 0, stream, a);
    } else {
        // 64 views per wave, or 32 where those are fewer than 2048 workgroups, 8
        // per CU (64 rows of 1344 channels, 300 views: 30 us with 32, 33 with 64;
        // 600 views: 92 and 88)
        auto blocks_z = [&](int views) { return static_cast<unsigned>((a.n_proj_out + views - 1) / views); };
        const int views = row_blocks * blocks_z(64) < 2048 ? 32 : 64;
        const dim3 g(grid.x, grid.y, blocks_z(views));
        if (a.kind <= 1) hipLaunchKernelGGL(rebin_ring_kernel<1>, g, dim3(256), 0, stream, a, views);
        else hipLaunchKernelGGL(rebin_ring_kernel<2>, g, dim3(256), 0, stream, a, views);
    }
    return hipGetLastError() == hipSuccess ? CTBB_OK : CTBB_ERR_HIP;
}

}  // namespace ctbb
