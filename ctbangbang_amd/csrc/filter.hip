// Ramp / apodisation filter of rebinned rows as a Toeplitz matrix product on
// the CDNA4 matrix cores:
//     Y[m][l] = sum_k X[m][k] * taps[n + l - k]        (k, l in [0, n))
// which is the convolution of reference include/rebin_filter.cuh:369-409
// (and of the FFT form in src/rebin_filter_cpu.cu:647-709).
//
// The Toeplitz operand is never materialised: every workgroup keeps the 2n
// taps in LDS and forms the B fragments from them on the fly
// (B[k][l] = taps[n + l - k]).
//
// Variants (ctbb_filter_mode):
//   F32     v_mfma_f32_16x16x4_f32, FP32 operands, FP32 accumulation
//   BF16X3  v_mfma_f32_32x32x16_bf16 on hi/lo bfloat16 splits of both
//           operands: X*T ~= Xh*Th + Xh*Tl + Xl*Th, FP32 accumulation
//   F16X3   the same with float16 splits; taps are pre-scaled by 2^10 (and
//           the result by 2^-10) to keep the low parts out of the subnormals
//   FFT32   FP32 FFT convolution of 3072 or 4096 points (the form of the
//           reference's CPU path), for n <= 2048; wider rows fall back to F32
// Toeplitz tiles are 64 rows x 64 columns (F32) or 128 x 192 (split forms).  The
// split forms require n % 64 == 0 (1472 and 1344 for the 736- and 672-channel
// scanners); other widths take the F32 product, on the vector ALUs where
// n % 4 != 0.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace ctbb {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

constexpr int BM = 64, BN = 64, BK = 32;
constexpr int TAP_MARGIN = 64;     // >= BN - 4 columns past the row
constexpr int A_STRIDE = BK + 4;   // 36 floats: 16-byte aligned rows

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}

// FP32 Toeplitz product on v_mfma_f32_16x16x4_f32, n % 4 == 0 (the sums end with
// the row: a zero past it would bring in taps that a column does not have, NaN
// for infinite ones; columns past it are not stored).  One chain of sums in the order
// of the samples: a row's smooth part cancels from the far taps to the near ones,
// where chains over parts of the row keep the parts' large sums and their
// rounding (4x the largest error).  Matrix-core bound, 118 to
// 125 of the 153 TFLOP/s that a large FP32 matrix product reaches.
template <bool kEnd>
__global__ __launch_bounds__(256) void toeplitz_f32_kernel(FilterArgs a) {
    extern __shared__ float smem[];
    const int n = a.n;
    float *Tf = smem + 2 * BM * A_STRIDE;      // [2n] taps; kEnd: a margin of zeros behind them

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    const size_t m0 = static_cast<size_t>(blockIdx.y) * BM;
    const int n0 = blockIdx.x * BN;

    for (int j = tid; j < 2 * n + (kEnd ? TAP_MARGIN : 0); j += 256) Tf[j] = !kEnd || j < 2 * n ? a.taps[j] : 0.0f;

    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int lr = lane & 15, lk = lane >> 4;
    const int arow = tid >> 2, aseg = (tid & 3) * 8;
    const size_t gm = m0 + arow;
    const bool row_ok = gm < a.rows;
    const float *xrow = a.in + gm * n + aseg;
    f32x4 x0 = f32x4{0.f, 0.f, 0.f, 0.f}, x1 = x0;
    auto load = [&](int k0) {
        if (kEnd) x0 = x1 = f32x4{0.f, 0.f, 0.f, 0.f};
        if (row_ok && (!kEnd || k0 + aseg < n)) x0 = *reinterpret_cast<const f32x4 *>(xrow + k0);
        if (row_ok && (!kEnd || k0 + aseg + 4 < n)) x1 = *reinterpret_cast<const f32x4 *>(xrow + k0 + 4);
    };
    load(0);

    // two chunks in LDS in turn: one barrier per chunk
    auto chunk = [&](int k0) {
        float *As = smem + (k0 & BK) * (BM * A_STRIDE / BK);
        f32x4 *dst = reinterpret_cast<f32x4 *>(As + arow * A_STRIDE + aseg);
        dst[0] = x0;
        dst[1] = x1;
        __syncthreads();
        return As;
    };
    auto step = [&](const float *As, int k0, int kk) {
        float af[2], bfv[2];
#pragma unroll
        for (int rt = 0; rt < 2; rt++) af[rt] = As[(wr * 32 + rt * 16 + lr) * A_STRIDE + kk + lk];
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            const int col = n0 + wc * 32 + ct * 16 + lr;
            bfv[ct] = Tf[n + col - (k0 + kk + lk)];
        }
#pragma unroll
        for (int rt = 0; rt < 2; rt++)
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
                acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[rt], bfv[ct], acc[rt][ct], 0, 0, 0);
    };
    int k0 = 0;
    for (; k0 + BK <= n; k0 += BK) {
        const float *As = chunk(k0);
        // prefetch the next K chunk of this thread's row while the MFMAs run
        if (k0 + BK < n) load(k0 + BK);
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) step(As, k0, kk);
    }
    if (kEnd && k0 < n) {
        const float *As = chunk(k0);
        for (int kk = 0; k0 + kk < n; kk += 4) step(As, k0, kk);
    }

    // D layout of 16x16 MFMA tiles: lane l, register e -> row 4*(l/16)+e, column l%16
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
        for (int ct = 0; ct < 2; ct++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const size_t om = m0 + wr * 32 + rt * 16 + 4 * lk + e;
                const int col = n0 + wc * 32 + ct * 16 + lr;
                if (om < a.rows && (!kEnd || col < n)) {
                    const float y = acc[rt][ct][e];
                    if (a.out_bf16)
                        reinterpret_cast<uint16_t *>(a.out)[om * n + col] = f32_to_bf16_rne(y);
                    else
                        reinterpret_cast<float *>(a.out)[om * n + col] = y;
                }
            }
}

// Split-precision Toeplitz product: X = Xh + Xl and T = Th + Tl in bfloat16
// (MODE BF16X3) or float16 (MODE F16X3, taps scaled by 2^10 to keep the low
// parts out of the subnormals), accumulated in FP32 as Xl*Th + Xh*Tl + Xh*Th
// on gfx950's v_mfma_f32_32x32x16_{bf16,f16} (measured on MI355X at about
// 1.7x the rate of the 16x16x32 forms).  Workgroup = 128 rows x 32 CT columns;
// each wave owns 32 rows as CT = 6 tiles of 32 x 32, the three products of a
// k-step one after the other over the tiles, so that a tile's dependent MFMAs
// are six apart.
// The A operand goes straight from global memory into MFMA fragments: K is
// reduced in chunks of 32, and within a chunk lane l (half h = l / 32) holds
// k = 16 h + 8 s + e, e = 0..7, for k-step s, so its two A fragments are the
// 16 consecutive samples of its row (four float4 loads), split into hi/lo
// in registers once for all column tiles; the next chunk's loads are
// issued before the current chunk's MFMAs.  Only the reversed taps live in
// LDS (four copies shifted by 0..3 so that every B fragment, 8 consecutive
// reversed taps, is two 8-byte reads), written once, so the K loop has no
// barriers.  Columns past the row are not stored.  D layout (32 x 32): lane l,
// register r -> row 8 (r / 4) + 4 h + r % 4, column l % 32.  Workgroups are
// ordered so that the column tiles of a 128-row band run on the same XCD and
// share its L2 copy of the band.
// Bound by power: with random rows the clock falls to 1.5-1.9 GHz at 50% busy
// matrix cores, so what counts is the other work per MFMA.  Per wave tile, rows
// x columns, 119168 rows of 1344 in F16X3 / 30011 of 1472 in BF16X3: 64 x 64
// (each split operand used for 2 column tiles) 1.93 / 0.65 ms, 64 x 128 1.68 /
// 0.49, 32 x 192 1.49 / 0.47, 32 x 224 1.48 / 0.53, 32 x 256 1.73 / 0.55 (spills).
constexpr int SPLIT_TM = 128;                                   // rows of a workgroup
// taps of one shifted copy for 32 CT columns
__host__ __device__ constexpr int split_taps(int n, int CT) { return n + 32 * CT + 8; }

// CT column tiles per wave: 6, or fewer (launch_split).
template <int MODE, int CT>
__global__ __launch_bounds__(256, 2) void toeplitz_split_kernel(FilterArgs a, int n_rt, int n_ct) {
    constexpr int TM = SPLIT_TM, TN = 32 * CT, TK = 32;
    typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
    typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
    typedef short i16x8 __attribute__((ext_vector_type(8)));
    typedef float f32x16 __attribute__((ext_vector_type(16)));
    extern __shared__ uint16_t sh[];
    const int n = a.n;
    const int tw = split_taps(n, CT);             // taps per copy
    uint16_t *Gh = sh;                         // [4][tw]
    uint16_t *Gl = Gh + 4 * tw;                // [4][tw]

    int tile = blockIdx.x;
    const int n_tiles = n_rt * n_ct;
    if ((n_tiles & 7) == 0) tile = (blockIdx.x & 7) * (n_tiles >> 3) + (blockIdx.x >> 3);
    const int rt_i = tile / n_ct, ct_i = tile - rt_i * n_ct;
    const size_t m0 = static_cast<size_t>(rt_i) * TM;
    const int n0 = ct_i * TN;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, h = lane >> 5;
    const int jb = n - 1 - (n0 + TN - 1);      // first reversed-tap index this tile needs
    const float tscale = MODE == CTBB_FILTER_F16X3 ? 1024.0f : 1.0f;
    auto split = [&](float v, uint16_t &hi, uint16_t &lo) {
        if (MODE == CTBB_FILTER_BF16X3) {
            const __bf16 hb = static_cast<__bf16>(v);
            hi = __builtin_bit_cast(uint16_t, hb);
            lo = __builtin_bit_cast(uint16_t, static_cast<__bf16>(v - static_cast<float>(hb)));
        } else {
            const _Float16 hf = static_cast<_Float16>(v);
            hi = __builtin_bit_cast(uint16_t, hf);
            lo = __builtin_bit_cast(uint16_t, static_cast<_Float16>(v - static_cast<float>(hf)));
        }
    };
    for (int m = tid; m < tw + 3; m += 256) {
        const int j = jb + m;                 // reversed-tap index
        uint16_t hi, lo;
        split(j >= 0 && j < 2 * n ? a.taps[2 * n - 1 - j] * tscale : 0.0f, hi, lo);
#pragma unroll
        for (int s = 0; s < 4; s++)           // copy s holds it at m - s
            if (m >= s && m - s < tw) {
                Gh[s * tw + m - s] = hi;
                Gl[s * tw + m - s] = lo;
            }
    }
    __syncthreads();
    f32x16 acc[CT];
#pragma unroll
    for (int j = 0; j < CT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[j][r] = 0.0f;
    // fragment row of this lane; rows past the end read the last row (their
    // results are not stored)
    const size_t gm = m0 + wave * 32 + l32;
    const float *xrow = a.in + (gm < a.rows ? gm : a.rows - 1) * n + 16 * h;
    auto load = [&](float4 (&x)[4], int k0) {
#pragma unroll
        for (int q = 0; q < 4; q++) x[q] = *reinterpret_cast<const float4 *>(xrow + k0 + 4 * q);
    };
    auto mma = [&](const float4 (&x)[4], int k0) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const float4 u = x[2 * s], w = x[2 * s + 1];
            const float v[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
            i16x8 ah, al;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                uint16_t hi, lo;
                split(v[e], hi, lo);
                ah[e] = static_cast<short>(hi);
                al[e] = static_cast<short>(lo);
            }
            i16x8 bh[CT], bl[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                const int col = n0 + ct * 32 + l32;
                const int mm = (n - 1 - col + k0 + 16 * h + 8 * s) - jb;
                const int sft = mm & 3;
                const uint16_t *ph = Gh + sft * tw + (mm - sft);
                const uint16_t *pl = Gl + sft * tw + (mm - sft);
                const i16x4 h0 = *reinterpret_cast<const i16x4 *>(ph), h1 = *reinterpret_cast<const i16x4 *>(ph + 4);
                const i16x4 l0 = *reinterpret_cast<const i16x4 *>(pl), l1 = *reinterpret_cast<const i16x4 *>(pl + 4);
                bh[ct] = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
                bl[ct] = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
            }
#pragma unroll
            for (int p = 0; p < 3; p++)         // lo x hi, hi x lo, hi x hi
#pragma unroll
                for (int ct = 0; ct < CT; ct++) {
                    const i16x8 A = p == 0 ? al : ah, B = p == 1 ? bl[ct] : bh[ct];
                    if (MODE == CTBB_FILTER_BF16X3)
                        acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(bf16x8, A), __builtin_bit_cast(bf16x8, B), acc[ct], 0, 0, 0);
                    else
                        acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            __builtin_bit_cast(f16x8, A), __builtin_bit_cast(f16x8, B), acc[ct], 0, 0, 0);
                }
        }
    };
    // n % 64 == 0, so the chunks come in pairs
    float4 xa[4], xb[4];
    load(xa, 0);
    for (int k0 = 0; k0 < n; k0 += 2 * TK) {
        load(xb, k0 + TK);
        mma(xa, k0);
        if (k0 + 2 * TK < n) load(xa, k0 + 2 * TK);
        mma(xb, k0 + TK);
    }

    const float oscale = 1.0f / tscale;
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const size_t om = m0 + wave * 32 + 8 * (r / 4) + 4 * h + (r % 4);
            const int col = n0 + ct * 32 + l32;
            if (om < a.rows && col < n) {
                const float y = acc[ct][r] * oscale;
                if (a.out_bf16)
                    reinterpret_cast<uint16_t *>(a.out)[om * n + col] = f32_to_bf16_rne(y);
                else
                    reinterpret_cast<float *>(a.out)[om * n + col] = y;
            }
        }
}

// Direct FP32 convolution on the vector ALUs for widths that are not a
// multiple of 4: one workgroup per row, taps and row staged in LDS.
__global__ __launch_bounds__(256) void conv_valu_kernel(FilterArgs a) {
    extern __shared__ float smem[];
    const int n = a.n;
    float *xr = smem;          // [n]
    float *tp = smem + n;      // [2n]
    const size_t row = blockIdx.x;
    for (int j = threadIdx.x; j < 2 * n; j += blockDim.x) tp[j] = a.taps[j];
    for (int j = threadIdx.x; j < n; j += blockDim.x) xr[j] = a.in[row * n + j];
    __syncthreads();
    for (int l = threadIdx.x; l < n; l += blockDim.x) {
        float acc = 0.0f;
        for (int k = 0; k < n; k++) acc = fmaf(tp[n + l - k], xr[k], acc);
        if (a.out_bf16)
            reinterpret_cast<uint16_t *>(a.out)[row * n + l] = f32_to_bf16_rne(acc);
        else
            reinterpret_cast<float *>(a.out)[row * n + l] = acc;
    }
}

// ---------------------------------------------------------------------------
// FP32 FFT form of the same convolution (CTBB_FILTER_FFT32).
// Embedding: with L >= 2n and h[m] = taps[(m + n) mod L] (0 where that is >= 2n),
// the circular convolution y = x (*) h of the zero-padded row gives
// y[l] = sum_k x[k] taps[n + l - k] for l in [0, n) without wrap-around
// (n + l - k lies in [1, 2n - 1]).  Two rows a, b travel as one complex
// signal a + i b: h is real, so y = (a (*) h) + i (b (*) h).
// H = DFT_L(h) / L and the twiddles come from filter_spectrum_kernel, evaluated
// in FP64 and rounded once.  L = 3072 where 2n <= 3072 (the shipped scanners:
// 1472 and 1344 oversampled channels), else 4096.
// Transforms (Stockham, the passes in between through LDS; the inverse is
// conj(DFT(conj(Y)))):
//   L = 4096: radix 16, 16, 16, each pass 256 threads x 16 points;
//   L = 3072: forward radix 12, 16, 16 (256 threads x 12 points, then
//   192 x 16), the inverse in the reverse order 16, 16, 12, so each
//   transform starts from the layout the previous one ended in.
// Bound by VALU issue (and, over long runs, by the clock that the power leaves:
// 1.8 GHz), so the passes are built from few instructions:
//   - the upper half of the samples is zero and, with the taps turned by n, only
//     the lower half of the results is wanted: the first and the last pass leave
//     those out;
//   - constant twiddles are split into a factor and a vector with an entry of 1;
//     the factor becomes the multiplicand of additions that follow anyway;
//   - in each exchange the padding makes the address linear in the point's
//     number (a constant offset of the LDS instruction) and spreads the banks;
//   - rows are read and written through buffer descriptors of their length
//     (zeros past the end, no stores there).
// A pass's twiddles are w^r of one w per thread; w, w^2, w^4 and w^8 come from a
// table in the threads' order and the others are formed by products.  All
// fifteen from a table load 40% more data: 665 us where this takes 534.
// Butterflies of six FMAs (a - t b as 2a - (a + t b)) are as fast but add 25% to
// the rounding error.
// 119168 rows of 1472: 634 -> 534 us (1454 -> 1036 VALU instructions per wave),
// 60001 of 1344: 293 -> 245 us, 45001 of 1840: 265 -> 235 us; the traffic alone
// would take 290, 130 and 135 us.
constexpr int FFT_L = 4096;
constexpr int FFT_L3 = 3072;
constexpr size_t FFT_LDS3 = 13 * 256 * sizeof(float2);
// Twiddles of a pass of stride Ns and radix R: 4 x Ns entries w^(2^m), w = e^(-2
// pi i t / (Ns R)), t < Ns.  Their places in the table:
constexpr int TW_16 = 0, TW_256 = 64, TW_END = TW_256 + 4 * 256;                       // L = 4096
constexpr int TW3_12 = 0, TW3_16 = 48, TW3_192 = 112, TW3_256 = 880, TW3_END = 1904;   // L = 3072
constexpr float FFT_S3 = 0.86602540378443865f;   // sin(pi / 3)

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(fmaf(a.x, b.x, -a.y * b.y), fmaf(a.x, b.y, a.y * b.x));
}

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }

// in-place 4-point DFT, forward sign: X1 = a0 - i a1 - a2 + i a3
__device__ __forceinline__ void dft4(float2 &a0, float2 &a1, float2 &a2, float2 &a3) {
    const float2 s02 = cadd(a0, a2), d02 = csub(a0, a2), s13 = cadd(a1, a3), d13 = csub(a1, a3);
    a0 = cadd(s02, s13);
    a2 = csub(s02, s13);
    a1 = make_float2(d02.x + d13.y, d02.y - d13.x);
    a3 = make_float2(d02.x - d13.y, d02.y + d13.x);
}

// in-place 3-point DFT, forward sign: X1 = a0 + w a1 + w^2 a2, w = e^(-2 pi i / 3)
__device__ __forceinline__ void dft3(float2 &a0, float2 &a1, float2 &a2) {
    const float2 t = cadd(a1, a2);
    const float2 d = make_float2(FFT_S3 * (a1.x - a2.x), FFT_S3 * (a1.y - a2.y));
    const float2 c = make_float2(fmaf(-0.5f, t.x, a0.x), fmaf(-0.5f, t.y, a0.y));
    a0 = cadd(a0, t);
    a1 = make_float2(c.x + d.y, c.y - d.x);     // c - i d
    a2 = make_float2(c.x - d.y, c.y + d.x);     // c + i d
}

// v[r] *= w^r for r = 1 .. 15, from b[m] = w^(2^m), m = 0..3: the other
// powers are products of at most three of them (each product rounds once,
// so the twiddles stay within a few FP32 ulps of the table values).
// (R = 12: r = 1 .. 11 only)
template <int R = 16>
__device__ __forceinline__ void twiddle16(float2 (&v)[16], const float2 (&b)[4]) {
    static_assert(R == 12 || R == 16, "radix 12 or 16");
    const float2 w3 = cmul(b[1], b[0]);
    const float2 w5 = cmul(b[2], b[0]);
    const float2 w6 = cmul(b[2], b[1]);
    const float2 w7 = cmul(b[2], w3);
    v[1] = cmul(v[1], b[0]);
    v[2] = cmul(v[2], b[1]);
    v[3] = cmul(v[3], w3);
    v[4] = cmul(v[4], b[2]);
    v[5] = cmul(v[5], w5);
    v[6] = cmul(v[6], w6);
    v[7] = cmul(v[7], w7);
    v[8] = cmul(v[8], b[3]);
    v[9] = cmul(v[9], cmul(b[3], b[0]));
    v[10] = cmul(v[10], cmul(b[3], b[1]));
    v[11] = cmul(v[11], cmul(b[3], w3));
    if (R == 12) return;
    v[12] = cmul(v[12], cmul(b[3], b[2]));
    v[13] = cmul(v[13], cmul(b[3], w5));
    v[14] = cmul(v[14], cmul(b[3], w6));
    v[15] = cmul(v[15], cmul(b[3], w7));
}

// a (c - i s) for constants c and s, of which those of size 0 and 1 cost nothing
__device__ __forceinline__ float2 turn(float2 a, float c, float s) {
    auto mul2 = [](float x, float c, float y, float s) {
        if (s == 0.0f) return c == 1.0f ? x : c == -1.0f ? -x : c * x;
        if (c == 0.0f) return s == 1.0f ? y : s == -1.0f ? -y : s * y;
        if (c == 1.0f) return s == 1.0f ? x + y : s == -1.0f ? x - y : fmaf(s, y, x);
        if (c == -1.0f) return s == 1.0f ? y - x : s == -1.0f ? -x - y : fmaf(s, y, -x);
        if (s == 1.0f) return fmaf(c, x, y);
        return fmaf(c, x, -y);       // s == -1
    };
    return make_float2(mul2(a.x, c, a.y, s), mul2(a.y, c, a.x, -s));
}

// 4-point DFT of a0, f1 u1, f2 u2 and f1 u3 into a0, x1, x2, x3
__device__ __forceinline__ void dft4s(float2 &a0, float2 u1, float2 u2, float2 u3, float f2, float f1, float2 &x1,
                                      float2 &x2, float2 &x3) {
    const float2 s02 = make_float2(fmaf(f2, u2.x, a0.x), fmaf(f2, u2.y, a0.y));
    const float2 d02 = make_float2(fmaf(-f2, u2.x, a0.x), fmaf(-f2, u2.y, a0.y));
    const float2 s13 = make_float2(u1.x + u3.x, u1.y + u3.y), d13 = make_float2(u1.x - u3.x, u1.y - u3.y);
    a0 = make_float2(fmaf(f1, s13.x, s02.x), fmaf(f1, s13.y, s02.y));
    x2 = make_float2(fmaf(-f1, s13.x, s02.x), fmaf(-f1, s13.y, s02.y));
    x1 = make_float2(fmaf(f1, d13.y, d02.x), fmaf(-f1, d13.x, d02.y));
    x3 = make_float2(fmaf(-f1, d13.y, d02.x), fmaf(f1, d13.x, d02.y));
}

// the same with f3 = 1: a0, f1 u1, f2 u2, u3
__device__ __forceinline__ void dft4t(float2 &a0, float2 u1, float2 u2, float2 u3, float f2, float f1, float2 &x1,
                                      float2 &x2, float2 &x3) {
    const float2 s02 = make_float2(fmaf(f2, u2.x, a0.x), fmaf(f2, u2.y, a0.y));
    const float2 d02 = make_float2(fmaf(-f2, u2.x, a0.x), fmaf(-f2, u2.y, a0.y));
    const float2 s13 = make_float2(fmaf(f1, u1.x, u3.x), fmaf(f1, u1.y, u3.y));
    const float2 d13 = make_float2(fmaf(f1, u1.x, -u3.x), fmaf(f1, u1.y, -u3.y));
    a0 = make_float2(s02.x + s13.x, s02.y + s13.y);
    x2 = make_float2(s02.x - s13.x, s02.y - s13.y);
    x1 = make_float2(d02.x + d13.y, d02.y - d13.x);
    x3 = make_float2(d02.x - d13.y, d02.y + d13.x);
}

// 16-point DFT of w^r v[r] (kTw: w^(2^m) in b[m]; else w = 1) in natural order,
// as 4 x 4: inner DFTs over r2 (r = r1 + 4 r2), twiddles W16^(r1 k2), outer DFTs
// over r1; X[k2 + 4 k1] ends in slot k1 + 4 k2.  kHalfIn: v[8 .. 15] are taken as
// zero; kHalfOut: X[0 .. 7] only.
template <bool kTw, bool kHalfIn = false, bool kHalfOut = false>
__device__ __forceinline__ void fft16(float2 (&v)[16], const float2 (&b)[4]) {
    // cos(pi / 8), tan(pi / 8), sqrt(1 / 2)
    constexpr float C1 = 0.92387953251128674f, T1 = 0.41421356237309503f, H2 = 0.70710678118654757f;
    if (kTw) twiddle16(v, b);
#pragma unroll
    for (int r1 = 0; r1 < 4; r1++) {
        if (kHalfIn) {
            const float2 a = v[r1], c = v[r1 + 4];
            v[r1] = cadd(a, c);
            v[r1 + 8] = csub(a, c);
            v[r1 + 4] = make_float2(a.x + c.y, a.y - c.x);
            v[r1 + 12] = make_float2(a.x - c.y, a.y + c.x);
        } else {
            dft4(v[r1], v[r1 + 4], v[r1 + 8], v[r1 + 12]);
        }
    }
    // (W16^m = cos(pi m / 8) - i sin(pi m / 8), m = r1 k2)
    dft4(v[0], v[1], v[2], v[3]);
    dft4s(v[4], turn(v[5], 1.0f, T1), turn(v[6], 1.0f, 1.0f), turn(v[7], T1, 1.0f), H2, C1, v[5], v[6], v[7]);
    dft4s(v[8], turn(v[9], 1.0f, 1.0f), turn(v[10], 0.0f, 1.0f), turn(v[11], -1.0f, 1.0f), 1.0f, H2, v[9], v[10], v[11]);
    dft4s(v[12], turn(v[13], T1, 1.0f), turn(v[14], -1.0f, 1.0f), turn(v[15], -1.0f, -T1), H2, C1, v[13], v[14], v[15]);
    float2 o[16];
#pragma unroll
    for (int k = 0; k < (kHalfOut ? 8 : 16); k++) o[k] = v[(k >> 2) + 4 * (k & 3)];
#pragma unroll
    for (int k = 0; k < (kHalfOut ? 8 : 16); k++) v[k] = o[k];
}

// 12-point DFTs as 3 x 4: inner 3-point DFTs over r2 (r = r1 + 4 r2), twiddles
// W12^(r1 k2), outer 4-point DFTs over r1; X[k2 + 3 k1] ends in slot k1 + 4 k2.
// The part after the 3-point DFTs:
__device__ __forceinline__ void fft12_tail(float2 (&v)[16]) {
    constexpr float T3 = 0.57735026918962573f, R3 = 1.7320508075688772f;   // 1 / sqrt(3), sqrt(3)
    dft4(v[0], v[1], v[2], v[3]);
    dft4t(v[4], turn(v[5], 1.0f, T3), turn(v[6], 1.0f, R3), turn(v[7], 0.0f, 1.0f), 0.5f, FFT_S3, v[5], v[6], v[7]);
    dft4t(v[8], turn(v[9], 1.0f, R3), turn(v[10], -1.0f, R3), turn(v[11], -1.0f, 0.0f), 0.5f, 0.5f, v[9], v[10], v[11]);
    float2 o[12];
#pragma unroll
    for (int k = 0; k < 12; k++) o[k] = v[k / 3 + 4 * (k % 3)];
#pragma unroll
    for (int k = 0; k < 12; k++) v[k] = o[k];
}

// v[6 .. 11] are taken as zero
__device__ __forceinline__ void fft12_first(float2 (&v)[16]) {
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const float2 a0 = v[r], a1 = v[r + 4];
        const float2 m = make_float2(fmaf(-0.5f, a1.x, a0.x), fmaf(-0.5f, a1.y, a0.y));
        v[r] = make_float2(a0.x + a1.x, a0.y + a1.y);
        v[r + 4] = make_float2(fmaf(FFT_S3, a1.y, m.x), fmaf(-FFT_S3, a1.x, m.y));
        v[r + 8] = make_float2(fmaf(-FFT_S3, a1.y, m.x), fmaf(FFT_S3, a1.x, m.y));
    }
    v[6] = v[10] = v[2];
    v[7] = v[11] = v[3];
    fft12_tail(v);
}

// of w^r v[r], w^(2^m) in b[m]
__device__ __forceinline__ void fft12_last(float2 (&v)[16], const float2 (&b)[4]) {
    twiddle16<12>(v, b);
#pragma unroll
    for (int r1 = 0; r1 < 4; r1++) dft3(v[r1], v[r1 + 4], v[r1 + 8]);
    fft12_tail(v);
}

// Rows ra and ra + 1 as the parts of v[r] = x[j + 256 r], r < R; their R x 256
// samples cover the row.
template <int R>
__device__ __forceinline__ void fft_load(float2 (&v)[16], const FilterArgs &a, size_t ra, bool has_b, int j) {
    const __amdgpu_buffer_rsrc_t xa = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.in + ra * a.n), static_cast<short>(0), a.n * static_cast<int>(sizeof(float)), 0x00020000);
    const __amdgpu_buffer_rsrc_t xb =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.in + (ra + has_b) * a.n), static_cast<short>(0),
                                          has_b ? a.n * static_cast<int>(sizeof(float)) : 0, 0x00020000);
#pragma unroll
    for (int r = 0; r < R; r++) {
        v[r].x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xa, 4 * j + 1024 * r, 0, 0));
        v[r].y = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xb, 4 * j + 1024 * r, 0, 0));
    }
}

// the conjugates of v[r], r < R, as rows ra and ra + 1 of the result
template <int R>
__device__ __forceinline__ void fft_store(const float2 (&v)[16], const FilterArgs &a, size_t ra, bool has_b, int j) {
    const int es = a.out_bf16 ? 2 : 4;
    char *const out = reinterpret_cast<char *>(a.out);
    const __amdgpu_buffer_rsrc_t ya =
        __builtin_amdgcn_make_buffer_rsrc(out + ra * a.n * es, static_cast<short>(0), a.n * es, 0x00020000);
    const __amdgpu_buffer_rsrc_t yb = __builtin_amdgcn_make_buffer_rsrc(
        out + (ra + has_b) * a.n * es, static_cast<short>(0), has_b ? a.n * es : 0, 0x00020000);
    if (a.out_bf16) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16_rne(v[r].x), ya, 2 * j + 512 * r, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16_rne(-v[r].y), yb, 2 * j + 512 * r, 0, 0);
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[r].x), ya, 4 * j + 1024 * r, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(-v[r].y), yb, 4 * j + 1024 * r, 0, 0);
        }
    }
}

// v <- conj(v H): the inverse transform is conj(DFT(conj))
template <int STEP>
__device__ __forceinline__ void fft_apply(float2 (&v)[16], const float2 *__restrict__ H) {
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const float2 h = H[STEP * r];
        v[r] = make_float2(fmaf(v[r].x, h.x, -v[r].y * h.y), fmaf(-v[r].x, h.y, -v[r].y * h.x));
    }
}

// v[r] -> LDS -> v[r], all threads or those of the first three waves at either
// end: point r goes to `to` + S_TO r and comes from `from` + S_FROM r.
template <int S, int R>
__device__ __forceinline__ void fft_put(const float2 (&v)[16], float2 *to) {
#pragma unroll
    for (int r = 0; r < R; r++) to[S * r] = v[r];
}
template <int S, int R>
__device__ __forceinline__ void fft_get(float2 (&v)[16], const float2 *from) {
#pragma unroll
    for (int r = 0; r < R; r++) v[r] = from[S * r];
}

// A pass of radix R and stride Ns takes butterfly j from x[j + r L / R], turns
// it by w^r, w = e^(-2 pi i (j mod Ns) / (Ns R)), and leaves output r at (j / Ns)
// Ns R + j mod Ns + r Ns.  spec = [H (L)] followed by the twiddles; a pass's four
// powers of w are requested one pass ahead.
// One workgroup per pair of rows, 2n <= 3072.  64 registers (the compiler would
// take 74, no faster: its LDS is passed at the launch so that the bound of 8
// waves stands): the next block's filter runs beside a backprojection, which
// leaves 64 per lane, and takes the issue slots that it leaves idle, in place of
// following it.  512^2 volume of 7 blocks: 44.5 -> 43.3 ms.
__global__ __launch_bounds__(256, 8) void fft3072_filter_kernel(FilterArgs a) {
    extern __shared__ float2 sh2[];
    float2 *const sh = sh2;
    const int j = threadIdx.x;
    const bool act = j < 192;               // butterflies of the radix-16 passes
    const float2 *__restrict__ tw = a.spec + FFT_L3;
    const size_t ra = 2 * static_cast<size_t>(blockIdx.x);
    const bool has_b = ra + 1 < a.rows;
    float2 v[16], b[4];
    fft_load<6>(v, a, ra, has_b, j);
#pragma unroll
    for (int m = 0; m < 4; m++) b[m] = tw[TW3_12 + 12 * m + j % 12];
    fft12_first(v);                                     // R 12, Ns 1
    // point i at i + i / 12
    fft_put<1, 12>(v, sh + 13 * j);
    __syncthreads();
    if (act) {
        fft_get<208, 16>(v, sh + j + j / 12);
        fft16<true>(v, b);                              // R 16, Ns 12
#pragma unroll
        for (int m = 0; m < 4; m++) b[m] = tw[TW3_192 + 192 * m + j];
    }
    __syncthreads();
    // point i at i + 12 (i / 192)
    if (act) fft_put<12, 16>(v, sh + j / 12 * 204 + j % 12);
    __syncthreads();
    if (act) {
        fft_get<204, 16>(v, sh + j);
        fft16<true>(v, b);                              // R 16, Ns 192
        fft_apply<192>(v, a.spec + j);
#pragma unroll
        for (int m = 0; m < 4; m++) b[m] = tw[TW3_16 + 16 * m + (j & 15)];
        fft16<false>(v, b);                             // R 16, Ns 1
    }
    __syncthreads();
    // point i at i + i / 16
    if (act) fft_put<1, 16>(v, sh + 17 * j);
    __syncthreads();
    if (act) {
        fft_get<204, 16>(v, sh + j + (j >> 4));
        fft16<true>(v, b);                              // R 16, Ns 16
    }
#pragma unroll
    for (int m = 0; m < 4; m++) b[m] = tw[TW3_256 + 256 * m + j];
    __syncthreads();
    // point i at i + 16 (i / 256)
    if (act) fft_put<16, 16>(v, sh + (j >> 4) * 272 + (j & 15));
    __syncthreads();
    fft_get<272, 12>(v, sh + j);
    fft12_last(v, b);                                   // R 12, Ns 256
    fft_store<6>(v, a, ra, has_b, j);
}

// The same for 2n <= 4096.
__global__ __launch_bounds__(256) void fft4096_filter_kernel(FilterArgs a) {
    __shared__ float2 sh[17 * 256];
    const int j = threadIdx.x;
    const float2 *__restrict__ tw = a.spec + FFT_L;
    const size_t ra = 2 * static_cast<size_t>(blockIdx.x);
    const bool has_b = ra + 1 < a.rows;
    float2 v[16], b[4];
    fft_load<8>(v, a, ra, has_b, j);
    auto twiddles = [&](int NS, const float2 *T) {
#pragma unroll
        for (int m = 0; m < 4; m++) b[m] = T[NS * m];
    };
    // points i at i + i / 16, then at i + 16 (i / 256)
    float2 *const to1 = sh + 17 * j, *const to2 = sh + (j >> 4) * 272 + (j & 15);
    const float2 *const from1 = sh + j + (j >> 4), *const from2 = sh + j;
    twiddles(16, tw + TW_16 + (j & 15));
    fft16<false, true>(v, b);                           // Ns 1
    fft_put<1, 16>(v, to1);
    __syncthreads();
    fft_get<272, 16>(v, from1);
    fft16<true>(v, b);                                  // Ns 16
    twiddles(256, tw + TW_256 + j);
    __syncthreads();
    fft_put<16, 16>(v, to2);
    __syncthreads();
    fft_get<272, 16>(v, from2);
    fft16<true>(v, b);                                  // Ns 256
    fft_apply<256>(v, a.spec + j);
    twiddles(16, tw + TW_16 + (j & 15));
    fft16<false>(v, b);                                 // Ns 1
    __syncthreads();
    fft_put<1, 16>(v, to1);
    __syncthreads();
    fft_get<272, 16>(v, from1);
    fft16<true>(v, b);                                  // Ns 16
    twiddles(256, tw + TW_256 + j);
    __syncthreads();
    fft_put<16, 16>(v, to2);
    __syncthreads();
    fft_get<272, 16>(v, from2);
    fft16<true, false, true>(v, b);                     // Ns 256
    fft_store<8>(v, a, ra, has_b, j);
}

// Spectrum of the taps and twiddles of the FFT form: spec[k] = DFT_L(h)[k] / L
// (h: the taps zero-padded from `count` = 2n to L and turned by n), then
// the twiddles of the passes, evaluated in FP64 and rounded once.  The taps are real, so one wave takes
// bin k <= L / 2 and also writes bin L - k as its conjugate.  Each lane sums
// its taps m = lane, lane + 64, ... by Horner's rule in w^64 (w = e^(-2 pi i
// k / L), at most 64 steps: error far below FP32), times w^lane; 3072 x 2944
// products took 7.4 ms on a host core, with a copy of the taps back and an
// upload around them, and take 6.1 us here (8.2 us for 4096; bound by latency:
// 1537 waves of 46 dependent FP64 steps and three sine/cosine pairs; loading
// the taps one step at a time took 12 and 26 us).
constexpr int SPEC_WAVES = 4;

__global__ __launch_bounds__(64 * SPEC_WAVES) void filter_spectrum_kernel(const float *__restrict__ taps, int count,
                                                                          int L, float2 *__restrict__ spec) {
    const int lane = threadIdx.x & 63;
    const int k = blockIdx.x * SPEC_WAVES + (threadIdx.x >> 6);
    const int t = blockIdx.x * (64 * SPEC_WAVES) + threadIdx.x;
    double sn, cs;
    const bool l3 = L == FFT_L3;
    if (t < (l3 ? TW3_END : TW_END)) {
        const int from = l3 ? (t < TW3_16 ? TW3_12 : t < TW3_192 ? TW3_16 : t < TW3_256 ? TW3_192 : TW3_256)
                            : (t < TW_256 ? TW_16 : TW_256);
        const int ns = l3 ? (t < TW3_16 ? 12 : t < TW3_192 ? 16 : t < TW3_256 ? 192 : 256) : (t < TW_256 ? 16 : 256);
        const int rad = l3 && t >= TW3_256 ? 12 : 16, q = t - from;
        sincospi(-2.0 * ((q % ns) << (q / ns)) / (rad * ns), &sn, &cs);
        spec[L + t] = make_float2(static_cast<float>(cs), static_cast<float>(sn));
    }
    if (k > L / 2) return;
    // (products of indices reduced mod L: exact angles)
    sincospi(-2.0 * ((64 * k) % L) / L, &sn, &cs);
    // (the last group may be short; the others are loaded eight at a time,
    // ahead of the dependent products)
    const int last = (count - 1) >> 6;
    double re = 64 * last + lane < count ? static_cast<double>(taps[64 * last + lane]) : 0.0, im = 0.0;
    auto step = [&](float x) {
        const double nr = fma(re, cs, fma(-im, sn, static_cast<double>(x)));
        im = fma(re, sn, im * cs);
        re = nr;
    };
    int q = last - 1;
    for (; q >= 7; q -= 8) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = taps[64 * (q - e) + lane];
#pragma unroll
        for (int e = 0; e < 8; e++) step(x[e]);
    }
    for (; q >= 0; q--) step(taps[64 * q + lane]);
    sincospi(-2.0 * (k * (lane - count / 2) % L) / L, &sn, &cs);
    double hr = fma(re, cs, -im * sn), hi = fma(re, sn, im * cs);
    for (int s = 32; s > 0; s >>= 1) {
        hr += __shfl_xor(hr, s, 64);
        hi += __shfl_xor(hi, s, 64);
    }
    if (lane == 0) {
        const float fr = static_cast<float>(hr / L), fi = static_cast<float>(hi / L);
        spec[k] = make_float2(fr, fi);
        if (k > 0 && 2 * k < L) spec[L - k] = make_float2(fr, -fi);
    }
}

// widest rows that are no multiple of 64 channels (a row and its taps in 64 KB
// of LDS)
constexpr int CONV_MAX_N = 64 * 1024 / (3 * static_cast<int>(sizeof(float)));

template <int MODE, int CT>
int launch_split_ct(const FilterArgs &a, size_t lds, hipStream_t stream) {
    const size_t n_rt = (a.rows + SPLIT_TM - 1) / SPLIT_TM, n_ct = (static_cast<size_t>(a.n) + 32 * CT - 1) / (32 * CT);
    if (n_rt * n_ct > 0x7fffffffu) return CTBB_ERR_SHAPE;
    const void *kf = reinterpret_cast<const void *>(&toeplitz_split_kernel<MODE, CT>);
    if (lds > 65536 &&
        hipFuncSetAttribute(kf, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) != hipSuccess)
        return CTBB_ERR_SHAPE;
    hipLaunchKernelGGL((toeplitz_split_kernel<MODE, CT>), dim3(static_cast<unsigned>(n_rt * n_ct)), dim3(256), lds,
                       stream, a, static_cast<int>(n_rt), static_cast<int>(n_ct));
    return hipGetLastError() == hipSuccess ? CTBB_OK : CTBB_ERR_HIP;
}

template <int MODE>
int launch_split(const FilterArgs &a, hipStream_t stream) {
    int dev = 0, n_cu = 0, max_lds = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
        return CTBB_ERR_HIP;
    auto lds_of = [&](int ct) { return 8 * static_cast<size_t>(split_taps(a.n, ct)) * sizeof(uint16_t); };
    auto tiles = [&](size_t ct) { return (a.rows + SPLIT_TM - 1) / SPLIT_TM * ((a.n + 32 * ct - 1) / (32 * ct)); };
    // A workgroup's time hardly depends on the other CUs, so few rows take the
    // narrowest tile that one per CU still covers (rows of 1472, F16X3, us with
    // CT = 2 / 4 / 6: 128 rows 30 / 39 / 48, 1500 rows 48 / 43 / 52, 2600 rows
    // 57 / 53 / 59, 4000 rows 85 / 72 / 66, 20000 rows 384 / 303 / 277), as do rows
    // so wide (n > 10000) that the taps of six leave no room in LDS.
    const size_t room = static_cast<size_t>(max_lds), cus = static_cast<size_t>(n_cu);
    if (lds_of(2) > room) return CTBB_ERR_SHAPE;
    if (tiles(2) <= cus || lds_of(6) > room) return launch_split_ct<MODE, 2>(a, lds_of(2), stream);
    if (tiles(4) <= cus) return launch_split_ct<MODE, 4>(a, lds_of(4), stream);
    return launch_split_ct<MODE, 6>(a, lds_of(6), stream);
}

}  // namespace

int launch_filter_spectrum(const float *d_taps, int count, int L, float2 *d_spec, hipStream_t stream) {
    if (!d_taps || !d_spec || count <= 0 || count > L || (L != FFT_L && L != FFT_L3)) return CTBB_ERR_ARG;
    const unsigned grid = static_cast<unsigned>((L / 2 + 1 + SPEC_WAVES - 1) / SPEC_WAVES);
    // (grid * 256 threads >= L > TW_END, TW3_END: the twiddles are covered)
    hipLaunchKernelGGL(filter_spectrum_kernel, dim3(grid), dim3(64 * SPEC_WAVES), 0, stream, d_taps, count, L, d_spec);
    return hipGetLastError() == hipSuccess ? CTBB_OK : CTBB_ERR_HIP;
}

int launch_filter(const FilterArgs &a, hipStream_t stream) {
    if (!a.in || !a.out || !a.taps || a.n <= 0) return CTBB_ERR_ARG;
    if (a.rows == 0) return CTBB_OK;
    // (the spectrum's length a.fft_len: 3072 or 4096, 0 without one)
    const bool fft = a.mode == CTBB_FILTER_FFT32 && 2 * a.n <= FFT_L;
    const bool fft3 = fft && a.fft_len == FFT_L3 && 2 * a.n <= FFT_L3;
    if (fft && !fft3 && a.spec && a.fft_len != FFT_L) return CTBB_ERR_ARG;
    {
        // In place (out == in) only for the FFT kernel with FP32 output: each
        // of its workgroups reads its two rows completely before writing the
        // same two rows.  Narrower (bfloat16) output rows, an offset overlap,
        // or the tiled kernels (which read rows other workgroups write) would
        // race, so any other overlap is refused.
        const uintptr_t ib = reinterpret_cast<uintptr_t>(a.in), ob = reinterpret_cast<uintptr_t>(a.out);
        const uintptr_t ie = ib + a.rows * static_cast<size_t>(a.n) * sizeof(float);
        const uintptr_t oe = ob + a.rows * static_cast<size_t>(a.n) * (a.out_bf16 ? sizeof(uint16_t) : sizeof(float));
        if (ib < oe && ob < ie && !(fft && !a.out_bf16 && ib == ob)) return CTBB_ERR_ARG;
    }
    if (fft) {
        // grid.x is limited to 2^31 - 1
        if (!a.spec) return CTBB_ERR_ARG;
        const size_t n_pairs = (a.rows + 1) / 2;
        const size_t max_pairs = 0x7fffffffu;
        for (size_t p0 = 0; p0 < n_pairs; p0 += max_pairs) {
            FilterArgs s = a;
            const size_t np = n_pairs - p0 < max_pairs ? n_pairs - p0 : max_pairs;
            s.in = a.in + 2 * p0 * a.n;
            if (a.out_bf16) s.out = reinterpret_cast<uint16_t *>(a.out) + 2 * p0 * a.n;
            else s.out = reinterpret_cast<float *>(a.out) + 2 * p0 * a.n;
            s.rows = a.rows - 2 * p0 < 2 * np ? a.rows - 2 * p0 : 2 * np;
            if (fft3)
                hipLaunchKernelGGL(fft3072_filter_kernel, dim3(static_cast<unsigned>(np)), dim3(256), FFT_LDS3, stream, s);
            else
                hipLaunchKernelGGL(fft4096_filter_kernel, dim3(static_cast<unsigned>(np)), dim3(256), 0, stream, s);
            if (hipGetLastError() != hipSuccess) return CTBB_ERR_HIP;
        }
        return CTBB_OK;
    }
    // FFT32 with 2n > 4096 uses the FP32 Toeplitz product below
    // Split products on the double-K MFMAs.  Widths that are no multiple of 64
    // get FP32 products in every mode, on the matrix cores if the rows can be
    // read 16 bytes at a time (30000 rows of 1840: 1.67 ms, 10.7 ms on the
    // vector ALUs; 30000 of 36: 18 us, 30 us).
    if (a.mode == CTBB_FILTER_BF16X3 && a.n % 64 == 0) return launch_split<CTBB_FILTER_BF16X3>(a, stream);
    if (a.mode == CTBB_FILTER_F16X3 && a.n % 64 == 0) return launch_split<CTBB_FILTER_F16X3>(a, stream);
    if (a.n % 64 == 0 && a.mode != CTBB_FILTER_F32 && a.mode != CTBB_FILTER_FFT32) return CTBB_ERR_ARG;
    if (a.n % 64 != 0 && (a.n > CONV_MAX_N || a.rows > 0x7fffffffu)) return CTBB_ERR_SHAPE;
    if (a.n % 64 != 0 && (a.n % 4 != 0 || reinterpret_cast<uintptr_t>(a.in) % 16 != 0)) {
        const size_t lds = 3 * static_cast<size_t>(a.n) * sizeof(float);
        hipLaunchKernelGGL(conv_valu_kernel, dim3(static_cast<unsigned>(a.rows)), dim3(256), lds, stream, a);
        return hipGetLastError() == hipSuccess ? CTBB_OK : CTBB_ERR_HIP;
    }
    const size_t gy = (a.rows + BM - 1) / BM;
    // FP32 Toeplitz product (CTBB_FILTER_F32, and FFT32 rows wider than 2048)
    if ((BM * A_STRIDE + 2 * static_cast<size_t>(a.n)) * sizeof(float) > 64 * 1024) return CTBB_ERR_SHAPE;
    const bool end = a.n % 64 != 0;
    const size_t lds = (2 * BM * A_STRIDE + 2 * static_cast<size_t>(a.n) + (end ? TAP_MARGIN : 0)) * sizeof(float);
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute(end ? reinterpret_cast<const void *>(&toeplitz_f32_kernel<true>)
                                : reinterpret_cast<const void *>(&toeplitz_f32_kernel<false>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) != hipSuccess)
        return CTBB_ERR_SHAPE;
    // grid.y may exceed 65535 for very tall inputs: split into launches
    const size_t max_y = 65535;
    for (size_t y0 = 0; y0 < gy; y0 += max_y) {
        FilterArgs s = a;
        const size_t ny = (gy - y0 < max_y) ? gy - y0 : max_y;
        s.in = a.in + y0 * BM * a.n;
        if (a.out_bf16) s.out = reinterpret_cast<uint16_t *>(a.out) + y0 * BM * a.n;
        else s.out = reinterpret_cast<float *>(a.out) + y0 * BM * a.n;
        s.rows = a.rows - y0 * BM < ny * BM ? a.rows - y0 * BM : ny * BM;
        dim3 grid((a.n + BN - 1) / BN, static_cast<unsigned>(ny));
        if (end) hipLaunchKernelGGL(toeplitz_f32_kernel<true>, grid, dim3(256), lds, stream, s);
        else hipLaunchKernelGGL(toeplitz_f32_kernel<false>, grid, dim3(256), lds, stream, s);
        if (hipGetLastError() != hipSuccess) return CTBB_ERR_HIP;
    }
    return CTBB_OK;
}

}  // namespace ctbb
