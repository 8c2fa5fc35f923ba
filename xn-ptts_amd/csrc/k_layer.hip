// The rest of the flow-LM layer and the flow LM around it: LayerNorm, the q8 projection GEMM on
// MFMA with its epilogues, the f32 linears of batch-1 frames, and the row gathers.
#include "kernels_common.h"

#include <type_traits>

namespace xnp {

// ---------------------------------------------------------------------------------------------
// the rest of the flow-LM layer (transformer.rs:591-634): LayerNorm, and the q8 projections as
// MFMA GEMMs with per-channel int8 weights

// LayerNorm over rows of `dim` bf16 values (norm1, norm2: transformer.rs:547-548): one wave per
// row, each lane holding dim / 64 values; mean and biased variance in f32 (two passes over the
// registers), y = (x - mean) * (1 / sqrt(var + eps)) (* w + b when MODE has kLnAffine), rounded
// to bf16.  With kLnMod, then the AdaLN modulation (mlp.rs:4-11) as bf16 tensor operations round
// it: bf16(bf16(y * bf16(scale + 1)) + shift), with shift and scale bf16 rows of stride ld_mod.
constexpr int kLnAffine = 1, kLnMod = 2;

template <int CH, int MODE>
__global__ __launch_bounds__(256) void k_layer_norm(const uint16_t *x, int rows, int dim, const float *w,
                                                    const float *b, float eps, const uint16_t *shift,
                                                    const uint16_t *scale, int ld_mod, uint16_t *out) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    const uint16_t *xr = x + (size_t)row * dim;
    float v[CH][8];
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const uint4 raw = *(const uint4 *)(xr + (c * 64 + lane) * 8);
        const uint32_t *u = (const uint32_t *)&raw;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[c][2 * i] = bf16_value(u[i] & 0xffffu);
            v[c][2 * i + 1] = bf16_value(u[i] >> 16);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) sum += v[c][i];
    }
    uint4 rsh[CH], rsc[CH]; // the modulation's rows, loaded with x
    if constexpr ((MODE & kLnMod) != 0) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            rsh[c] = *(const uint4 *)(shift + (size_t)row * ld_mod + (c * 64 + lane) * 8);
            rsc[c] = *(const uint4 *)(scale + (size_t)row * ld_mod + (c * 64 + lane) * 8);
        }
    }
    float4 aw[CH][2], ab[CH][2]; // the affine's weights and biases, loaded with x too
    if constexpr ((MODE & kLnAffine) != 0) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int e0 = (c * 64 + lane) * 8;
            aw[c][0] = *(const float4 *)(w + e0);
            aw[c][1] = *(const float4 *)(w + e0 + 4);
            ab[c][0] = *(const float4 *)(b + e0);
            ab[c][1] = *(const float4 *)(b + e0 + 4);
        }
    }
    // a scheduling barrier: keeps the loads above here, issued together with x's, rather than
    // sunk to their uses after the row's reductions (a second round trip)
    __builtin_amdgcn_sched_barrier(0);
    sum = wave_sum(sum);
    const float mean = sum / (float)dim;
    float sq = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float d = v[c][i] - mean;
            sq = __builtin_fmaf(d, d, sq);
        }
    sq = wave_sum(sq);
    const float rstd = 1.0f / __builtin_sqrtf(sq / (float)dim + eps);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int e0 = (c * 64 + lane) * 8;
        float ww[8], bb[8];
        if constexpr ((MODE & kLnAffine) != 0) {
            const float4 w0 = aw[c][0], w1 = aw[c][1], b0 = ab[c][0], b1 = ab[c][1];
            const float wv[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
            const float bv[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) ww[i] = wv[i], bb[i] = bv[i];
        }
        uint32_t o4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float y[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int e = 2 * i + j;
                y[j] = (v[c][e] - mean) * rstd;
                if constexpr ((MODE & kLnAffine) != 0) y[j] = y[j] * ww[e] + bb[e];
                if constexpr ((MODE & kLnMod) != 0) {
                    const uint32_t us = ((const uint32_t *)&rsc[c])[i], uh = ((const uint32_t *)&rsh[c])[i];
                    const float sc1 = bf16_value(bf16_bits(bf16_value(j ? us >> 16 : us & 0xffffu) + 1.0f));
                    const float p = bf16_value(bf16_bits(bf16_value(bf16_bits(y[j])) * sc1));
                    y[j] = p + bf16_value(j ? uh >> 16 : uh & 0xffffu);
                }
            }
            o4[i] = pack_bf16(y[0], y[1]);
        }
        st_stream(out + (size_t)row * dim + e0, make_uint4(o4[0], o4[1], o4[2], o4[3]));
    }
}

template <int MODE>
static hipError_t layer_norm_mode(const void *x, int rows, int dim, const float *w, const float *b, float eps,
                                  const void *shift, const void *scale, int ld_mod, void *out, hipStream_t stream) {
    const dim3 grid((rows + 3) / 4), block(256);
    const uint16_t *xs = (const uint16_t *)x, *sh = (const uint16_t *)shift, *sc = (const uint16_t *)scale;
    uint16_t *o = (uint16_t *)out;
#define XNP_LN(C) hipLaunchKernelGGL((k_layer_norm<C, MODE>), grid, block, 0, stream, xs, rows, dim, w, b, eps, sh, sc, ld_mod, o)
    switch (dim / 512) {
    case 1: XNP_LN(1); break;
    case 2: XNP_LN(2); break;
    case 3: XNP_LN(3); break;
    case 4: XNP_LN(4); break;
    default: return hipErrorInvalidValue;
    }
#undef XNP_LN
    return hipGetLastError();
}

hipError_t launch_layer_norm_mod(const void *x, int rows, int dim, const float *w, const float *b, float eps,
                                 const void *shift, const void *scale, int ld_mod, void *out, hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    if (dim % 512 || (w == nullptr) != (b == nullptr) || (shift == nullptr) != (scale == nullptr) ||
        (shift && ld_mod % 8))
        return hipErrorInvalidValue;
    if (w && shift) return layer_norm_mode<kLnAffine | kLnMod>(x, rows, dim, w, b, eps, shift, scale, ld_mod, out, stream);
    if (w) return layer_norm_mode<kLnAffine>(x, rows, dim, w, b, eps, shift, scale, ld_mod, out, stream);
    if (shift) return layer_norm_mode<kLnMod>(x, rows, dim, w, b, eps, shift, scale, ld_mod, out, stream);
    return layer_norm_mode<0>(x, rows, dim, w, b, eps, shift, scale, ld_mod, out, stream);
}

hipError_t launch_layer_norm(const void *x, int rows, int dim, const float *w, const float *b, float eps, void *out,
                             hipStream_t stream) {
    return launch_layer_norm_mod(x, rows, dim, w, b, eps, nullptr, nullptr, 0, out, stream);
}

// gelu(y) = y Phi(y) for the bf16 epilogues (the erf form), from the tail Q(a) = 1 - Phi(a) = exp(-a^2 / 2)
// p(t), t = 1 / (1 + 0.3 a), p a polynomial of degree 8 fitted to exp(a^2 / 2) Q(a) (the scaled
// complementary error function) over a in [0, 13.5], 5.7e-8 relative at most; 17 VALU instructions in
// one path, where 0.5 y (1 + erff(y / sqrt 2)) took 38 (linear1 at 16384 rows: 20 of its 75 us).  For
// every finite bf16 y the result rounds to the bf16 nearest the exact value, but for -13.25 to -13.5, whose
// results are subnormal and whose exponential the hardware rounds to zero; the erff form, whose 1 + erff
// cancels on the negative side, missed it for 197.  Infinities and NaN as in the erff form.
__device__ __forceinline__ float gelu_erf(float y) {
    const float a = fminf(fabsf(y), 40.f);
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(a, 0.3f, 1.f));
    float p = 0.03833426907658577f;
    p = __builtin_fmaf(p, t, -0.16895195841789246f);
    p = __builtin_fmaf(p, t, 0.22821731865406036f);
    p = __builtin_fmaf(p, t, -0.07599961757659912f);
    p = __builtin_fmaf(p, t, 0.14218507707118988f);
    p = __builtin_fmaf(p, t, 0.09483297169208527f);
    p = __builtin_fmaf(p, t, 0.12188205868005753f);
    p = __builtin_fmaf(p, t, 0.11949305981397629f);
    p = __builtin_fmaf(p, t, 6.8529375312209595e-06f);
    const float q = p * fast_exp2(a * (a * -0.72134752f));
    return y * (y < 0.f ? q : 1.f - q);
}

// y = epilogue(s[n] * sum_k A[m][k] W[n][k]): A [M][K] bf16, W [N][K] int8 with one f32 scale per
// output channel (row of W), the sum on v_mfma_f32_16x16x32_bf16 with W widened to bf16 exactly
// (|q| <= 127).  One work group of 4 waves per 64 x 64 tile of y, each wave 32 x 32 (2 x 2 MFMA
// tiles); K in chunks of 64 staged through LDS, double-buffered, with the loads of the next three
// chunks in flight while one is multiplied.  The product, plus the bias when given, is rounded to bf16 (the
// projection's output tensor), then: kStore writes it (column ranges may go to separate outputs:
// q, k and v), kGelu* write gelu(y) rounded, kResidual adds y (times the layer scale, rounded,
// when given) into X and rounds: X + layer_scale(linear(..)) as transformer.rs:612-633 does; the
// flow net's epilogues are listed with their enum.  N may be any width (columns past N are
// neither loaded nor stored) and K any multiple of 16 (the last chunk's loads past K read zeros).
constexpr int kGmT = 64;  // tile rows and columns
constexpr int kGmK = 64;  // K chunk
constexpr int kGmLd = 72; // LDS row length in bf16
constexpr int kGmPD = 3;  // K chunks of loads in flight

// MI: 16-row MFMA tiles per wave in M, so tiles of 32 MI rows.  MI = 1 doubles the work groups of a
// narrow projection (N = 512 at 2048 rows gives 256 groups of 64 rows: one wave per SIMD).  MI = 4
// (128 x 64 tiles, each wave 64 x 32) for wide ones that still give two groups per CU: a wave's
// MFMAs per LDS byte read, and per staged byte, rise by a third.
//
// KS: groups of KS x 256 threads.  Half h (256 threads, the tile's 4 waves) takes K chunks h, h + KS,
// .. into its own LDS buffers; at the end half 1 hands its sums to half 0 through LDS, which adds
// them and runs the epilogue.  For long K (linear2: K = 2048), where a group's chunks run one
// after another.
// STG: the epilogue goes through LDS (N % 8 == 0, the outputs and their rows 16-byte aligned in
// 8-column steps): y, rounded to bf16, as [row][col], then a thread takes 8 consecutive columns of
// a row, so that its accesses to the output (and to x, the gate, aux) are 16 bytes (32 for f32
// rows) instead of 2, with its operands loaded before the K loop.  Measured in the layer step at
// 2048 rows: the epilogue took 2.4-3.1 us of each projection with 2-byte stores.
// NKC: K is exactly NKC x KS chunks (8 or 16 per half: the flow LM's 512-2048 wide projections),
// so the rounds run unrolled whole and without the past-K clamps and masks; 0: any K, in a loop.
// Tiles go to the XCDs in contiguous runs (xcd_tile), so each XCD's L2 holds about an eighth of A.

// The staged epilogue: a thread takes 8 consecutive columns of a row (y rounded to bf16), with the
// operands of that piece (epi_load) and of its columns (epi_cols), and writes 16 bytes (32 for f32 rows).
struct EpiPiece {
    uint4 x, gate; // kResidual, kGated: the output's old values; kGated: the gate
    float4 ax[2];  // kAxpyF32, kAddF32: the auxiliary row
};
struct EpiCols {
    float4 v[2]; // kResidual: the layer scale (ones without); kSiluAddVec: the vector
    char *out;   // row 0 of the output at these columns
    int ld;      // its row stride in values
};
template <int EPI> __device__ __forceinline__ void epi_load(const GemmOut &go, int m, int n, EpiPiece &p) {
    if constexpr (EPI == kResidual || EPI == kGated)
        p.x = *(const uint4 *)((const uint16_t *)go.out[0] + (size_t)m * go.ld[0] + n);
    if constexpr (EPI == kGated) p.gate = *(const uint4 *)((const uint16_t *)go.aux + (size_t)m * go.ld_aux + n);
    if constexpr (EPI == kAxpyF32 || EPI == kAddF32) {
        p.ax[0] = *(const float4 *)((const float *)go.aux + (size_t)m * go.ld_aux + n);
        p.ax[1] = *(const float4 *)((const float *)go.aux + (size_t)m * go.ld_aux + n + 4);
    }
}
template <int EPI> __device__ __forceinline__ void epi_cols(const GemmOut &go, int n, EpiCols &c) {
    constexpr int ES = EPI == kAxpyF32 || EPI == kStoreF32 ? 4 : 2;
    c.out = (char *)go.out[0] + (size_t)n * ES;
    c.ld = go.ld[0];
    if constexpr (EPI == kStore) { // constant indices: the kernel's arguments stay scalars
        if (go.nseg > 1 && n >= go.col0[1]) c.out = (char *)go.out[1] + (size_t)(n - go.col0[1]) * ES, c.ld = go.ld[1];
        if (go.nseg > 2 && n >= go.col0[2]) c.out = (char *)go.out[2] + (size_t)(n - go.col0[2]) * ES, c.ld = go.ld[2];
    }
    if constexpr (EPI == kResidual) {
        c.v[0] = c.v[1] = make_float4(1.f, 1.f, 1.f, 1.f);
        if (go.ls) {
            c.v[0] = *(const float4 *)(go.ls + n);
            c.v[1] = *(const float4 *)(go.ls + n + 4);
        }
    }
    if constexpr (EPI == kSiluAddVec) {
        c.v[0] = *(const float4 *)((const float *)go.aux + n);
        c.v[1] = *(const float4 *)((const float *)go.aux + n + 4);
    }
}
// one value: y to the output value, i its place in the piece
template <int EPI>
__device__ __forceinline__ float epi_value(float y, int i, const EpiPiece &p, const EpiCols &c, const GemmOut &go) {
    const uint32_t *xw = (const uint32_t *)&p.x, *gw = (const uint32_t *)&p.gate;
    const float *ax = (const float *)&p.ax[0], *cv = (const float *)&c.v[0];
    if constexpr (EPI == kGeluErf) {
        return gelu_erf(y);
    } else if constexpr (EPI == kGeluTanh) {
        const float cc = 0.7978845608028654f;
        return 0.5f * y * (1.0f + tanhf(cc * (y + 0.044715f * y * y * y)));
    } else if constexpr (EPI == kResidual) {
        const float a = go.ls ? bf16_value(bf16_bits(y * cv[i])) : y;
        return bf16_value((i & 1) ? xw[i >> 1] >> 16 : xw[i >> 1] & 0xffffu) + a;
    } else if constexpr (EPI == kSilu) {
        return y / (1.0f + expf(-y));
    } else if constexpr (EPI == kSiluAddVec) {
        const float z = bf16_value(bf16_bits(y + cv[i]));
        return z / (1.0f + expf(-z));
    } else if constexpr (EPI == kGated) {
        const float gate = bf16_value((i & 1) ? gw[i >> 1] >> 16 : gw[i >> 1] & 0xffffu);
        return bf16_value((i & 1) ? xw[i >> 1] >> 16 : xw[i >> 1] & 0xffffu) + bf16_value(bf16_bits(gate * y));
    } else if constexpr (EPI == kAxpyF32) {
        return bf16_value(bf16_bits(bf16_value(bf16_bits(ax[i])) + bf16_value(bf16_bits(y * go.alpha))));
    } else if constexpr (EPI == kAddF32) {
        return bf16_value(bf16_bits(ax[i])) + y;
    } else { // kStore, kStoreF32
        return y;
    }
}
// the piece's 8 output values to row m
template <int EPI> __device__ __forceinline__ void epi_write(const float (&r)[8], int m, const EpiCols &c) {
    if constexpr (EPI == kAxpyF32 || EPI == kStoreF32) {
        float *o = (float *)c.out + (size_t)m * c.ld;
        *(float4 *)o = make_float4(r[0], r[1], r[2], r[3]);
        *(float4 *)(o + 4) = make_float4(r[4], r[5], r[6], r[7]);
    } else {
        st_stream((uint16_t *)c.out + (size_t)m * c.ld,
                  make_uint4(pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3]), pack_bf16(r[4], r[5]), pack_bf16(r[6], r[7])));
    }
}
__device__ __forceinline__ float epi_y(const uint4 &yv, int i) { // value i of the staged y
    const uint32_t u = ((const uint32_t *)&yv)[i >> 1];
    return bf16_value((i & 1) ? u >> 16 : u & 0xffffu);
}
template <int EPI>
__device__ __forceinline__ void epi_store(const GemmOut &go, int m, const uint4 &yv, const EpiPiece &p, const EpiCols &c) {
    float r[8];
    if (EPI == kResidual && !go.ls) { // apart, so that the scaled form is not computed beside it
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = epi_y(p.x, i) + epi_y(yv, i);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = epi_value<EPI>(epi_y(yv, i), i, p, c, go);
    }
    epi_write<EPI>(r, m, c);
}

template <int EPI, bool AF32, int MI, int NI, int KS, bool STG, int NKC>
__global__ __launch_bounds__(256 * KS, NI > 2 ? 2 : 1) void k_gemm_q8(const uint16_t *A, int M, int K, const int8_t *W, const float *s,
                                                      int N, GemmOut go) {
    constexpr int BM = 32 * MI, BN = 32 * NI;
    constexpr int KC = kGmK, LD = kGmLd; // K chunk, LDS row length in bf16
    // K chunks of loads in flight (a wide tile's round is twice as long; its registers are full)
    constexpr int PD = NI > 2 ? 2 : kGmPD;
    static_assert(NI == 2 || STG, "wide tiles come with the staged epilogue");
    static_assert(KS == 1 || KS == 2, "one or two halves");
    struct Tiles {
        uint16_t A[KS][2][BM][LD], W[KS][2][BN][LD];
    };
    __shared__ __attribute__((aligned(16))) Tiles smem;
    auto &As = smem.A;
    auto &Ws = smem.W;
    const int ntn = (N + BN - 1) / BN, tile = xcd_tile(blockIdx.x, gridDim.x);
    const int m0 = (tile / ntn) * BM, n0 = (tile % ntn) * BN;
    const int tid = threadIdx.x & 255, h = KS > 1 ? (int)(threadIdx.x >> 8) : 0;
    const int w = tid >> 6, lane = tid & 63, g = lane >> 4, l16 = lane & 15;
    const int wm = w & 1, wn = w >> 1;

    // staging: A rows a_r + RA i (the tile's 32 MI rows), 8 values at k 8 a_k; W rows w_r + RW i,
    // 16 int8 at k 16 w_k.
    // PD chunks of loads are in flight: set c % PD holds chunk c from its load until it is
    // written to LDS.  The words stay as loaded until then -- zeroing past K, rounding f32 A rows
    // and widening W happen at the LDS store, since any use at the load would make the wave wait
    // for it there.
    constexpr int UA = KC / 8, UW = KC / 16, RA = 256 / UA, RW = 256 / UW; // pieces a row, rows a pass
    constexpr int NA = BM / RA, NW = BN / RW;                                // A and W rows a thread stages
    const int a_r = tid / UA, a_k = tid % UA, w_r = tid / UW, w_k = tid % UW;
    int ar[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) ar[i] = min(m0 + a_r + RA * i, M - 1);
    int wr[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) wr[i] = min(n0 + w_r + RW * i, N - 1);
    constexpr int AW = AF32 ? 2 : 1; // uint4 per 8 A values
    uint4 ra[NA][PD][AW], rw[NW][PD];
    // NKC > 0: K is a whole number of chunks, so nothing reaches past it and the clamps and masks
    // below drop out (they were 14-18 of a round's 47-51 VALU instructions)
    constexpr bool kWhole = NKC > 0;
    auto load = [&](int kc, int set) {
        // past K (K % 16 == 0, so no 16-byte load straddles it): an in-bounds address, zeroed at
        // the store
        const int k0 = kc * KC;
        const int ka = kWhole || k0 + 8 * a_k < K ? k0 + 8 * a_k : 0, kw = kWhole || k0 + 16 * w_k < K ? k0 + 16 * w_k : 0;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            if constexpr (AF32) {
                const float *af = (const float *)A;
                ra[i][set][0] = *(const uint4 *)(af + (size_t)ar[i] * K + ka);
                ra[i][set][AW - 1] = *(const uint4 *)(af + (size_t)ar[i] * K + ka + 4);
            } else {
                ra[i][set][0] = *(const uint4 *)(A + (size_t)ar[i] * K + ka);
            }
        }
#pragma unroll
        for (int i = 0; i < NW; ++i) rw[i][set] = *(const uint4 *)(W + (size_t)wr[i] * K + kw);
    };
    auto masked = [](const uint4 &u, uint32_t m) { return make_uint4(u.x & m, u.y & m, u.z & m, u.w & m); };
    auto bf16_row = [&](const uint4 (&u)[AW]) { // 8 A values as bf16 pairs
        if constexpr (AF32) {
            return make_uint4(pack_bf16(__uint_as_float(u[0].x), __uint_as_float(u[0].y)),
                              pack_bf16(__uint_as_float(u[0].z), __uint_as_float(u[0].w)),
                              pack_bf16(__uint_as_float(u[AW - 1].x), __uint_as_float(u[AW - 1].y)),
                              pack_bf16(__uint_as_float(u[AW - 1].z), __uint_as_float(u[AW - 1].w)));
        } else {
            return u[0];
        }
    };
    auto widen2 = [](uint32_t u, int sh) { // two int8 -> a bf16 pair (exact: |q| <= 127)
        return pack_bf16((float)(int8_t)((u >> sh) & 0xffu), (float)(int8_t)((u >> (sh + 8)) & 0xffu));
    };
    auto store = [&](int buf, int set, int kc) {
        uint4 av[NA], wq[NW];
#pragma unroll
        for (int i = 0; i < NW; ++i) wq[i] = rw[i][set];
#pragma unroll
        for (int i = 0; i < NA; ++i) av[i] = bf16_row(ra[i][set]);
        // words past K zeroed with masks rather than under a branch: a branch here splits the
        // loop, and past the join the compiler no longer knows which loads are still in flight
        // (it then waits for all of them before the next load)
        if constexpr (!kWhole) {
            const int k0 = kc * KC;
            const uint32_t ma = k0 + 8 * a_k < K ? ~0u : 0u, mw = k0 + 16 * w_k < K ? ~0u : 0u;
#pragma unroll
            for (int i = 0; i < NA; ++i) av[i] = masked(av[i], ma);
#pragma unroll
            for (int i = 0; i < NW; ++i) wq[i] = masked(wq[i], mw);
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) *(uint4 *)&As[h][buf][a_r + RA * i][8 * a_k] = av[i];
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const uint4 q = wq[i];
            uint16_t *ws = &Ws[h][buf][w_r + RW * i][16 * w_k];
            *(uint4 *)ws = make_uint4(widen2(q.x, 0), widen2(q.x, 16), widen2(q.y, 0), widen2(q.y, 16));
            *(uint4 *)(ws + 8) = make_uint4(widen2(q.z, 0), widen2(q.z, 16), widen2(q.w, 0), widen2(q.w, 16));
        }
    };

    // the epilogue's per-column operands, loaded before the loop so that they arrive with it
    float sc[NI], bn[NI], lsn[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
        const int n = min(n0 + 16 * NI * wn + 16 * ni + l16, N - 1);
        sc[ni] = s[n];
        bn[ni] = go.bias ? go.bias[n] : 0.f;
        lsn[ni] = (EPI == kResidual && go.ls) ? go.ls[n] : 1.f;
    }

    // the staged epilogue's pieces (rows er + ER e, columns n0 + ec ..) and their operands (wide tiles:
    // loaded after the K loop, whose registers they would take)
    constexpr int PR = BN / 8, ER = 256 / PR, NE = BM / ER; // pieces a row, rows a pass, passes
    const int er = tid / PR, ec = 8 * (tid % PR), ne = n0 + ec;
    EpiPiece piece[NE];
    auto operands = [&] {
        if (h == 0) {
#pragma unroll
            for (int e = 0; e < NE; ++e) epi_load<EPI>(go, min(m0 + er + ER * e, M - 1), ne < N ? ne : 0, piece[e]);
        }
    };
    EpiCols cols;
    if constexpr (STG) epi_cols<EPI>(go, ne < N ? ne : 0, cols);
    if constexpr (STG && NI == 2) operands();

    f32x4_t acc[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // this half's chunks: c = 0 .. nkh - 1 is chunk h + KS c.  Both halves run nkmax rounds, one
    // barrier each, whatever their own count (the launcher takes KS = 2 only when nk >= 2 KS).
    // Every round loads and stores unconditionally, past this half's last chunk its last chunk
    // again (a duplicate nobody reads): loads under a branch leave the compiler unsure which loads
    // are in flight after it, and it then drains them all before the next one.  NKC > 0: K is
    // NKC x KS chunks exactly, and the rounds are unrolled whole -- the back edge of a loop makes
    // the compiler copy load registers still in flight, which waits for them.
    const int nk = NKC > 0 ? NKC * KS : (K + KC - 1) / KC;
    const int nkh = NKC > 0 ? NKC : (nk - h + KS - 1) / KS, nkmax = NKC > 0 ? NKC : (nk + KS - 1) / KS;
    auto chunk = [&](int c) { return h + KS * min(c, nkh - 1); };
    auto round = [&](int c, int u) { // u = c % PD: set indices stay constants
        const int buf = c & 1;
        load(chunk(c + PD), u); // set u held chunk c, already in LDS
        if (c < nkh) {
#pragma unroll
            for (int ks = 0; ks < KC / 32; ++ks) {
                bf16x8_t a[MI], bw[NI];
#pragma unroll
                for (int i = 0; i < MI; ++i)
                    a[i] = as_bf16x8(*(const uint4 *)&As[h][buf][16 * MI * wm + 16 * i + l16][32 * ks + 8 * g]);
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    bw[i] = as_bf16x8(*(const uint4 *)&Ws[h][buf][16 * NI * wn + 16 * i + l16][32 * ks + 8 * g]);
#pragma unroll
                for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                    for (int ni = 0; ni < NI; ++ni)
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mi], bw[ni], acc[mi][ni], 0, 0, 0);
            }
        }
        // buffer buf ^ 1's last readers finished before the previous barrier
        store(buf ^ 1, (u + 1) % PD, chunk(c + 1));
        __syncthreads();
    };
#pragma unroll
    for (int c = 0; c < PD; ++c) load(chunk(c), c);
    store(0, 0, h);
    __syncthreads();
    if constexpr (NKC > 0) {
#pragma unroll
        for (int c = 0; c < NKC; ++c) round(c, c % PD);
    } else {
        for (int cb = 0; cb < nkmax; cb += PD) {
#pragma unroll
            for (int u = 0; u < PD; ++u) {
                if (cb + u >= nkmax) break; // uniform over the group
                round(cb + u, u);
            }
        }
    }
    if constexpr (KS > 1) {
        // half 1's sums to half 0 through LDS (the tiles are free: every half passed the loop's
        // last barrier after its last read); half 0 adds them, in the same order in every group
        static_assert(sizeof(smem) >= 256 * MI * NI * 4 * sizeof(float), "room for half 1's sums");
        float *red = (float *)&smem;
        if (h == 1) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                    for (int r = 0; r < 4; ++r) red[((mi * NI + ni) * 4 + r) * 256 + tid] = acc[mi][ni][r];
        }
        __syncthreads();
        if (!STG && h == 1) return;
        if (h == 0) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[mi][ni][r] += red[((mi * NI + ni) * 4 + r) * 256 + tid];
        }
    }

    if constexpr (STG) {
        // y into LDS (lane: column 16 NI wn + 16 ni + l16, rows 16 MI wm + 16 mi + 4 g + r); both halves
        // meet at the barriers, half 1 with nothing to store
        constexpr int kGsLd = BN + 8; // the staged epilogue's LDS row in bf16
        static_assert(sizeof(smem) >= BM * kGsLd * sizeof(uint16_t), "room for the tile");
        uint16_t(*st)[kGsLd] = (uint16_t(*)[kGsLd]) & smem;
        if constexpr (NI > 2) operands();
        if constexpr (KS > 1) __syncthreads(); // half 0 has read half 1's sums
        if (h == 0) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float v = go.bias ? acc[mi][ni][r] * sc[ni] + bn[ni] : acc[mi][ni][r] * sc[ni];
                        st[16 * MI * wm + 16 * mi + 4 * g + r][16 * NI * wn + 16 * ni + l16] = (uint16_t)bf16_bits(v);
                    }
        }
        __syncthreads();
        if (h != 0) return;
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const int m = m0 + er + ER * e;
            if (m >= M || ne >= N) continue;
            epi_store<EPI>(go, m, *(const uint4 *)&st[er + ER * e][ec], piece[e], cols);
        }
        return;
    }

    // lane: column n0 + 16 NI wn + 16 ni + l16, rows m0 + 16 MI wm + 16 mi + 4 g + r
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
        const int n = n0 + 16 * NI * wn + 16 * ni + l16;
        if (n >= N) continue;
        int seg = 0;
        if constexpr (EPI == kStore) {
            if (go.nseg > 1 && n >= go.col0[1]) seg = (go.nseg > 2 && n >= go.col0[2]) ? 2 : 1;
        }
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + 16 * MI * wm + 16 * mi + 4 * g + r;
                if (m >= M) continue;
                const float y = bf16_value(bf16_bits(go.bias ? acc[mi][ni][r] * sc[ni] + bn[ni] : acc[mi][ni][r] * sc[ni]));
                if constexpr (EPI == kStore) {
                    ((uint16_t *)go.out[seg])[(size_t)m * go.ld[seg] + (n - go.col0[seg])] = (uint16_t)bf16_bits(y);
                } else if constexpr (EPI == kGeluErf || EPI == kGeluTanh) {
                    float gv;
                    if constexpr (EPI == kGeluErf) {
                        gv = gelu_erf(y);
                    } else {
                        const float c = 0.7978845608028654f;
                        gv = 0.5f * y * (1.0f + tanhf(c * (y + 0.044715f * y * y * y)));
                    }
                    ((uint16_t *)go.out[0])[(size_t)m * go.ld[0] + n] = (uint16_t)bf16_bits(gv);
                } else if constexpr (EPI == kResidual) {
                    const float a = go.ls ? bf16_value(bf16_bits(y * lsn[ni])) : y;
                    uint16_t *xp = (uint16_t *)go.out[0] + (size_t)m * go.ld[0] + n;
                    *xp = (uint16_t)bf16_bits(bf16_value(*xp) + a);
                } else if constexpr (EPI == kSilu) {
                    ((uint16_t *)go.out[0])[(size_t)m * go.ld[0] + n] = (uint16_t)bf16_bits(y / (1.0f + expf(-y)));
                } else if constexpr (EPI == kSiluAddVec) {
                    const float z = bf16_value(bf16_bits(y + ((const float *)go.aux)[n]));
                    ((uint16_t *)go.out[0])[(size_t)m * go.ld[0] + n] = (uint16_t)bf16_bits(z / (1.0f + expf(-z)));
                } else if constexpr (EPI == kGated) {
                    const float gate = bf16_value(((const uint16_t *)go.aux)[(size_t)m * go.ld_aux + n]);
                    uint16_t *xp = (uint16_t *)go.out[0] + (size_t)m * go.ld[0] + n;
                    *xp = (uint16_t)bf16_bits(bf16_value(*xp) + bf16_value(bf16_bits(gate * y)));
                } else if constexpr (EPI == kAxpyF32) {
                    const float cur = bf16_value(bf16_bits(((const float *)go.aux)[(size_t)m * go.ld_aux + n]));
                    ((float *)go.out[0])[(size_t)m * go.ld[0] + n] =
                        bf16_value(bf16_bits(cur + bf16_value(bf16_bits(y * go.alpha))));
                } else if constexpr (EPI == kAddF32) {
                    const float c = bf16_value(bf16_bits(((const float *)go.aux)[(size_t)m * go.ld_aux + n]));
                    ((uint16_t *)go.out[0])[(size_t)m * go.ld[0] + n] = (uint16_t)bf16_bits(c + y);
                } else { // kStoreF32
                    ((float *)go.out[0])[(size_t)m * go.ld[0] + n] = y;
                }
            }
    }
}

// The same product for K = 512 and many rows, with W in registers: one work group of 8 waves per CU
// holds 256 columns of W for a run of 32-row tiles, each wave 32 columns over all of K as the 32 A
// operands of v_mfma_f32_32x32x16_bf16 (128 registers, widened once).  The rows stream through a
// ring of 3 LDS slots (32 KB, loaded straight into LDS two tiles ahead), and a wave's inner loop is one
// 16-byte LDS read per MFMA: k_gemm_q8's tiles pay a barrier, the W widening and an LDS round trip of
// both operands per 64 k, and no unit of theirs was busy half the time (16384 rows, qkv: MFMA 28 %, LDS
// 50 %, VALU 32 %), whatever their size or prefetch.  16384 rows: qkv 48.7 (128 x 64 tiles), 41 (128 x 128),
// here 31.5 us (818 TFLOP/s); linear1 with its GELU 83, 65, 51.4 us, bound by the GELU's VALU work.
//
// The k order is the same for both operands and otherwise free: lane (col, hi) of W loads 16
// consecutive k (32 j + 16 hi ..), its halves the operands of steps 2 j and 2 j + 1, so row unit (8 k)
// 4 j + 2 hi + b is read at step 2 j + b.  Units sit at unit ^ (row & 15): a read's 8 rows fall in
// distinct banks, and a row of a tile is one 1 KB load.
// D = W A^T holds, per lane, row l % 32 and columns 8 (r / 4) + 4 (l / 32) + r % 4: rounded to bf16 they
// go through LDS as [row][col], and 8 columns a thread leave by the staged epilogue one tile later.
constexpr int kWrK = 512, kWrRows = 32, kWrCols = 256, kWrSlots = 3;

template <int EPI>
__global__ __launch_bounds__(512, 2) void k_gemm_q8_wres(const uint16_t *A, int M, const int8_t *W, const float *s, int N,
                                                         GemmOut go, int per) {
    __shared__ __attribute__((aligned(16))) uint16_t As[kWrSlots][kWrRows][kWrK];
    __shared__ __attribute__((aligned(16))) uint16_t st[2][kWrRows][kWrCols + 8]; // rows 16 bytes further apart in banks
    const int ntn = (N + kWrCols - 1) / kWrCols, tile = xcd_tile(blockIdx.x, gridDim.x);
    const int n0 = tile % ntn * kWrCols, t0 = tile / ntn * per, t1 = min(t0 + per, (M + kWrRows - 1) / kWrRows);
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, hi = lane >> 5, col = lane & 31;
    const uint32_t as_at = lds_addr(&As[0][0][0]);
    // tile t's rows 4 w .. 4 w + 3 into slot: lane l's 16 bytes are unit l ^ (row & 15) of the row
    auto issue = [&](int t, int slot) {
        const int ln = lane_here(lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 4 * w + i, m = min(t * kWrRows + row, M - 1);
            dma16_at(A + (size_t)m * kWrK + 8 * (ln ^ (row & 15)), as_at + (uint32_t)((slot * kWrRows + row) * kWrK * 2));
        }
    };
    // W, then the first two tiles behind it
    const int nw = n0 + 32 * w; // the wave's columns
    bf16x8_t wf[32];
    {
        const int8_t *wr = W + (size_t)min(nw + col, N - 1) * kWrK + 16 * hi;
        uint4 raw[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) raw[j] = *(const uint4 *)(wr + 32 * j);
        __builtin_amdgcn_sched_barrier(0);
        issue(t0, 0);
        if (t0 + 1 < t1) issue(t0 + 1, 1);
        auto widen2 = [](uint32_t u, int sh) { // two int8 -> a bf16 pair (exact: |q| <= 127)
            return pack_bf16((float)(int8_t)((u >> sh) & 0xffu), (float)(int8_t)((u >> (sh + 8)) & 0xffu));
        };
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            wf[2 * j] = as_bf16x8(make_uint4(widen2(raw[j].x, 0), widen2(raw[j].x, 16), widen2(raw[j].y, 0), widen2(raw[j].y, 16)));
            wf[2 * j + 1] = as_bf16x8(make_uint4(widen2(raw[j].z, 0), widen2(raw[j].z, 16), widen2(raw[j].w, 0), widen2(raw[j].w, 16)));
        }
    }
    float sc[16], bn[16]; // of columns nw + 8 (r / 4) + 4 hi + r % 4
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int n = min(nw + 8 * (r >> 2) + 4 * hi + (r & 3), N - 1);
        sc[r] = s[n];
        bn[r] = go.bias ? go.bias[n] : 0.f;
    }
    // the pieces this thread stores: rows er and er + 16, 8 columns.  Past the last row or column the
    // last one again, bit for bit what its own thread stores: no branch parts the products below
    const int er = tid >> 5, ne = min(n0 + 8 * (tid & 31), N - 8), ec = ne - n0;
    static_assert(EPI == kStore || EPI == kGeluErf || EPI == kGeluTanh, "epilogues without operands of their own");
    EpiCols cols;
    epi_cols<EPI>(go, ne, cols);
    auto row_of = [&](int t, int e) { return min(t * kWrRows + er + 16 * e, M - 1); };
    auto store_tile = [&](int t) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int m = row_of(t, e);
            epi_store<EPI>(go, m, *(const uint4 *)&st[t & 1][m - t * kWrRows][ec], EpiPiece(), cols);
        }
    };
    // the lane's LDS offsets within a slot for steps 0 .. 7 (steps 8 i + .. lie 256 i bytes further: a
    // row's units 16 i .. keep their place in 16s)
    uint32_t aofs[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) aofs[k] = col * (kWrK * 2) + 16 * ((4 * (k >> 1) + 2 * hi + (k & 1)) ^ (col & 15));
    constexpr int FD = 6; // LDS reads ahead
    auto tile_body = [&](int t, int slot, auto FIRST) {
        // this lane's loads of tile t have landed: tile t + 1's 4 went out after them, last of all (the
        // stores of the iteration before are older)
        if (t + 1 < t1)
            asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        else
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier(); // tile t is in LDS; every wave is done with tile t - 1's slot and has staged its outputs
        const char *base = (const char *)&As[slot][0][0];
        auto frag = [&](int k) { return as_bf16x8(*(const uint4 *)(base + aofs[k & 7] + 256 * (k >> 3))); };
        f32x16_t acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
        bf16x8_t f[FD];
#pragma unroll
        for (int k = 0; k < FD; ++k) f[k] = frag(k);
        uint4 yv[2];
        float o8[8];
        if constexpr (!decltype(FIRST)::value) {
#pragma unroll
            for (int e = 0; e < 2; ++e) yv[e] = *(const uint4 *)&st[(t - 1) & 1][row_of(t - 1, e) - (t - 1) * kWrRows][ec];
        }
        // FD LDS reads stay ahead of the products, one issued after each, and the previous tile's outputs
        // are finished a value a product and leave between them: the waves of a SIMD are in the same
        // phase (one barrier a tile), so nothing else would run beside the matrix pipe.  The scheduling
        // barriers hold that order (VALU instructions may cross them); left alone, the compiler reads
        // each operand right before its product, an LDS round trip each.
#pragma unroll
        for (int k = 0; k < 32; ++k) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[k], f[k % FD], acc, 0, 0, 0);
            if (k + FD < 32) f[k % FD] = frag(k + FD);
            __builtin_amdgcn_sched_barrier(0x6);
            if constexpr (!decltype(FIRST)::value) {
                if (k >= 4 && k < 20) {
                    const int e = (k - 4) >> 3, i = (k - 4) & 7;
                    o8[i] = epi_value<EPI>(epi_y(yv[e], i), i, EpiPiece(), cols, go);
                    if (i == 7) epi_write<EPI>(o8, row_of(t - 1, e), cols);
                }
            }
            if (k == 21 && t + 2 < t1) issue(t + 2, slot == 0 ? 2 : slot - 1);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float y[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = acc[4 * q + r] * sc[4 * q + r] + bn[4 * q + r];
            *(uint2 *)&st[t & 1][col][32 * w + 8 * q + 4 * hi] = make_uint2(pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3]));
        }
    };
    tile_body(t0, 0, std::true_type{});
    int slot = 1;
    for (int t = t0 + 1; t < t1; ++t) {
        tile_body(t, slot, std::false_type{});
        slot = slot == 2 ? 0 : slot + 1;
    }
    lds_barrier();
    store_tile(t1 - 1);
}

// The same product for few rows (K of 512, 1024 or 2048), with a LayerNorm of the rows in front when
// LNM is not 0 (K = 512; LNM - 1 is k_layer_norm's MODE).  At these sizes a launch is a chain of round
// trips, not work: k_gemm_q8 stages K chunk by chunk and the LayerNorm was a launch of its own.  Here one
// work group of 8 waves takes 16 MT rows x 32 columns, wave w the K slice from w K / 8, and loads its
// whole share of A and W at once, straight into the MFMA's operand layout (lane (l16, g): row or column
// l16, 16 consecutive k from 64 i + 16 g, whose halves are the operands of two products; the k order is
// the same for both).  D = W A^T (lane: row l16, columns 4 g + r) goes to LDS, the waves' shares are
// added in k order, y leaves by the staged epilogue.
//
// The LayerNorm is k_layer_norm's to the bit: its lane j holds k 8 j .. + 7, here the two halves of
// lane (l16, g) of wave w (j = 8 w + 2 g, + 1), and its reduction pairs j over bits 0, 1, .. 5: the
// halves, g's two bits by row swaps, the waves' three through LDS.  (Rows and both sides' times: the
// rule at gemm_small.)
struct LnIn {
    const float *w = nullptr, *b = nullptr;
    float eps = 1e-5f;
    const uint16_t *shift = nullptr, *scale = nullptr;
    int ld_mod = 0;
};

template <int EPI, int NS, int MT, int LNM>
__global__ __launch_bounds__(512) void k_gemm_q8_small(const uint16_t *A, int M, const int8_t *W, const float *s, int N,
                                                       GemmOut go, LnIn ln) {
    static_assert(LNM == 0 || NS == 1, "the LayerNorm takes rows of 512");
    constexpr int K = 512 * NS, MODE = LNM - 1;
    __shared__ __attribute__((aligned(16))) float red[8][16 * MT][36];
    __shared__ __attribute__((aligned(16))) uint16_t yt[16 * MT][40];
    __shared__ float mom[2][8][16 * MT];
    // row tiles fastest: an XCD's run of groups shares its columns of W
    const int mts = (M + 16 * MT - 1) / (16 * MT), tile = xcd_tile(blockIdx.x, gridDim.x);
    const int m0 = tile % mts * (16 * MT), n0 = tile / mts * 32;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 4, l16 = lane & 15;
    const int k0 = 64 * NS * w + 16 * g;
    uint4 wr[2][NS], ar[MT][NS][2];
#pragma unroll
    for (int i = 0; i < NS; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) wr[j][i] = *(const uint4 *)(W + (size_t)min(n0 + 16 * j + l16, N - 1) * K + k0 + 64 * i);
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int b = 0; b < 2; ++b)
                ar[j][i][b] = *(const uint4 *)(A + (size_t)min(m0 + 16 * j + l16, M - 1) * K + k0 + 64 * i + 8 * b);
    }
    float4 aw[4], ab[4];
    uint4 rsh[MT][2], rsc[MT][2];
    if constexpr (LNM > 0) {
        if constexpr ((MODE & kLnAffine) != 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                aw[i] = *(const float4 *)(ln.w + k0 + 4 * i);
                ab[i] = *(const float4 *)(ln.b + k0 + 4 * i);
            }
        }
        if constexpr ((MODE & kLnMod) != 0) {
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const size_t o = (size_t)min(m0 + 16 * j + l16, M - 1) * ln.ld_mod + k0 + 8 * b;
                    rsh[j][b] = *(const uint4 *)(ln.shift + o);
                    rsc[j][b] = *(const uint4 *)(ln.scale + o);
                }
        }
    }
    // what the tail needs: this thread's sum is row tid / 32 (+ 16 j), column tid % 32; the first 64 MT
    // threads store 8 columns of a row
    const int sn = min(n0 + (tid & 31), N - 1);
    const float sc = s[sn], bn = go.bias ? go.bias[sn] : 0.f;
    const int er = tid >> 2, ec = 8 * (tid & 3), em = m0 + er, ne = n0 + ec;
    const bool mine = tid < 64 * MT && em < M && ne < N;
    EpiPiece piece;
    EpiCols cols;
    if (mine) {
        epi_load<EPI>(go, em, ne, piece);
        epi_cols<EPI>(go, ne, cols);
    }
    __builtin_amdgcn_sched_barrier(0); // the loads above go out together

    if constexpr (LNM > 0) {
        float v[MT][2][8];
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < 8; ++i) v[j][b][i] = epi_y(ar[j][0][b], i);
        auto moment = [&](float (&p)[MT], int which) {
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                p[j] = swap_sum<32>(swap_sum<16>(p[j]));
                if (g == 0) mom[which][w][16 * j + l16] = p[j];
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                float q[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) q[i] = mom[which][i][16 * j + l16];
                p[j] = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
            }
        };
        float sum[MT], sq[MT];
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            float p[2] = {0.f, 0.f};
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < 8; ++i) p[b] += v[j][b][i];
            sum[j] = p[0] + p[1];
        }
        moment(sum, 0);
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            sum[j] = sum[j] / (float)K; // the mean
            float p[2] = {0.f, 0.f};
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float d = v[j][b][i] - sum[j];
                    p[b] = __builtin_fmaf(d, d, p[b]);
                }
            sq[j] = p[0] + p[1];
        }
        moment(sq, 1);
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const float rstd = 1.0f / __builtin_sqrtf(sq[j] / (float)K + ln.eps);
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                float y[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    y[i] = (v[j][b][i] - sum[j]) * rstd;
                    if constexpr ((MODE & kLnAffine) != 0)
                        y[i] = y[i] * ((const float *)&aw[2 * b])[i] + ((const float *)&ab[2 * b])[i];
                    if constexpr ((MODE & kLnMod) != 0) {
                        const float sc1 = bf16_value(bf16_bits(epi_y(rsc[j][b], i) + 1.0f));
                        y[i] = bf16_value(bf16_bits(bf16_value(bf16_bits(y[i])) * sc1)) + epi_y(rsh[j][b], i);
                    }
                }
                ar[j][0][b] = make_uint4(pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3]), pack_bf16(y[4], y[5]), pack_bf16(y[6], y[7]));
            }
        }
    }
    f32x4_t acc[MT][2];
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[j][0] = acc[j][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto widen4 = [](uint32_t a, uint32_t b) { // 8 int8 -> bf16 (exact: |q| <= 127)
        auto two = [](uint32_t u, int sh) {
            return pack_bf16((float)(int8_t)((u >> sh) & 0xffu), (float)(int8_t)((u >> (sh + 8)) & 0xffu));
        };
        return as_bf16x8(make_uint4(two(a, 0), two(a, 16), two(b, 0), two(b, 16)));
    };
#pragma unroll
    for (int i = 0; i < NS; ++i)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const bf16x8_t w0 = widen4(wr[n][i].x, wr[n][i].y), w1 = widen4(wr[n][i].z, wr[n][i].w);
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                acc[j][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0, as_bf16x8(ar[j][i][0]), acc[j][n], 0, 0, 0);
                acc[j][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1, as_bf16x8(ar[j][i][1]), acc[j][n], 0, 0, 0);
            }
        }
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int n = 0; n < 2; ++n) *(f32x4_t *)&red[w][16 * j + l16][16 * n + 4 * g] = acc[j][n];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int row = 16 * j + (tid >> 5), col = tid & 31;
        float v = red[0][row][col];
#pragma unroll
        for (int i = 1; i < 8; ++i) v += red[i][row][col]; // in k order
        yt[row][col] = (uint16_t)bf16_bits(go.bias ? v * sc + bn : v * sc);
    }
    __syncthreads();
    if (mine) epi_store<EPI>(go, em, *(const uint4 *)&yt[er][ec], piece, cols);
}

// The staged epilogue's conditions: 8-column pieces that stay inside N and inside one kStore segment,
// and 16-byte aligned accesses to every output and operand row.
static bool gemm_staged(int N, int epi, const GemmOut &go) {
    if (N % 8) return false;
    const int nout = epi == kStore ? go.nseg : 1;
    for (int j = 0; j < nout; ++j)
        if (!go.out[j] || go.ld[j] % 8 || (uintptr_t)go.out[j] % 16 || (epi == kStore && go.col0[j] % 8)) return false;
    if ((epi == kGated || epi == kAxpyF32 || epi == kAddF32) && (go.ld_aux % 8 || (uintptr_t)go.aux % 16)) return false;
    if (epi == kSiluAddVec && (uintptr_t)go.aux % 16) return false;
    if (epi == kResidual && go.ls && (uintptr_t)go.ls % 16) return false;
    return true;
}

template <int MI, int NI, int KS, bool STG, int NKC>
static hipError_t gemm_q8_stg(const void *A, int M, int K, const int8_t *W, const float *s, int N, int epi,
                              const GemmOut &go, hipStream_t stream) {
    const dim3 grid(((N + 32 * NI - 1) / (32 * NI)) * ((M + 32 * MI - 1) / (32 * MI))), block(256 * KS);
    const uint16_t *a = (const uint16_t *)A;
#define XNP_GEMM(E) hipLaunchKernelGGL((k_gemm_q8<E, false, MI, NI, KS, STG, NKC>), grid, block, 0, stream, a, M, K, W, s, N, go)
    if (go.a_f32) {
        if constexpr (NKC == 0) {
            if (epi == kStore)
                hipLaunchKernelGGL((k_gemm_q8<kStore, true, MI, NI, KS, STG, 0>), grid, block, 0, stream, a, M, K, W, s, N, go);
            else if (epi == kAddF32)
                hipLaunchKernelGGL((k_gemm_q8<kAddF32, true, MI, NI, KS, STG, 0>), grid, block, 0, stream, a, M, K, W, s, N, go);
            else
                return hipErrorInvalidValue;
            return hipGetLastError();
        }
        return hipErrorInvalidValue;
    }
    switch (epi) {
    case kStore: XNP_GEMM(kStore); break;
    case kGeluErf: XNP_GEMM(kGeluErf); break;
    case kGeluTanh: XNP_GEMM(kGeluTanh); break;
    case kResidual: XNP_GEMM(kResidual); break;
    case kSilu: XNP_GEMM(kSilu); break;
    case kSiluAddVec: XNP_GEMM(kSiluAddVec); break;
    case kGated: XNP_GEMM(kGated); break;
    case kAxpyF32: XNP_GEMM(kAxpyF32); break;
    case kStoreF32: XNP_GEMM(kStoreF32); break;
    case kAddF32: XNP_GEMM(kAddF32); break;
    default: return hipErrorInvalidValue;
    }
#undef XNP_GEMM
    return hipGetLastError();
}

// Runs of row tiles the 256-column groups of k_gemm_q8_wres split M into (a group per CU), or 0 where it
// is not taken: a group's start (its 128 KB of W loaded and widened) costs about 4 us, so it wants three
// tiles and more to a run.  2048 rows (two tiles): qkv 10.2 against 9.7 us, linear1 12.5 against 12.8; 5000
// rows: 14.0 against 17.7 and 20.7 against 26.5; 512 columns (out_proj) 18.8 against 17.6 even at 16384
// rows.  The epilogues with operands of their own would not fit its registers.
static int gemm_wres_runs(int M, int K, int N, int epi, const GemmOut &go) {
    if (K != kWrK || N < 1024 || go.a_f32 || (epi != kStore && epi != kGeluErf && epi != kGeluTanh)) return 0;
    const int ntn = (N + kWrCols - 1) / kWrCols, tiles = (M + kWrRows - 1) / kWrRows;
    const int runs = std::min(tiles, std::max(1, 256 / ntn));
    return (tiles + runs - 1) / runs >= 3 && gemm_staged(N, epi, go) ? runs : 0;
}

static hipError_t gemm_q8_wres(const void *A, int M, const int8_t *W, const float *s, int N, int epi, const GemmOut &go,
                               hipStream_t stream) {
    const int ntn = (N + kWrCols - 1) / kWrCols, tiles = (M + kWrRows - 1) / kWrRows;
    const int runs = gemm_wres_runs(M, kWrK, N, epi, go), per = (tiles + runs - 1) / runs;
    const dim3 grid(ntn * ((tiles + per - 1) / per)), block(512);
    const uint16_t *a = (const uint16_t *)A;
    switch (epi) {
    case kStore: hipLaunchKernelGGL(k_gemm_q8_wres<kStore>, grid, block, 0, stream, a, M, W, s, N, go, per); break;
    case kGeluErf: hipLaunchKernelGGL(k_gemm_q8_wres<kGeluErf>, grid, block, 0, stream, a, M, W, s, N, go, per); break;
    case kGeluTanh: hipLaunchKernelGGL(k_gemm_q8_wres<kGeluTanh>, grid, block, 0, stream, a, M, W, s, N, go, per); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// The staged epilogue's kernels come unrolled whole for K of 8 or 16 chunks per half (the flow
// LM's 512-2048 wide projections); others run the rounds in a loop.
template <int MI, int KS>
static hipError_t gemm_q8_mi(const void *A, int M, int K, const int8_t *W, const float *s, int N, int epi,
                             const GemmOut &go, hipStream_t stream) {
    if (!gemm_staged(N, epi, go)) return gemm_q8_stg<MI, 2, KS, false, 0>(A, M, K, W, s, N, epi, go, stream);
    if (!go.a_f32 && K == 8 * KS * kGmK) return gemm_q8_stg<MI, 2, KS, true, 8>(A, M, K, W, s, N, epi, go, stream);
    if (!go.a_f32 && K == 16 * KS * kGmK) return gemm_q8_stg<MI, 2, KS, true, 16>(A, M, K, W, s, N, epi, go, stream);
    return gemm_q8_stg<MI, 2, KS, true, 0>(A, M, K, W, s, N, epi, go, stream);
}

// k_gemm_q8_small's row tiles a group: two (its columns of W read and widened for both) once one-tile groups are
// more than the CUs: linear1 at 128 rows 4.3 -> 4.0 us, linear2 at 331 rows 9.2 -> 7.9.  And its groups.
static bool small_two(int M, int N) { return (int64_t)((N + 31) / 32) * ((M + 15) / 16) > 256; }
static int64_t small_groups(int M, int N) { return (int64_t)((N + 31) / 32) * (small_two(M, N) ? (M + 31) / 32 : (M + 15) / 16); }

// Rows up to which k_gemm_q8_small is taken: each of its groups reads its rows and columns over all of K
// (no tile larger than 32 x 32), which the larger tiles of k_gemm_q8 overtake.  A step of 9 layers (512
// wide, FF 2048, caches of up to 800 rows; k_gemm_q8 with the LayerNorms apart, then here): 32 rows 360 and
// 272 us, 128 rows 472 and 408, 256 rows 625 and 597, 300 rows 685 and 696.  The four projections alone,
// warm: 40 rows 20.7 and 15.1 us, 256 rows 21.4 and 19.4, 600 rows 26.1 and 36.8.
//
// And no more groups than CUs, since a second round costs what the first did (K x N, larger tiles and here: 1024 x
// 3072 at 64 rows, 192 groups, 6.4 and 5.1 us, at 100 rows, 384 groups, 6.5 and 7.8; 2048 x 4096 at 64 rows, 256
// groups, 9.0 and 8.3, at 100 rows 10.2 and 13.6; 512 x 6144 at 33 rows, 384 groups, 4.6 and 5.0).  With the norm
// inside too, though it saves a launch there (a layer of FF 2048 at 200 rows, linear1 in 448 groups, 32.6 us and
// apart 31.7; FF 4096 at 128 rows, 512 groups, 43.3 and 41.7; at 200 rows 51.0 and 47.5): one rule for both keeps
// the layer step equal to its pieces to the bit.
constexpr int kSmallRows = 256;
static bool gemm_small(int M, int K, int N, int epi, const GemmOut &go) {
    return M <= kSmallRows && (K == 512 || K == 1024 || K == 2048) && !go.a_f32 && small_groups(M, N) <= 256 &&
           gemm_staged(N, epi, go);
}

template <int EPI, int NS, int LNM>
static hipError_t gemm_q8_small(const void *A, int M, const int8_t *W, const float *s, int N, const GemmOut &go,
                                const LnIn &ln, hipStream_t stream) {
    const dim3 grid(small_groups(M, N));
    const uint16_t *a = (const uint16_t *)A;
    if (small_two(M, N))
        hipLaunchKernelGGL((k_gemm_q8_small<EPI, NS, 2, LNM>), grid, dim3(512), 0, stream, a, M, W, s, N, go, ln);
    else
        hipLaunchKernelGGL((k_gemm_q8_small<EPI, NS, 1, LNM>), grid, dim3(512), 0, stream, a, M, W, s, N, go, ln);
    return hipGetLastError();
}

template <int NS>
static hipError_t gemm_q8_small_epi(const void *A, int M, const int8_t *W, const float *s, int N, int epi, const GemmOut &go,
                                    hipStream_t stream) {
    switch (epi) {
    case kStore: return gemm_q8_small<kStore, NS, 0>(A, M, W, s, N, go, LnIn(), stream);
    case kGeluErf: return gemm_q8_small<kGeluErf, NS, 0>(A, M, W, s, N, go, LnIn(), stream);
    case kGeluTanh: return gemm_q8_small<kGeluTanh, NS, 0>(A, M, W, s, N, go, LnIn(), stream);
    case kResidual: return gemm_q8_small<kResidual, NS, 0>(A, M, W, s, N, go, LnIn(), stream);
    case kSilu: return gemm_q8_small<kSilu, NS, 0>(A, M, W, s, N, go, LnIn(), stream);
    case kSiluAddVec: return gemm_q8_small<kSiluAddVec, NS, 0>(A, M, W, s, N, go, LnIn(), stream);
    case kGated: return gemm_q8_small<kGated, NS, 0>(A, M, W, s, N, go, LnIn(), stream);
    case kAxpyF32: return gemm_q8_small<kAxpyF32, NS, 0>(A, M, W, s, N, go, LnIn(), stream);
    case kStoreF32: return gemm_q8_small<kStoreF32, NS, 0>(A, M, W, s, N, go, LnIn(), stream);
    case kAddF32: return gemm_q8_small<kAddF32, NS, 0>(A, M, W, s, N, go, LnIn(), stream);
    default: return hipErrorInvalidValue;
    }
}

// LayerNorm (norm: the affine, the modulation) then the projection; h: M x K bf16 of scratch, taken where
// the two run apart.  Fused for few rows of 512 with the epilogues the flow LM pairs with a norm.
hipError_t launch_norm_gemm_q8(const void *x, int M, int K, const RowNorm &norm, void *h, const int8_t *W, const float *s,
                               int N, int epi, const GemmOut &go, hipStream_t stream) {
    if (M <= 0) return hipSuccess;
    if (K == 512 && gemm_small(M, K, N, epi, go) && (norm.w == nullptr) == (norm.b == nullptr) &&
        (norm.shift == nullptr) == (norm.scale == nullptr) && (!norm.shift || norm.ld_mod % 8 == 0)) {
        LnIn ln;
        ln.w = norm.w, ln.b = norm.b, ln.eps = norm.eps;
        ln.shift = (const uint16_t *)norm.shift, ln.scale = (const uint16_t *)norm.scale, ln.ld_mod = norm.ld_mod;
        const int mode = (norm.w ? kLnAffine : 0) | (norm.shift ? kLnMod : 0);
        if (mode == kLnAffine && epi == kStore) return gemm_q8_small<kStore, 1, 1 + kLnAffine>(x, M, W, s, N, go, ln, stream);
        if (mode == kLnAffine && epi == kGeluErf) return gemm_q8_small<kGeluErf, 1, 1 + kLnAffine>(x, M, W, s, N, go, ln, stream);
        if (mode == kLnAffine && epi == kGeluTanh) return gemm_q8_small<kGeluTanh, 1, 1 + kLnAffine>(x, M, W, s, N, go, ln, stream);
        if (mode == (kLnAffine | kLnMod) && epi == kSilu)
            return gemm_q8_small<kSilu, 1, 1 + (kLnAffine | kLnMod)>(x, M, W, s, N, go, ln, stream);
        if (mode == kLnMod && epi == kAxpyF32) return gemm_q8_small<kAxpyF32, 1, 1 + kLnMod>(x, M, W, s, N, go, ln, stream);
        if (mode == kLnMod && epi == kStoreF32) return gemm_q8_small<kStoreF32, 1, 1 + kLnMod>(x, M, W, s, N, go, ln, stream);
    }
    const hipError_t e = launch_layer_norm_mod(x, M, K, norm.w, norm.b, norm.eps, norm.shift, norm.scale, norm.ld_mod, h, stream);
    return e != hipSuccess ? e : launch_gemm_q8(h, M, K, W, s, N, epi, go, stream);
}

hipError_t launch_gemm_q8(const void *A, int M, int K, const int8_t *W, const float *s, int N, int epi,
                          const GemmOut &go, hipStream_t stream) {
    if (M <= 0) return hipSuccess;
    if (N <= 0 || K <= 0 || K % 16) return hipErrorInvalidValue;
    if (gemm_small(M, K, N, epi, go)) {
        if (K == 512) return gemm_q8_small_epi<1>(A, M, W, s, N, epi, go, stream);
        if (K == 1024) return gemm_q8_small_epi<2>(A, M, W, s, N, epi, go, stream);
        return gemm_q8_small_epi<4>(A, M, W, s, N, epi, go, stream);
    }
    // 32-row tiles when 64-row ones would leave the chip's 1024 SIMDs under two waves each; 128-row
    // tiles when those still give 512 groups (two per CU)
    const int64_t ntn = (N + kGmT - 1) / kGmT;
    const int64_t groups64 = ntn * ((M + kGmT - 1) / kGmT), groups128 = ntn * ((M + 127) / 128);
    const bool mi1 = groups64 < 512;
    if (gemm_wres_runs(M, K, N, epi, go) > 0) return gemm_q8_wres(A, M, W, s, N, epi, go, stream);
    // 128 x 128 tiles (twice the products per barrier and per byte staged of 128 x 64) where they fill the
    // chip's places in nearly whole rounds.  K of 512 and 1024: two groups a CU (74 KB of LDS each), 512 places,
    // four fifths and more of them in every round.  512 columns, smaller tiles then these: K = 512 at 12288
    // rows (three quarters) 17.7 and 18.2 us, 13057 rows 20.7 and 18.1, 16384 rows 21.5 and 19.2, 20480 rows
    // (two rounds, five eighths) 26.3 and 26.7.  K = 2048, two halves a group (147 KB): one a CU, 256 places,
    // from three quarters on: 4096 rows (half) 23.0 and 26.7 us, 6144 rows (three quarters) 31.3 and 27.5, 8192
    // rows 38.0 and 28.0, 10240 rows (two rounds, five eighths) 43.5 and 48.0, 12288 rows (three quarters)
    // 51.0 and 48.3, 16384 rows 66.4 and 50.5.  (Each alone, warm.)
    const int64_t wide = (N + 127) / 128 * (int64_t)((M + 127) / 128), places = K == 32 * kGmK ? 256 : 512;
    const int64_t room = places * ((wide + places - 1) / places); // of every round it takes
    if ((places == 256 ? 4 * wide >= 3 * room : 5 * wide >= 4 * room) && !go.a_f32 && gemm_staged(N, epi, go)) {
        if (K == 8 * kGmK) return gemm_q8_stg<4, 4, 1, true, 8>(A, M, K, W, s, N, epi, go, stream);
        if (K == 16 * kGmK) return gemm_q8_stg<4, 4, 1, true, 16>(A, M, K, W, s, N, epi, go, stream);
        if (K == 32 * kGmK) return gemm_q8_stg<4, 4, 2, true, 16>(A, M, K, W, s, N, epi, go, stream);
    }
    // two halves per group on alternate K chunks when K is long (32 chunks and more)
    if (K >= 32 * kGmK)
        return mi1 ? gemm_q8_mi<1, 2>(A, M, K, W, s, N, epi, go, stream) : gemm_q8_mi<2, 2>(A, M, K, W, s, N, epi, go, stream);
    if (groups128 >= 512 && !go.a_f32) return gemm_q8_mi<4, 1>(A, M, K, W, s, N, epi, go, stream);
    return mi1 ? gemm_q8_mi<1, 1>(A, M, K, W, s, N, epi, go, stream) : gemm_q8_mi<2, 1>(A, M, K, W, s, N, epi, go, stream);
}

// ---------------------------------------------------------------------------------------------
// f32 pieces of the flow LM around the transformer (flow_lm.rs, mlp.rs, conditioners.rs):
// linears with bias and fused epilogues, LayerNorm with the AdaLN modulation, the LUT gather.
// Batch-1 frames make these matrix-vector products: one wave per output channel, the weight
// row held in registers, each row of x reduced across the wave.

// NORM: a bit set of kNormLn (LayerNorm the row of x over K), kNormAffine (then * w + b) and
// kNormMod (then the AdaLN modulation y * (1 + scale) + shift, mlp.rs:4-11).  Compile-time, so
// that the norm's operands load together with x instead of behind a branch after the reductions.
constexpr int kNormLn = 1, kNormAffine = 2, kNormMod = 4;

// The (epilogue, norm) pairs of the flow LM's linears, the only ones built: no norm in front of input_linear,
// out_proj, linear2, the flow net's linears of its own rows and, behind z_proj, the EOS logit and cond_embed;
// the affine norm in front of in_proj, linear1, z_proj, the EOS logit and cond_embed; with the modulation in
// front of mlp.0; the modulation alone in front of the final linear.
constexpr bool linear_built(int epi, int norm) {
    return norm == 0 ? epi != kLinGeluErf && epi != kLinGeluTanh
           : norm == (kNormLn | kNormAffine)
               ? epi == kLinStore || epi == kLinGeluErf || epi == kLinGeluTanh || epi == kLinSilu || epi == kLinSiluAddVec
           : norm == (kNormLn | kNormAffine | kNormMod) ? epi == kLinSilu
                                                        : norm == (kNormLn | kNormMod) && (epi == kLinStore || epi == kLinAxpy);
}

// y (bias added) to the output value: eo the auxiliary operand, er the output's old value
template <int EPI> __device__ __forceinline__ float linear_epilogue(float y, float eo, float er, float alpha) {
    if constexpr (EPI == kLinStore) {
        return y;
    } else if constexpr (EPI == kLinGeluErf) {
        return 0.5f * y * (1.0f + erff(y * 0.7071067811865476f));
    } else if constexpr (EPI == kLinGeluTanh) {
        const float c = 0.7978845608028654f;
        return 0.5f * y * (1.0f + tanhf(c * (y + 0.044715f * y * y * y)));
    } else if constexpr (EPI == kLinSilu) {
        return y / (1.0f + expf(-y));
    } else if constexpr (EPI == kLinSiluAddVec) {
        const float z = y + eo;
        return z / (1.0f + expf(-z));
    } else if constexpr (EPI == kLinResidual) {
        return er + y;
    } else if constexpr (EPI == kLinGated) {
        return er + eo * y;
    } else { // kLinAxpy
        return eo + y * alpha;
    }
}

template <int KC, int EPI, int NORM>
__global__ __launch_bounds__(256) void k_linear_f32(const float *x, int ldx, int M, int K, const float *W,
                                                    const float *bias, int N, LinOut lo, LinNorm ln) {
    const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (n >= N) return;
    // every load is issued unconditionally (the index clamped), so that all of them are in flight
    // together rather than each behind a branch and a wait.  Columns past K are zeroed on the x side,
    // inside the row loop: a select on w would be hoisted out of the loop, and every w load would
    // then be waited for before any x load is issued.
    float w[KC], nw[KC], nb[KC];
#pragma unroll
    for (int c = 0; c < KC; ++c) {
        const int kk = min(c * 64 + lane, K - 1);
        w[c] = W[(size_t)n * K + kk];
        if constexpr ((NORM & kNormAffine) != 0) {
            nw[c] = ln.w[kk];
            nb[c] = ln.b[kk];
        }
    }
    const float b = bias ? bias[n] : 0.f;
    for (int m = 0; m < M; ++m) {
        const float *xr = x + (size_t)m * ldx;
        float xv[KC], sh[KC], sc[KC];
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            const int kk = min(c * 64 + lane, K - 1);
            xv[c] = xr[kk];
            if constexpr ((NORM & kNormMod) != 0) {
                sh[c] = ln.shift[(size_t)m * ln.ld_mod + kk];
                sc[c] = ln.scale[(size_t)m * ln.ld_mod + kk];
            }
        }
        // the output's address (segments picked with constant indices, so the kernel arguments are
        // read as scalars), and the epilogue's operand loaded with x (every lane, the same word)
        float *o = lo.out[0] + (size_t)m * lo.ld[0] + (n - lo.col0[0]);
        if (lo.nseg > 1 && n >= lo.col0[1]) {
            if (lo.nseg > 2 && n >= lo.col0[2])
                o = lo.out[2] + (size_t)m * lo.ld[2] + (n - lo.col0[2]);
            else
                o = lo.out[1] + (size_t)m * lo.ld[1] + (n - lo.col0[1]);
        }
        float eo = 0.f, er = 0.f; // the auxiliary operand; the residual (the output's old value)
        if constexpr (EPI == kLinResidual || EPI == kLinGated) er = *o;
        if constexpr (EPI == kLinSiluAddVec)
            eo = lo.aux[n];
        else if constexpr (EPI == kLinGated || EPI == kLinAxpy)
            eo = lo.aux[(size_t)m * lo.ld_aux + n];
        // a scheduling barrier: the loads above stay here, issued together, rather than sunk to
        // their uses after the reductions (a round trip each)
        __builtin_amdgcn_sched_barrier(0);
        if constexpr ((NORM & kNormLn) != 0) {
            // mean, then the centred sum of squares: the two passes of a textbook LayerNorm
            float sum = 0.f;
#pragma unroll
            for (int c = 0; c < KC; ++c) sum += c * 64 + lane < K ? xv[c] : 0.f;
            sum = wave_sum(sum);
            const float mean = sum / (float)K;
            float sq = 0.f;
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                const float d = c * 64 + lane < K ? xv[c] - mean : 0.f;
                sq = __builtin_fmaf(d, d, sq);
            }
            sq = wave_sum(sq);
            const float rstd = 1.0f / __builtin_sqrtf(sq / (float)K + ln.eps);
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                float y = (xv[c] - mean) * rstd;
                if constexpr ((NORM & kNormAffine) != 0) y = y * nw[c] + nb[c];
                if constexpr ((NORM & kNormMod) != 0) y = y * (sc[c] + 1.0f) + sh[c];
                xv[c] = y;
            }
        }
        float acc = 0.f;
#pragma unroll
        for (int c = 0; c < KC; ++c) acc = __builtin_fmaf(w[c], c * 64 + lane < K ? xv[c] : 0.f, acc);
        acc = wave_sum(acc);
        if (lane != 0) continue;
        *o = linear_epilogue<EPI>(acc + b, eo, er, lo.alpha);
    }
}

// The same product for several rows (prompts, batches of f32 streams), on v_mfma_f32_16x16x4_f32: one
// work group of 8 waves per 16 MT rows x 16 columns, the waves splitting K.  A wave's whole share of x
// and W is loaded at once, 16 bytes a lane: lane (l16, g) holds row (column) l16 at k = 16 i + 4 g .. + 3,
// whose four values go to four products of 4 k each (x and W in the same (g, value) slot, so every k
// meets its own).  Four sums a tile, one per value, then the waves' shares through LDS in a fixed
// order.  A product adds its 4 k one after another, so the even and the odd products are summed apart where the
// registers hold both: chains as short as k_linear_f32's.  (Summed in one, a 1024-wide model's first frame
// stood 6.6e-7 from 64 bits where k_linear_f32's stands 5.4e-7, and 5.7e-7 so; rms of 16 streams.)  The
// LayerNorm's moments are taken the same way (the lane's values, its row's 4 lanes, the 8 waves), in two passes
// over the registers.  Its operands are loaded with x and W, or (LATE: K above 512 with many of them) as they
// are used, since a wave holds 256 registers at most: loaded ahead, the affine and modulated norm spilled 97 of
// K = 1024's and 456 of K = 2048's (two row tiles); a 2048-wide model of 2 layers, 16 prompts of 20 tokens:
// 1296 and 949 us, its frame 376 and 292.
//
// At prompt sizes this is bound by the launch and one round trip to memory; k_linear_f32 took the rows
// one after another, a round trip and three wave sums each (64 rows of 512: 15-27 us a launch, here
// 4-10).
template <int NST, int MT, int EPI, int NORM>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(NST > 4 || (MT > 1 && (NORM & kNormMod)) ? 2 : 4)))
void k_linear_f32_rows(const float *x, int ldx, int M, int K, const float *W,
                                                         const float *bias, int N, LinOut lo, LinNorm ln) {
    typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4))); // rows need word alignment only
    __shared__ float red[8][MT][16][17];
    __shared__ float mom[2][8][MT * 16];
    const int ntn = (N + 15) / 16, m0 = (int)blockIdx.x / ntn * (16 * MT), n0 = (int)blockIdx.x % ntn * 16;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, l16 = lane & 15;
    constexpr bool AFF = (NORM & kNormAffine) != 0, MOD = (NORM & kNormMod) != 0;
    constexpr bool LATE = (MT + 1 + 2 * AFF + 2 * MT * MOD) * NST > 40; // 16 bytes a lane each
    constexpr int NL = LATE ? 1 : NST, NA = MT * NST > 16 ? 1 : 2; // norm operands held; sums a value
    // every load is unconditional, its row and k clamped; values past K are zeroed on the x side
    f32x4_a4 xv[MT][NST], wv[NST], sh[MT][NL], sc[MT][NL], nw[NL], nb[NL];
    int k[NST];
    auto norm_load = [&](int i, int s) { // k[i]'s norm operands, into place s
        const int kk = min(k[i], K - 4);
        if constexpr (AFF) {
            nw[s] = *(const f32x4_a4 *)(ln.w + kk);
            nb[s] = *(const f32x4_a4 *)(ln.b + kk);
        }
        if constexpr (MOD) {
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                const size_t o = (size_t)min(m0 + 16 * j + l16, M - 1) * ln.ld_mod + kk;
                sh[j][s] = *(const f32x4_a4 *)(ln.shift + o);
                sc[j][s] = *(const f32x4_a4 *)(ln.scale + o);
            }
        }
    };
    const float *wr = W + (size_t)min(n0 + l16, N - 1) * K;
#pragma unroll
    for (int i = 0; i < NST; ++i) {
        k[i] = 16 * (w * NST + i) + 4 * g;
        const int kk = min(k[i], K - 4);
        wv[i] = *(const f32x4_a4 *)(wr + kk);
#pragma unroll
        for (int j = 0; j < MT; ++j) xv[j][i] = *(const f32x4_a4 *)(x + (size_t)min(m0 + 16 * j + l16, M - 1) * ldx + kk);
        if constexpr (!LATE) norm_load(i, i);
    }
    // the output this thread finishes (tile row er of row tile ej, column n0 + en) and its operands
    const int ej = threadIdx.x >> 8, er_ = (threadIdx.x >> 4) & 15, en = threadIdx.x & 15;
    const int om = m0 + 16 * ej + er_, on = n0 + en;
    const bool mine = ej < MT && om < M && on < N;
    float *o = nullptr;
    float eo = 0.f, er = 0.f, b = 0.f;
    if (mine) {
        o = lo.out[0] + (size_t)om * lo.ld[0] + (on - lo.col0[0]);
        if (lo.nseg > 1 && on >= lo.col0[1]) {
            if (lo.nseg > 2 && on >= lo.col0[2])
                o = lo.out[2] + (size_t)om * lo.ld[2] + (on - lo.col0[2]);
            else
                o = lo.out[1] + (size_t)om * lo.ld[1] + (on - lo.col0[1]);
        }
        if (bias) b = bias[on];
        if constexpr (EPI == kLinResidual || EPI == kLinGated) er = *o;
        if constexpr (EPI == kLinSiluAddVec)
            eo = lo.aux[on];
        else if constexpr (EPI == kLinGated || EPI == kLinAxpy)
            eo = lo.aux[(size_t)om * lo.ld_aux + on];
    }
    __builtin_amdgcn_sched_barrier(0); // the loads above go out together
    if constexpr ((NORM & kNormLn) != 0) {
        // a row's moment from every lane that holds a share of it: rows 16 j + l16
        auto moment = [&](float (&v)[MT], int which, float (&out)[MT]) {
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                const float s = swap_sum<32>(swap_sum<16>(v[j]));
                if (g == 0) mom[which][w][16 * j + l16] = s;
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                float p[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) p[q] = mom[which][q][16 * j + l16];
                out[j] = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            }
        };
        float v[MT], sum[MT], sq[MT];
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            v[j] = 0.f;
#pragma unroll
            for (int i = 0; i < NST; ++i)
                if (k[i] < K) v[j] += (xv[j][i].x + xv[j][i].y) + (xv[j][i].z + xv[j][i].w);
        }
        moment(v, 0, sum);
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const float mean = sum[j] / (float)K;
            v[j] = 0.f;
#pragma unroll
            for (int i = 0; i < NST; ++i) {
                xv[j][i] -= mean;
                const f32x4_a4 d = xv[j][i] * xv[j][i];
                if (k[i] < K) v[j] += (d.x + d.y) + (d.z + d.w);
            }
        }
        moment(v, 1, sq);
#pragma unroll
        for (int j = 0; j < MT; ++j) sq[j] = 1.0f / __builtin_sqrtf(sq[j] / (float)K + ln.eps);
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const int s = LATE ? 0 : i;
            if constexpr (LATE) {
                if (i % 4 == 0) __builtin_amdgcn_sched_barrier(0); // four places' loads at a time
                norm_load(i, 0);
            }
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                xv[j][i] *= sq[j];
                if constexpr (AFF) xv[j][i] = xv[j][i] * nw[s] + nb[s];
                if constexpr (MOD) xv[j][i] = xv[j][i] * (sc[j][s] + 1.0f) + sh[j][s];
            }
        }
    }
    f32x4_t acc[MT][4][NA];
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int c = 0; c < 4 * NA; ++c) acc[j][c / NA][c % NA] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NST; ++i) {
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const bool in = k[i] < K;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                acc[j][c][i % NA] =
                    __builtin_amdgcn_mfma_f32_16x16x4f32(in ? xv[j][i][c] : 0.f, wv[i][c], acc[j][c][i % NA], 0, 0, 0);
        }
    }
    if constexpr (NA > 1) {
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[j][c][0] += acc[j][c][NA - 1];
    }
    // lane: column l16, rows 4 g + r of each row tile
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            red[w][j][4 * g + r][l16] = (acc[j][0][0][r] + acc[j][1][0][r]) + (acc[j][2][0][r] + acc[j][3][0][r]);
    __syncthreads();
    if (!mine) return;
    float p[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) p[q] = red[q][ej][er_][en];
    const float y = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7])) + b;
    *o = linear_epilogue<EPI>(y, eo, er, lo.alpha);
}

// Rows from which k_linear_f32_rows is taken: a whole row tile.  A prompt of the 6-layer model with its
// first frame (row by row, then on row tiles): 4 tokens 391 and 365 us, 8 tokens 431 and 373, 16 tokens
// 560 and 387, 64 tokens 1231 and 424.  Below 16 the gain is small, and the other order of the sums there
// moves a model that feeds its latents back (5 frames from two 5-token prompts) past the 1e-5 of the oracle that
// f32 results are held to (1.1e-5, most of it the oracle's own: its sums stand 1.3e-5 from 64 bits after five
// such frames, either kernel's 3e-6 to 6e-6).
constexpr int kLinRows = 16;

template <int NST, int MT, int NORM>
static hipError_t linear_f32_rows_mt(const float *x, int ldx, int M, int K, const float *W, const float *b, int N, int epi,
                                     const LinOut &lo, const LinNorm &ln, hipStream_t stream) {
    const dim3 grid((N + 15) / 16 * ((M + 16 * MT - 1) / (16 * MT))), block(512);
#define XNP_LIN(E)                                                                                                 \
    if constexpr (linear_built(E, NORM))                                                                           \
        hipLaunchKernelGGL((k_linear_f32_rows<NST, MT, E, NORM>), grid, block, 0, stream, x, ldx, M, K, W, b, N, lo, ln); \
    else                                                                                                           \
        return hipErrorInvalidValue
    switch (epi) {
    case kLinStore: XNP_LIN(kLinStore); break;
    case kLinGeluErf: XNP_LIN(kLinGeluErf); break;
    case kLinGeluTanh: XNP_LIN(kLinGeluTanh); break;
    case kLinSilu: XNP_LIN(kLinSilu); break;
    case kLinSiluAddVec: XNP_LIN(kLinSiluAddVec); break;
    case kLinResidual: XNP_LIN(kLinResidual); break;
    case kLinGated: XNP_LIN(kLinGated); break;
    case kLinAxpy: XNP_LIN(kLinAxpy); break;
    default: return hipErrorInvalidValue;
    }
#undef XNP_LIN
    return hipGetLastError();
}

template <int NST, int NORM>
static hipError_t linear_f32_rows(const float *x, int ldx, int M, int K, const float *W, const float *b, int N, int epi,
                                  const LinOut &lo, const LinNorm &ln, hipStream_t stream) {
    // two row tiles a group (W read once for both) once one-tile groups fill the chip twice over, where the
    // registers hold them
    if constexpr (NST <= 8 || NORM == 0) {
        if ((int64_t)((N + 15) / 16) * ((M + 15) / 16) >= 1024)
            return linear_f32_rows_mt<NST, 2, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
    }
    return linear_f32_rows_mt<NST, 1, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
}

template <int KC, int NORM>
static hipError_t linear_f32_kc(const float *x, int ldx, int M, int K, const float *W, const float *b, int N, int epi,
                                const LinOut &lo, const LinNorm &ln, hipStream_t stream) {
    const dim3 grid((N + 3) / 4), block(256);
#define XNP_LIN(E)                                                                                                 \
    if constexpr (linear_built(E, NORM))                                                                           \
        hipLaunchKernelGGL((k_linear_f32<KC, E, NORM>), grid, block, 0, stream, x, ldx, M, K, W, b, N, lo, ln);     \
    else                                                                                                           \
        return hipErrorInvalidValue
    switch (epi) {
    case kLinStore: XNP_LIN(kLinStore); break;
    case kLinGeluErf: XNP_LIN(kLinGeluErf); break;
    case kLinGeluTanh: XNP_LIN(kLinGeluTanh); break;
    case kLinSilu: XNP_LIN(kLinSilu); break;
    case kLinSiluAddVec: XNP_LIN(kLinSiluAddVec); break;
    case kLinResidual: XNP_LIN(kLinResidual); break;
    case kLinGated: XNP_LIN(kLinGated); break;
    case kLinAxpy: XNP_LIN(kLinAxpy); break;
    default: return hipErrorInvalidValue;
    }
#undef XNP_LIN
    return hipGetLastError();
}

template <int NORM>
static hipError_t linear_f32_norm(const float *x, int ldx, int M, int K, const float *W, const float *b, int N, int epi,
                                  const LinOut &lo, const LinNorm &ln, hipStream_t stream) {
    const int kc = (K + 63) / 64;
    if (M >= kLinRows && K % 4 == 0 && K >= 128) {
        if (K <= 256) return linear_f32_rows<2, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
        if (K <= 512) return linear_f32_rows<4, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
        if (K <= 1024) return linear_f32_rows<8, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
        if (K <= 2048) return linear_f32_rows<16, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
    }
    if (kc <= 1) return linear_f32_kc<1, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
    if (kc <= 4) return linear_f32_kc<4, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
    if (kc <= 8) return linear_f32_kc<8, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
    if (kc <= 16) return linear_f32_kc<16, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
    if (kc <= 32) return linear_f32_kc<32, NORM>(x, ldx, M, K, W, b, N, epi, lo, ln, stream);
    return hipErrorInvalidValue;
}

hipError_t launch_linear_f32(const float *x, int ldx, int M, int K, const float *W, const float *b, int N, int epi,
                             const LinOut &lo, hipStream_t stream, const LinNorm *ln) {
    if (M <= 0 || N <= 0) return hipSuccess;
    if (!ln) return linear_f32_norm<0>(x, ldx, M, K, W, b, N, epi, lo, LinNorm(), stream);
    if ((ln->w == nullptr) != (ln->b == nullptr) || (ln->shift == nullptr) != (ln->scale == nullptr))
        return hipErrorInvalidValue;
    if (ln->w && ln->shift) return linear_f32_norm<kNormLn | kNormAffine | kNormMod>(x, ldx, M, K, W, b, N, epi, lo, *ln, stream);
    if (ln->w) return linear_f32_norm<kNormLn | kNormAffine>(x, ldx, M, K, W, b, N, epi, lo, *ln, stream);
    if (ln->shift) return linear_f32_norm<kNormLn | kNormMod>(x, ldx, M, K, W, b, N, epi, lo, *ln, stream);
    return hipErrorInvalidValue; // no linear of the flow LM takes the norm alone
}

// LUTConditioner::embed_tokens (conditioners.rs:239-262): out[r] = table[ids[r]], rows of dim f32.
__global__ void k_embed_f32(const float *table, const int32_t *ids, int rows, int dim, float *out) {
    const int r = blockIdx.x;
    const float *src = table + (size_t)ids[r] * dim;
    for (int i = threadIdx.x; i < dim; i += blockDim.x) out[(size_t)r * dim + i] = src[i];
}

__global__ void k_gather_rows(const uint4 *table, const int32_t *ids, int row_u4, uint4 *out) {
    const int r = blockIdx.x;
    const uint4 *src = table + (size_t)ids[r] * row_u4;
    for (int i = threadIdx.x; i < row_u4; i += blockDim.x) out[(size_t)r * row_u4 + i] = src[i];
}

hipError_t launch_gather_rows(const void *table, const int32_t *ids, int rows, int row_bytes, void *out,
                              hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    if (row_bytes % 16) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_gather_rows, dim3(rows), dim3(256), 0, stream, (const uint4 *)table, ids, row_bytes / 16,
                       (uint4 *)out);
    return hipGetLastError();
}

hipError_t launch_embed_f32(const float *table, const int32_t *ids, int rows, int dim, float *out, hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_embed_f32, dim3(rows), dim3(256), 0, stream, table, ids, rows, dim, out);
    return hipGetLastError();
}


} // namespace xnp
