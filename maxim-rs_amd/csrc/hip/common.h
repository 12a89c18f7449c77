// Shared device helpers for the gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "kargs.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One 16x16x4 fp32 MFMA: acc[16x16] += A[16x4] * B[4x16].
// Lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16]; the accumulator
// holds D[4 * (l / 16) + r][l % 16] in element r.
__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// fp32 products on the bf16 matrix cores (the method of Henry, Tang and Heinecke,
// "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", ARITH 2019). A float splits exactly into three
// bf16 parts, x = h + m + l (8 + 8 + 8 significand bits, each part the rounded
// remainder of the last), and of the nine products of two split floats the six
// of order 2^0, 2^-8 and 2^-16 are kept; what is dropped is below 2^-24 of the
// product (a sum of one term is off by 1.1e-7 of it at most, an fp32 product by
// 6.0e-8). Each v_mfma_f32_16x16x32_bf16 adds 32 exact products in fp32 with
// one rounding, so a sum of K products is rounded 6 K / 32 times where the
// fp32 MFMA chain rounds K times: against 64-bit sums of N(0, 1) products the
// relative error is 3.7e-8 / 9.2e-8 / 1.5e-7 / 2.3e-7 at K = 32 / 64 / 128 /
// 256, the fp32 MFMA's 1.0e-7 / 1.4e-7 / 2.0e-7 / 2.9e-7. Six bf16 MFMAs take
// 96 cycles of a SIMD for the 32 k's that eight fp32 ones take 256 for, and
// leave most of the vector ALU's issue slots free (the fp32 MFMA does not).
// Both operands are taken 2^24 times as large (kSplitScale): every bit of a
// float, a subnormal one's too, is then in a part above 2^-126, below which
// bf16 operands may be flushed, so no operand is too small to split exactly,
// and sums 2^48 times as large are rounded like the plain ones wherever these
// are normal floats. At the other end an infinite or NaN operand, one past
// 2^104 or a sum past 2^80 leaves a sum that is not finite, which the wave
// forms again in fp32.
constexpr float kSplitScale = 0x1p24f, kUnsplit = 0x1p-48f;
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Two floats as packed bf16, rounded to nearest even.
__device__ __forceinline__ uint32_t bf2(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
// The three parts of two floats, packed in pairs: 3.5 vector operations per
// element, the remainders by the packed dot product with (-1, 0) and (0, -1)
// (exact: a remainder is a float). The constants come through registers,
// since the instruction's inline -1 is not a packed pair.
__device__ __forceinline__ void split2(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l) {
    uint32_t c0, c1;
    asm("s_mov_b32 %0, 0xbf80" : "=s"(c0));
    asm("s_mov_b32 %0, 0xbf800000" : "=s"(c1));
    const bf16x2 n0 = __builtin_bit_cast(bf16x2, c0), n1 = __builtin_bit_cast(bf16x2, c1);
    h = bf2(a, b);
    const bf16x2 hv = __builtin_bit_cast(bf16x2, h);
    const float r0 = __builtin_amdgcn_fdot2_f32_bf16(hv, n0, a, false);
    const float r1 = __builtin_amdgcn_fdot2_f32_bf16(hv, n1, b, false);
    m = bf2(r0, r1);
    const bf16x2 mv = __builtin_bit_cast(bf16x2, m);
    l = bf2(__builtin_amdgcn_fdot2_f32_bf16(mv, n0, r0, false), __builtin_amdgcn_fdot2_f32_bf16(mv, n1, r1, false));
}
// One 16x16x32 bf16 MFMA: lane l supplies eight k's of A's row l % 16 and of
// B's column l % 16 (which eight is the caller's, the same for both), the
// accumulator laid out as mfma16's.
__device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

// Work-group placement. The dispatcher deals consecutive work-group ids to
// the 8 XCDs in turn, and each XCD has its own L2, so neighbouring tiles
// (which share halo rows, cache lines and operands) land in different L2s.
// xcd_tile() renumbers the (gridDim.x x gridDim.y) grid so that each XCD
// walks one contiguous run of the new ids, and splits the new id into a tile
// index and a band (e.g. the output-channel block) with the band fastest, so
// every band of a tile is computed under the same L2.
__device__ __forceinline__ void xcd_tile(int &tile, int &band) {
    const int gy = gridDim.y, n = gridDim.x * gy;
    const int id = blockIdx.x + blockIdx.y * gridDim.x;
    const int x = id & 7, q = n >> 3, r = n & 7;
    const int nid = x * q + min(x, r) + (id >> 3);
    tile = nid / gy;
    band = nid - tile * gy;
}

__device__ __forceinline__ float4 ld4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ void st4(float *p, float4 v) { *reinterpret_cast<float4 *>(p) = v; }

// GELU, x Phi(x) = 0.5 x (1 + erf(x / sqrt 2)), branch-free: with
// R = Phi(-|x|), GELU is max(x, 0) - |x| R for either sign of x, and
// R = 2^q(t) at t = min(|x|, 6), q the degree-6 polynomial fitted by
// weighted least squares to log2 Phi(-t) over [0, 6] (each point weighted by
// how little error its GELU value allows, so the fit is tightest near 0),
// evaluated by Horner and raised on the transcendental unit (v_exp_f32, 1
// ulp): a min, six FMAs, one exp2, a max and an FMA (the |x| and the sign
// are source modifiers). Within 6.3e-8 * (1 + |x|) of the exact function
// (past |x| = 6 the clamped R is below 1e-9). The standalone GELU op and
// every fused epilogue use this one function, so fusing a GELU changes no
// bit.
__device__ __forceinline__ float gelu(float x) {
    const float ax = fabsf(x);
    const float t = fminf(ax, 6.0f);
    float q = __builtin_fmaf(3.3113869e-05f, t, -7.6996483e-04f);
    q = __builtin_fmaf(q, t, 8.0852984e-03f);
    q = __builtin_fmaf(q, t, -5.3423237e-02f);
    q = __builtin_fmaf(q, t, -4.5875868e-01f);
    q = __builtin_fmaf(q, t, -1.1512076e+00f);
    q = __builtin_fmaf(q, t, -9.9999213e-01f);
    const float r = __builtin_amdgcn_exp2f(q);  // Phi(-|x|)
    return __builtin_fmaf(-ax, r, fmaxf(x, 0.0f));
}

// 1 / (1 + e^-x) with e^-x = 2^(-x log2 e) on the transcendental unit and
// one hardware reciprocal (v_exp_f32, v_rcp_f32, 1 ulp each): within
// 1.3e-7 (1 + |x|) of the exact function, 0 and 1 in the tails where the
// power overflows or vanishes; held to the CPU path's 1 / (1 + expf(-x))
// within 4e-7 (1 + |x|). One function, so the standalone kernel, the CALayer
// block and the fused epilogue agree to the bit.
__device__ __forceinline__ float sigmoid(float x) {
    const float e = __builtin_amdgcn_exp2f(-x * 1.4426950408889634f);
    return __builtin_amdgcn_rcpf(1.0f + e);
}

// The fused epilogue (kargs.h, Epilogue) for output element `idx`, after bias.
__device__ __forceinline__ float epilogue(const Epilogue &e, float v, int64_t idx) {
    if (e.u) v = e.u[idx] * (v + 1.0f);
    if (e.act == MXK_ACT_GELU) v = gelu(v);
    else if (e.act == MXK_ACT_LRELU) v = v >= 0.0f ? v : e.slope * v;
    else if (e.act == MXK_ACT_SIGMOID) v = sigmoid(v);
    if (e.m) v = v * e.m[idx];
    if (e.r1) v = v + e.r1[idx];
    if (e.r2) v = v + e.r2[idx];
    return v;
}

// The same for the two elements idx, idx + 1, with 64-bit operand loads
// (idx even and every operand 8-byte aligned): each element's operations and
// their order are epilogue()'s.
__device__ __forceinline__ void epilogue2(const Epilogue &e, float &v0, float &v1, int64_t idx) {
    const float2 zero = make_float2(0.0f, 0.0f);
    const float2 u2 = e.u ? *reinterpret_cast<const float2 *>(e.u + idx) : zero;
    const float2 m2 = e.m ? *reinterpret_cast<const float2 *>(e.m + idx) : zero;
    const float2 a2 = e.r1 ? *reinterpret_cast<const float2 *>(e.r1 + idx) : zero;
    const float2 b2 = e.r2 ? *reinterpret_cast<const float2 *>(e.r2 + idx) : zero;
    const float uu[2] = {u2.x, u2.y}, mm[2] = {m2.x, m2.y}, aa[2] = {a2.x, a2.y}, bb[2] = {b2.x, b2.y};
    float v[2] = {v0, v1};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        float x = v[k];
        if (e.u) x = uu[k] * (x + 1.0f);
        if (e.act == MXK_ACT_GELU) x = gelu(x);
        else if (e.act == MXK_ACT_LRELU) x = x >= 0.0f ? x : e.slope * x;
        else if (e.act == MXK_ACT_SIGMOID) x = sigmoid(x);
        if (e.m) x = x * mm[k];
        if (e.r1) x = x + aa[k];
        if (e.r2) x = x + bb[k];
        v[k] = x;
    }
    v0 = v[0];
    v1 = v[1];
}

// The same for the four elements idx .. idx + 3, with 128-bit operand loads
// (idx % 4 == 0 and every operand 16-byte aligned): each element's operations
// and their order are epilogue()'s.
__device__ __forceinline__ void epilogue4(const Epilogue &e, float *v, int64_t idx) {
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 u4 = e.u ? *reinterpret_cast<const float4 *>(e.u + idx) : zero;
    const float4 m4 = e.m ? *reinterpret_cast<const float4 *>(e.m + idx) : zero;
    const float4 a4 = e.r1 ? *reinterpret_cast<const float4 *>(e.r1 + idx) : zero;
    const float4 b4 = e.r2 ? *reinterpret_cast<const float4 *>(e.r2 + idx) : zero;
    const float uu[4] = {u4.x, u4.y, u4.z, u4.w}, mm[4] = {m4.x, m4.y, m4.z, m4.w};
    const float aa[4] = {a4.x, a4.y, a4.z, a4.w}, bb[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float x = v[k];
        if (e.u) x = uu[k] * (x + 1.0f);
        if (e.act == MXK_ACT_GELU) x = gelu(x);
        else if (e.act == MXK_ACT_LRELU) x = x >= 0.0f ? x : e.slope * x;
        else if (e.act == MXK_ACT_SIGMOID) x = sigmoid(x);
        if (e.m) x = x * mm[k];
        if (e.r1) x = x + aa[k];
        if (e.r2) x = x + bb[k];
        v[k] = x;
    }
}
