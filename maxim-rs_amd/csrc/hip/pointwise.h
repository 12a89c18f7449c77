// Streaming matrix-core kernels for the Dense-shaped ops whose reduction is
// short next to their streamed axis: every 1x1 conv (K = c_in <= 512 over
// up to 286720 pixels) and both GateMm modes. Products of floats are formed
// from three-part bf16 operands (common.h): the weights split once, at upload
// (GemmArgs A3), the streamed operand X in registers on its way to the matrix
// cores. Each wave owns a 64 x (16 * TMW) output tile, or a quarter of its
// reduction.
//
// Two layouts share one body (D = the 16x16 MFMA tile, lane l = 16g + i):
//
//   CH  Y[m][n] = bias[m] + sum_k W[m][k] X[k][n]       (conv1x1, GateMm mode 0)
//       A operand = X^T: lane i of tile j supplies pixel n0 + 16 (i % 4) +
//       4 (i / 4) + j, so one 128-bit load feeds four tiles (and the sixteen
//       lanes of a row still read 256 contiguous bytes), and the output
//       D_j[4g + r][i] = Y[m0 + i][n0 + 16r + 4g + j]: for each r the four
//       lanes of a channel hold 16 adjacent pixels, one 64-byte run per store.
//   RW  Y[n][a] = bias[a] + sum_k X[n][k] W[a][k]       (GateMm mode 1)
//       A operand = W, B operand = X^T, so a lane holds four consecutive
//       outputs of one row: D[4g + r][i] = Y[n0 + 16j + i][a0 + 4g + r].
//
// X is loaded in supersteps of 16 k's: lane group g supplies k = 16 S + 4 g + t,
// t = 0..3, so each lane fetches its four k's of a row with one 128-bit load.
// Two supersteps make the 32 k's of an MFMA, whatever their order, as the
// weights are laid out in the same one. The six products of every 32 k's are
// added smallest first, and the 32s in ascending order, in every form of the
// kernel, and a sum that is not finite is formed in fp32 whatever its tile
// holds, so forms that differ in tile width or in how X reaches the matrix
// cores agree to the bit on any data.
//
// Measured on MI355X against the same kernels on fp32 MFMAs (which are bound by
// the SIMDs' issue: MFMA and VALU add up there): GateMm over 256 tokens, 32
// channels at 448x640, 60.2 -> 35.3 us (mode 0) and 66.1 -> 34.5 us (mode 1),
// 136 TFLOP/s; LayerNorm + Dense 128 -> 256 + GELU at 112x160 24.2 -> 14.7 us,
// 32 -> 64 at 448x640 28.0 -> 23.0 us; a 640x448 S-3 pass 22.8 -> 19.1 ms.
#pragma once

#include "common.h"

namespace pw {

enum { CH = 0, RW = 1 };

__device__ __forceinline__ float comp(const float4 &v, int t) {
    return t == 0 ? v.x : t == 1 ? v.y : t == 2 ? v.z : v.w;
}

// GemmArgs as used here: A = W ([M][K] for CH, [N][K] for RW), B = X
// ([K][N] for CH, [M][K] for RW), C = Y; M is the weight-output dimension for
// CH and the row count for RW. Preconditions (checked by the host): K % 16 ==
// 0 (K % 64 == 0 when KS = 4), N % 4 == 0, every pointer 16-byte aligned,
// batch strides % 4 == 0.
//
// Work unit: one output tile of 64 streamed elements x TW weight outputs.
// KS = 1: every wave owns a tile; KS = 4: the four waves of a block split one
// tile's reduction into quarters and add the partial sums in LDS in a fixed
// order (wave 0 + 1 + 2 + 3), for the shapes with too few tiles to fill the
// chip.
// SH (KS = 1): SH consecutive waves of a block hold weight tiles of the same
// 64 streamed elements (the tile count per column block is a multiple of SH)
// and share X: per stage of 16 SH k's each wave loads one superstep, normalises
// and splits it once, and leaves the parts in LDS for all of them (24 KB a
// block), so an element of X is loaded, normalised and split once for 16 TMW SH
// outputs instead of 16 TMW. SH = 1: each wave feeds its own registers.
//
// Operand loads are clamped into range instead of guarded: an X column or
// weight row past the edge only feeds output rows/columns of the MFMA tile
// that are never stored, so no branch or select sits between the loads and
// the matrix cores. The next stage's (or 32 k's) loads are in flight while one
// (or its second half) multiplies.
// The image index of blocked index e (0 <= e < plane) under map q (32-bit:
// the host enables a map only below 2^31 elements).
// n / d for n < 2^31, with the host's multiplier m and shift s for d.
__device__ __forceinline__ uint32_t mdiv(uint32_t n, uint32_t m, int32_t s) { return __umulhi(n + n, m) >> s; }
__device__ __forceinline__ uint32_t unblock(const BlockMap &q, uint32_t e) {
    const uint32_t pp = (uint32_t)(q.fh * q.fw);
    const uint32_t gi = mdiv(e, q.mpp, q.spp), p = e - gi * pp;
    const uint32_t gy = mdiv(gi, q.mgw, q.sgw), gx = gi - gy * (uint32_t)q.gw;
    const uint32_t fy = mdiv(p, q.mfw, q.sfw), fx = p - fy * (uint32_t)q.fw;
    return (gy * q.fh + fy) * q.wd + gx * q.fw + fx;
}

// The epilogue's operand set as a compile-time mask (EP >= 0), so that a
// kernel specialised for it has no per-slot tests of the argument block and
// its memory waits count exactly the loads each use needs; EP = -1 reads the
// set from the argument block at run time (every combination, one kernel).
enum { EP_U = 1, EP_R1 = 2, EP_R2 = 4, EP_GELU = 8, EP_LRELU = 16, EP_YMAP = 32, EP_BIAS = 64, EP_R1MAP = 128 };

// LN: 0 no folded LayerNorm; 1 the LayerNorm's expression on X,
// (x - m) r w + c with w and c per input channel, in the LayerNorm kernels'
// order (folding w and c into the weights changes the rounding), with m and r
// read from a statistics pass; 2 the same with m and r computed here, from
// the X tile the block's four waves hold between them (KS = 4 with two
// supersteps per wave: 128 channels), so no statistics pass runs. Mode 2
// sums each pixel's channels in another order than the LayerNorm kernels
// (a wave's 32 in its lanes' order, the four lane groups pairwise, then the
// waves in turn), so its normalised X differs from theirs by rounding.
// (ux, nx): this block's index and the block count along x, by: the batch;
// a kernel pairing two launches in one grid passes each part its own.
// XR: the LDS pool comes from the caller (xpool, as many floats as `POOL`
// below), so two different instances in one kernel share one.
template <int LAYOUT, int TMW, int KS, bool FUSED, int LN, bool XM = false, bool XMUL = false, bool CT = false,
          bool LNO = false, int EP = -1, bool FOLD = false, bool XR = false, int SH = 1>
__device__ void body(const GemmArgs &a, int ux, int nx, int by, float *xpool = nullptr) {
    const bool has_u = EP < 0 ? a.e.u != nullptr : (EP & EP_U) != 0;
    const bool has_r1 = EP < 0 ? a.e.r1 != nullptr : (EP & EP_R1) != 0;
    const bool has_r2 = EP < 0 ? a.e.r2 != nullptr : (EP & EP_R2) != 0;
    const bool has_gelu = EP < 0 ? a.e.act == MXK_ACT_GELU : (EP & EP_GELU) != 0;
    const bool has_lrelu = EP < 0 ? a.e.act == MXK_ACT_LRELU : (EP & EP_LRELU) != 0;
    const bool has_ymap = EP < 0 ? a.ymap.on != 0 : (EP & EP_YMAP) != 0;
    const bool has_bias = EP < 0 ? a.bias != nullptr : (EP & EP_BIAS) != 0;
    const bool r1map = EP < 0 ? a.ymap.r1map != 0 : (EP & EP_R1MAP) != 0;
    constexpr int TW = 16 * TMW;    // weight outputs per tile
    constexpr int NACC = 16 * TMW;  // accumulator floats per lane
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int M = a.M, N = a.N, K = a.K;
    const int wout = LAYOUT == CH ? M : N;
    // CH with the batch folded into the columns: batch * N columns, batch
    // n / N holding column n (whole 4-column groups; the grid is 1-D)
    static_assert(!FOLD || (LAYOUT == CH && !LN && !CT && !LNO && !XMUL), "a folded batch: GateMm mode 0");
    constexpr bool fold = FOLD;
    const int slen = LAYOUT == CH ? (fold ? a.batch * N : N) : M;
    const int nib = (wout + TW - 1) / TW;
    const int ntiles = nib * ((slen + 63) / 64);  // < 2^31, checked by the host
    const int b = fold ? 0 : by;
    const float *W = a.A;
    const float *X = a.B + (int64_t)b * a.sB;
    float *Y = a.C + (int64_t)b * a.sC;
    // X's advance per superstep (16 k's): 16 rows (CH) or 16 columns (RW);
    // through a token map, whole rows of cells or of cell pixels.
    const BlockMap &xm = a.xmap;
    int64_t xstep = LAYOUT == CH ? 16 * (int64_t)N : 16;
    if (XM) xstep = LAYOUT == CH ? (int64_t)(16 / xm.gw) * xm.fh * xm.wd : (int64_t)(16 / xm.fw) * xm.wd;

    // One XCD per contiguous range of blocks, so neighbouring tiles (which
    // share operands) meet in the same L2.
    int unit = ux;
    const int nb = nx;
    if ((nb & 7) == 0) unit = (unit & 7) * (nb >> 3) + (unit >> 3);
    const int tile = KS == 1 ? unit * 4 + wave : unit;
    static_assert(SH == 1 || KS == 1, "X is shared by waves with whole reductions");
    // KS = 4: the whole block; SH > 1: waves past the last tile stay for the
    // block's barriers (their columns lie past the edge, nothing is stored)
    if (SH == 1 && tile >= ntiles) return;
    const int nS = K / 16;
    // this wave's first superstep: of its share of the reduction (KS = 4), of
    // its share of each stage (SH > 1)
    const int S0 = SH > 1 ? wave % SH : KS == 1 ? 0 : wave * (nS / 4);
    const int nSw = KS == 1 ? nS : nS / 4;  // supersteps of this wave's reduction

    const int w0 = (tile % nib) * TW;
    const int s0 = (tile / nib) * 64;
    // Input maps: X as the blocked view of an image-ordered tensor (an
    // elided forward permutation). With a folded LayerNorm (CH, xmap.on): X
    // is [channels][pixels] and only the pixel axis is blocked. XM (GateMm):
    // each batch's X is [cells][pixels of a cell] of one channel plane, so
    // element (r, c) sits at cell(r) + pixel(c); the host guarantees that 16
    // k's advance whole cell rows (CH: 16 % gw == 0) or whole pixel rows
    // (RW: 16 % fw == 0), and fw % 4 == 0 for the 128-bit reads.
    auto cell = [&](uint32_t r) -> int64_t {
        const uint32_t gy = mdiv(r, xm.mgw, xm.sgw), gx = r - gy * (uint32_t)xm.gw;
        return (int64_t)gy * xm.fh * xm.wd + (int64_t)gx * xm.fw;
    };
    auto pixel = [&](uint32_t c) -> int64_t {
        const uint32_t fy = mdiv(c, xm.mfw, xm.sfw), fx = c - fy * (uint32_t)xm.fw;
        return (int64_t)fy * xm.wd + fx;
    };
    // CH: this lane's four columns, s0 + 16 (i % 4) + 4 (i / 4) .. + 3 (with
    // a folded batch: column xcol of batch xb)
    int xcol = 0;
    int64_t xbo = 0;  // the folded batch's X offset
    if (LAYOUT == CH) {
        xcol = min(s0 + 16 * (i & 3) + 4 * (i >> 2), slen - 4);
        if (fold) {
            const uint32_t xb = mdiv((uint32_t)xcol, a.fmul, a.fsh);
            xcol -= (int)xb * N;
            xbo = (int64_t)xb * a.sB;
        }
        if (LN && xm.on) xcol = (int)unblock(xm, (uint32_t)xcol);
    }
    const float *xp[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (LAYOUT == CH) {  // row k = 16 S + 4 g + q
            if (XM)
                xp[q] = X + xbo + cell(16 * S0 + 4 * g + q) + pixel(xcol);
            else
                xp[q] = X + xbo + (int64_t)(4 * g + q) * N + xcol + S0 * xstep;
        } else {  // row s0 + 16 q + i, k = 16 S + 4 g .. + 3
            const int row = min(s0 + 16 * q + i, M - 1);
            if (XM)
                xp[q] = X + cell(row) + pixel(16 * S0 + 4 * g);
            else
                xp[q] = X + (int64_t)row * K + 4 * g + S0 * xstep;
        }
    }

    f32x4 acc[4][TMW];  // set by the first superstep

    // A folded LayerNorm (CH only): this lane's four pixels' statistics for
    // the whole tile, and each superstep's scale/bias for k = 16 S + 4 g + q.
    float4 lmean, lrstd;
    const float *lsc = nullptr, *lbi = nullptr;
    if (LN == 1) {  // a single 1x1 conv (no batch): statistics indexed like X's columns
        lmean = ld4(a.ln.mean + xcol);
        lrstd = ld4(a.ln.rstd + xcol);
    }
    if (LN) {
        {
            lsc = a.ln.scale + 4 * g + S0 * 16;
            lbi = a.ln.bias + 4 * g + S0 * 16;
        }
    }
    // A folded Mul: X = B * B2 elementwise, B2 read at X's offsets.
    const float *xq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) xq[q] = XMUL ? a.B2 + (int64_t)b * a.sB + (xp[q] - X) : nullptr;
    // superstep S0 + s of X, with what its normalisation or product needs
    auto load = [&](int s, float4 *xv, float4 *lv, float4 *mv) {
        // SH = 1: an offset the compiler takes as it is; a pointer kept per load
        // and advanced in the loop costs 10 to 20 VGPRs
        int64_t at = s * xstep;
        if (SH == 1) asm("" : "+s"(at));
#pragma unroll
        for (int q = 0; q < 4; ++q) xv[q] = ld4(xp[q] + at);
        if (XMUL) {
#pragma unroll
            for (int q = 0; q < 4; ++q) mv[q] = ld4(xq[q] + at);
        }
        if (LN) {
            lv[0] = ld4(lsc + s * 16);
            lv[1] = ld4(lbi + s * 16);
        }
    };
    auto norm = [&](float4 *xv, const float4 *lv, float sc) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float w = comp(lv[0], q) * sc, c = comp(lv[1], q) * sc;
            xv[q].x = (xv[q].x - lmean.x) * lrstd.x * w + c;
            xv[q].y = (xv[q].y - lmean.y) * lrstd.y * w + c;
            xv[q].z = (xv[q].z - lmean.z) * lrstd.z * w + c;
            xv[q].w = (xv[q].w - lmean.w) * lrstd.w * w + c;
        }
    };
    // the loaded values to X's: normalised, or multiplied (mx_mul's a * b),
    // times the power of two sc
    auto ready = [&](float4 *xv, const float4 *lv, const float4 *mv, float sc) {
        if (LN) {
            norm(xv, lv, sc);
            return;
        }
        if (XMUL) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                xv[q].x = xv[q].x * mv[q].x;
                xv[q].y = xv[q].y * mv[q].y;
                xv[q].z = xv[q].z * mv[q].z;
                xv[q].w = xv[q].w * mv[q].w;
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            xv[q].x = xv[q].x * sc;
            xv[q].y = xv[q].y * sc;
            xv[q].z = xv[q].z * sc;
            xv[q].w = xv[q].w * sc;
        }
    };
    // the superstep's four k's of streamed element j of this lane, split
    struct Half {
        uint32_t h[2], m[2], l[2];
    };
    auto split = [&](const float4 *xv, int j) {
        Half o;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if (LAYOUT == CH)
                split2(comp(xv[2 * t], j), comp(xv[2 * t + 1], j), o.h[t], o.m[t], o.l[t]);
            else
                split2(comp(xv[j], 2 * t), comp(xv[j], 2 * t + 1), o.h[t], o.m[t], o.l[t]);
        }
        return o;
    };
    // the weight parts of 32 k's (chunk c) for this wave's outputs
    const int nC = (K + 31) / 32;
    const u32x4 *w3[TMW];
#pragma unroll
    for (int mt = 0; mt < TMW; ++mt)
        w3[mt] = (const u32x4 *)a.A3 + (int64_t)min(w0 / 16 + mt, (wout + 15) / 16 - 1) * nC * 192 + lane;
    struct WParts {
        u32x4 p[TMW][3];
    };
    auto wload = [&](int c) {
        WParts w;
#pragma unroll
        for (int mt = 0; mt < TMW; ++mt)
#pragma unroll
            for (int q = 0; q < 3; ++q) w.p[mt][q] = w3[mt][(c * 3 + q) * 64];
        return w;
    };
    // the six products of streamed tiles j .. j + n - 1's 32 k's with the
    // weights, smallest first; first: the wave's first 32, which start from zero
    // (an inline-constant accumulator instead of register moves)
    struct Parts {
        u32x4 h, m, l;
    };
    auto mul = [&](int j, int n, const Parts *x, const WParts &w, bool first) {
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        auto one = [&](u32x4 Parts::*part, int q, bool z) {
#pragma unroll
            for (int t = 0; t < n; ++t)
#pragma unroll
                for (int mt = 0; mt < TMW; ++mt) {
                    const f32x4 c = z ? zero : acc[j + t][mt];
                    acc[j + t][mt] =
                        LAYOUT == CH ? mfma32(x[t].*part, w.p[mt][q], c) : mfma32(w.p[mt][q], x[t].*part, c);
                }
        };
        one(&Parts::h, 2, first);
        one(&Parts::l, 0, false);
        one(&Parts::m, 1, false);
        one(&Parts::h, 1, false);
        one(&Parts::m, 0, false);
        one(&Parts::h, 0, false);
    };
    // The bias of this lane's outputs, fetched before the reduction.
    float4 bias[TMW];
#pragma unroll
    for (int mt = 0; mt < TMW; ++mt) {
        if (!has_bias) continue;
        if (LAYOUT == CH) {
            const int m = min(w0 + mt * 16 + i, wout - 1);
            bias[mt].x = a.bias[CT ? (m % (2 * a.co)) >> 1 : m];  // CT: row (ky, oc, kx) has oc's bias
        }
        else bias[mt] = ld4(a.bias + min(w0 + mt * 16 + 4 * g, wout - 4));
    }

    // SH = 1: the two supersteps of the wave's first 32 k's (loads are
    // unconditional, a superstep outside the wave's share re-reads an end of
    // it and is zeroed); SH > 1: its superstep of the first stage.
    float4 xa[4], la[2], ma[4], xb[4], lb[2], mb[4];
    const int par = SH == 1 ? S0 & 1 : 0;  // the share starts at the second superstep of a chunk
    if (SH == 1) {
        load(0, xa, la, ma);
        load(min(1 - par, nSw - 1), xb, lb, mb);
    } else {
        load(0, xa, la, ma);
    }
    if constexpr (LN == 2) {
        static_assert(KS == 4 && LAYOUT == CH, "in-kernel statistics: the split-reduction channel-major form");
        // This lane's rows k = 16 S + 4 g + q of its two supersteps (xa, xb)
        // for pixels xcol .. xcol + 3; lanes i, i + 16, i + 32 and i + 48
        // hold the same pixels, the four waves the four quarters of k.
        __shared__ float4 lst[4][16][2];
        float4 p1 = xa[0], p2 = make_float4(xa[0].x * xa[0].x, xa[0].y * xa[0].y, xa[0].z * xa[0].z, xa[0].w * xa[0].w);
        auto add = [&](const float4 &v) {
            p1.x = p1.x + v.x;
            p1.y = p1.y + v.y;
            p1.z = p1.z + v.z;
            p1.w = p1.w + v.w;
            p2.x = p2.x + v.x * v.x;
            p2.y = p2.y + v.y * v.y;
            p2.z = p2.z + v.z * v.z;
            p2.w = p2.w + v.w * v.w;
        };
#pragma unroll
        for (int q = 1; q < 4; ++q) add(xa[q]);
#pragma unroll
        for (int q = 0; q < 4; ++q) add(xb[q]);
#pragma unroll
        for (int d = 16; d <= 32; d *= 2) {
            p1.x = p1.x + __shfl_xor(p1.x, d);
            p1.y = p1.y + __shfl_xor(p1.y, d);
            p1.z = p1.z + __shfl_xor(p1.z, d);
            p1.w = p1.w + __shfl_xor(p1.w, d);
            p2.x = p2.x + __shfl_xor(p2.x, d);
            p2.y = p2.y + __shfl_xor(p2.y, d);
            p2.z = p2.z + __shfl_xor(p2.z, d);
            p2.w = p2.w + __shfl_xor(p2.w, d);
        }
        if (g == 0) {
            lst[wave][i][0] = p1;
            lst[wave][i][1] = p2;
        }
        __syncthreads();
        float4 s1 = lst[0][i][0], s2 = lst[0][i][1];
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            const float4 t1 = lst[w][i][0], t2 = lst[w][i][1];
            s1.x = s1.x + t1.x;
            s1.y = s1.y + t1.y;
            s1.z = s1.z + t1.z;
            s1.w = s1.w + t1.w;
            s2.x = s2.x + t2.x;
            s2.y = s2.y + t2.y;
            s2.z = s2.z + t2.z;
            s2.w = s2.w + t2.w;
        }
        // mean, then 1 / std, as the LayerNorm statistics kernels form them
        // (K = 128: the product with 1 / K is the quotient to the bit; the
        // reciprocal square root on the transcendental unit, 1 ulp, where
        // those kernels divide by a correctly rounded square root)
        const float inv = 1.0f / (float)K;
        auto stat = [&](float a1, float a2, float &m, float &r) {
            m = a1 * inv;
            const float var = a2 * inv - m * m;
            r = __builtin_amdgcn_rsqf(fmaxf(var, 0.0f) + a.ln.eps);
        };
        stat(s1.x, s2.x, lmean.x, lrstd.x);
        stat(s1.y, s2.y, lmean.y, lrstd.y);
        stat(s1.z, s2.z, lmean.z, lrstd.z);
        stat(s1.w, s2.w, lmean.w, lrstd.w);
    }
    const int64_t cbase = (int64_t)b * a.sC;
    // Slot k of this lane: (mt, x) = (k / 4, k % 4) with KS = 1, and
    // (k, wave) with KS = 4 (the wave's share of the slots).
    constexpr int NK = KS == 1 ? 4 * TMW : TMW;
    // (the lane's first slot offset once; the others differ from it by a
    // wave-uniform amount)
    const int64_t obase = LAYOUT == CH ? (int64_t)(w0 + i) * N + s0 + 4 * g : (int64_t)(s0 + i) * N + w0 + 4 * g;
    auto where = [&](int k, int64_t &off) -> bool {
        const int mt = KS == 1 ? k / 4 : k, x = KS == 1 ? k % 4 : wave;
        if (LAYOUT == CH) {
            const int m = w0 + mt * 16 + i, n = s0 + 16 * x + 4 * g;
            if (fold) {  // batch nb, column n - nb N of it
                const uint32_t nb = mdiv((uint32_t)min(n, slen - 4), a.fmul, a.fsh);
                off = (int64_t)nb * a.sC + (int64_t)(w0 + i + mt * 16) * N + (n - (int)nb * N);
                return m < M && n < slen;
            }
            off = obase + (int64_t)(mt * 16) * N + 16 * x;
            return m < M && n < N;
        }
        const int row = s0 + 16 * x + i, c = w0 + mt * 16 + 4 * g;
        off = obase + (int64_t)(16 * x) * N + mt * 16;
        return row < M && c < N;
    };
    // The fused epilogue's operands are fetched one slot ahead, so their
    // latency overlaps the previous slot's arithmetic and store (the
    // compiler cannot move a load above a store that might alias it).
    // Where output element off (counted from this batch's Y) is stored: off
    // itself, or its image position under a folded backward permutation.
    auto placed = [&](int64_t off) -> int64_t {
        if (!has_ymap) return off;
        const uint32_t e = (uint32_t)(cbase + off), pl = (uint32_t)a.ymap.plane;
        const uint32_t base = mdiv(e, a.ymap.mpl, a.ymap.spl) * pl;
        return (int64_t)(base + unblock(a.ymap, e - base)) - cbase;
    };
    // Each slot's stored position is computed once, with its operands, and
    // serves both the residual read at that position and the store.
    float4 ou[2], o1[2], o2[2];
    int64_t pb[2] = {0, 0};
    auto operands = [&](int k, int buf) {
        int64_t off;
        const bool ok = where(k, off);
        const int64_t at = cbase + (ok ? off : 0);
        pb[buf] = placed(ok ? off : 0);
        if (has_u) ou[buf] = ld4(a.e.u + at);
        if (has_r1) o1[buf] = ld4(a.e.r1 + (r1map ? cbase + pb[buf] : at));
        if (has_r2) o2[buf] = ld4(a.e.r2 + at);
    };
    // A split reduction's wave takes both its slots' operands now, so their
    // latency hides behind the multiplies and the reduction (measured 2-5%
    // faster per launch; a whole-reduction wave keeps fetching one slot
    // ahead in its epilogue, which measured faster there).
    if (FUSED && KS == 4) {
        operands(0, 0);
        if (NK > 1) operands(1, 1);
    }
    // LNO: the wave whose tile is the output LayerNorm's channels keeps its
    // final values for it (and stores them raw only when asked to): with
    // KS = 1 in its own rows of LDS at once, with KS = 4 (where LDS still
    // holds the partial sums) in registers until every wave has read them.
    constexpr int PC = KS == 1 ? 64 : 16;  // pixel columns of a wave's tile
    constexpr int LDT = PC + 4;            // padded LDS row
    constexpr int PER = TW * LDT + 2 * PC;  // LDS floats per wave
    // one LDS pool: X's parts, then the split reduction's partial sums or the
    // output LayerNorm's tiles
    constexpr int STAGE = SH > 1 ? 4 * 64 * 24 : 0, RED = KS == 4 ? 4 * NACC * 64 : 0;
    constexpr int TILES = LNO && KS == 1 ? 4 * PER : 0;
    constexpr int POOL = STAGE > RED ? (STAGE > TILES ? STAGE : TILES) : (RED > TILES ? RED : TILES);
    __shared__ __align__(16) float pool_own[XR || POOL == 0 ? 4 : POOL];
    float *const pool = XR ? xpool : pool_own;
    if constexpr (SH == 1) {
        // chunk cc of the wave's share: supersteps 2 cc - par and the next
        const int nc = LN == 2 ? 1 : (nSw + par + 1) / 2, c0 = S0 >> 1;
        const float4 zero4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        auto step = [&](int cc, bool first) {
            const WParts w = wload(c0 + cc);
            ready(xa, la, ma, kSplitScale);
            ready(xb, lb, mb, kSplitScale);
            if (first && par) {
#pragma unroll
                for (int q = 0; q < 4; ++q) xa[q] = zero4;
            }
            if (2 * cc + 1 - par >= nSw) {
#pragma unroll
                for (int q = 0; q < 4; ++q) xb[q] = zero4;
            }
            auto parts = [&](int j) {
                const Half p = split(xa, j), q = split(xb, j);
                return Parts{u32x4{p.h[0], p.h[1], q.h[0], q.h[1]}, u32x4{p.m[0], p.m[1], q.m[0], q.m[1]},
                             u32x4{p.l[0], p.l[1], q.l[0], q.l[1]}};
            };
            // Two streamed tiles at a time: their accumulators' chains cover
            // each other's latency, and the next two are split meanwhile. The
            // next loads wait for the last two: with all four tiles split
            // before and 32 more registers filling, the split reductions took
            // 172 to 198 VGPRs, two waves a SIMD; now at most 168 and three
            // (with the in-kernel statistics, one chunk, 121 and four; with a
            // folded LayerNorm or Mul 168 to 220 and two). The 128-channel
            // gMLP layer at 56x80, whose 560-block launches then fit at once:
            // 76.9 -> 70.8 us.
            const Parts xs[4] = {parts(0), parts(1), parts(2), parts(3)};
            mul(0, 2, xs, w, first);
            auto next = [&]() {
                if (cc + 1 >= nc) return;
                load(2 * cc + 2 - par, xa, la, ma);
                load(min(2 * cc + 3 - par, nSw - 1), xb, lb, mb);
            };
            if (!XMUL) next();
            mul(2, 2, xs + 2, w, first);
            if (XMUL) next();  // (twice the registers)
        };
        step(0, true);
#pragma unroll 1
        for (int cc = 1; cc < nc; ++cc) step(cc, false);
    } else {
        // The parts of a stage in LDS: [chunk][part][lane group g][64 streamed
        // elements][8 k's], 16 bytes a lane, tile j's sixteen side by side;
        // superstep S fills the half S % 2 of chunk S / 2. Each group of SH
        // waves has its own.
        constexpr int SC = SH / 2;  // chunks per stage
        unsigned char *const sx = (unsigned char *)pool + (wave / SH) * (SH * 6144);
        unsigned char *const wr = sx + ((S0 >> 1) * 12 + g) * 1024 + i * 16 + (S0 & 1) * 8;
        const unsigned char *const rd = sx + g * 1024 + i * 16;
        const int nst = nS / SH;
        auto stage = [&](int st, bool first) {
            WParts w = wload(st * SC);
            ready(xa, la, ma, kSplitScale);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const Half p = split(xa, j);
                *(uint2 *)(wr + j * 256) = make_uint2(p.h[0], p.h[1]);
                *(uint2 *)(wr + 4096 + j * 256) = make_uint2(p.m[0], p.m[1]);
                *(uint2 *)(wr + 8192 + j * 256) = make_uint2(p.l[0], p.l[1]);
            }
            __syncthreads();
            WParts wn = w;
            if (SC > 1) wn = wload(st * SC + 1);
            if (st + 1 < nst) load((st + 1) * SH, xa, la, ma);
#pragma unroll
            for (int cc = 0; cc < SC; ++cc) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const unsigned char *r = rd + cc * 12288 + j * 256;
                    const Parts x = {*(const u32x4 *)r, *(const u32x4 *)(r + 4096), *(const u32x4 *)(r + 8192)};
                    mul(j, 1, &x, cc ? wn : w, first && cc == 0);
                }
            }
        };
        stage(0, true);
#pragma unroll 1
        for (int st = 1; st < nst; ++st) {
            __syncthreads();  // every wave has read the last stage's parts
            stage(st, false);
        }
        if (LNO) __syncthreads();
    }
    // An operand the split cannot hold (infinite, NaN, the largest floats)
    // leaves no finite sum in its outputs, and sums may overflow: a wave that
    // has such sums forms them in fp32, superstep by superstep, and keeps the
    // others, so that no output depends on what else is in its tile.
    float top = 0.0f;  // (the maximum that keeps a NaN)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int mt = 0; mt < TMW; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) top = __builtin_elementwise_maximum(top, __builtin_fabsf(acc[j][mt][r]));
    float us = kUnsplit;  // what the sums are multiplied by
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!__builtin_isfinite(top)) != 0, 0)) {
        us = 1.0f;
        const int first = SH > 1 ? -S0 : 0;
        const float *wp[TMW];
#pragma unroll
        for (int mt = 0; mt < TMW; ++mt)
            wp[mt] = W + (int64_t)min(w0 + mt * 16 + i, wout - 1) * K + 4 * g + (S0 + first) * 16;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32x4 f[TMW];
#pragma unroll
            for (int mt = 0; mt < TMW; ++mt) f[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (int s = 0; s < nSw; ++s) {
                float4 wv[TMW];
                load(first + s, xa, la, ma);
#pragma unroll
                for (int mt = 0; mt < TMW; ++mt) wv[mt] = ld4(wp[mt] + s * 16);
                ready(xa, la, ma, 1.0f);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int mt = 0; mt < TMW; ++mt)
                        f[mt] = LAYOUT == CH ? mfma16(comp(xa[t], j), comp(wv[mt], t), f[mt])
                                             : mfma16(comp(wv[mt], t), comp(xa[j], t), f[mt]);
            }
#pragma unroll
            for (int mt = 0; mt < TMW; ++mt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[j][mt][r] = __builtin_isfinite(acc[j][mt][r]) ? acc[j][mt][r] * kUnsplit : f[mt][r];
        }
    }

    float *const red = pool;
    __shared__ __align__(16) float rus[KS == 4 ? 4 : 1];  // each wave's us
    if (KS == 4) {
        if (lane == 0) rus[wave] = us;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int mt = 0; mt < TMW; ++mt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    red[((wave * NACC) + (j * TMW + mt) * 4 + r) * 64 + lane] = acc[j][mt][r];
        __syncthreads();
    }
    float *const lt = pool;
    const int lnspan = (KS == 1 ? a.lo.group : 1) * TW * a.lo.nband;  // rows with a LayerNorm
    const bool lnw = LNO && w0 >= a.lo.row0 && w0 < a.lo.row0 + lnspan;
    float4 vs[LNO && KS == 4 ? NK : 1];
    float4 us4;
    if (KS == 4) us4 = ld4(rus);
    if (FUSED && KS == 1) operands(0, 0);
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        if (LNO && KS == 4) vs[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (FUSED && k + 1 < NK && (KS == 1 || k + 1 > 1)) operands(k + 1, (k + 1) & 1);
        const int mt = KS == 1 ? k / 4 : k, x = KS == 1 ? k % 4 : wave;
        // Out-of-range slots run the arithmetic on clamped operands and skip
        // only the global stores, so the uniform branches below stay
        // uniform (no lane-divergent region around them).
        int64_t off;
        const bool inside = where(k, off);
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            // CH: v[u] = Y[m][n + u] is acc[u][mt][x]; RW: v[u] = Y[row][c + u] is acc[x][mt][u]
            const int j = LAYOUT == CH ? u : x, r = LAYOUT == CH ? x : u;
            // (a product with a power of two and one rounding of the sum)
            const float bb = !has_bias ? 0.0f : LAYOUT == CH ? bias[mt].x : comp(bias[mt], u);
            if (KS == 1) {
                v[u] = has_bias ? __builtin_fmaf(acc[j][mt][r], us, bb) : acc[j][mt][r] * us;
            } else {
                const int q = (j * TMW + mt) * 4 + r;
                float t = red[q * 64 + lane] * us4.x;
                t = __builtin_fmaf(red[(NACC + q) * 64 + lane], us4.y, t);
                t = __builtin_fmaf(red[(2 * NACC + q) * 64 + lane], us4.z, t);
                t = __builtin_fmaf(red[(3 * NACC + q) * 64 + lane], us4.w, t);
                v[u] = has_bias ? bb + t : t;
            }
        }
        if (FUSED) {
            const int bi = k & 1;
            if (has_u) {
                v[0] = ou[bi].x * (v[0] + 1.0f);
                v[1] = ou[bi].y * (v[1] + 1.0f);
                v[2] = ou[bi].z * (v[2] + 1.0f);
                v[3] = ou[bi].w * (v[3] + 1.0f);
            }
            if (has_gelu) {
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = gelu(v[u]);
            } else if (has_lrelu) {
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = v[u] >= 0.0f ? v[u] : a.e.slope * v[u];
            }
            if (has_r1) {
                v[0] = v[0] + o1[bi].x;
                v[1] = v[1] + o1[bi].y;
                v[2] = v[2] + o1[bi].z;
                v[3] = v[3] + o1[bi].w;
            }
            if (has_r2) {
                v[0] = v[0] + o2[bi].x;
                v[1] = v[1] + o2[bi].y;
                v[2] = v[2] + o2[bi].z;
                v[3] = v[3] + o2[bi].w;
            }
        }
        if (CT) {
            // Transposed 2x2 stride-2 conv: row m = (ky * co + oc) * 2 + kx, so
            // lanes i and i ^ 1 hold kx = 0 and 1 of one (ky, oc) for the same
            // four input pixels (x .. x + 3 of input row y): together the eight
            // contiguous outputs 2x .. 2x + 7 of output row 2y + ky, four each.
            float pv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) pv[u] = __shfl_xor(v[u], 1);
            if (!inside) continue;
            const int m = w0 + mt * 16 + i, two = 2 * a.co;
            const int ky = m / two, rem = m - ky * two, oc = rem >> 1, kx = rem & 1;
            const int n = (int)(off - (int64_t)m * N), y = n / a.wd, xx = n - y * a.wd;
            float *o = Y + (int64_t)oc * 4 * N + (int64_t)(2 * y + ky) * (2 * a.wd) + 2 * xx + 4 * kx;
            st4(o, kx == 0 ? make_float4(v[0], pv[0], v[1], pv[1]) : make_float4(pv[2], v[2], pv[3], v[3]));
            continue;
        }
        if (LNO && lnw) {
            if (KS == 1)
                st4(lt + wave * PER + (mt * 16 + i) * LDT + 16 * x + 4 * g, make_float4(v[0], v[1], v[2], v[3]));
            else
                vs[k] = make_float4(v[0], v[1], v[2], v[3]);
            if (!a.lo.keep) continue;
        }
        if (inside) st4(Y + (FUSED ? pb[k & 1] : placed(off)), make_float4(v[0], v[1], v[2], v[3]));
    }
    if constexpr (LNO) {
        // Per pixel, the LayerNorm's statistics in the LayerNorm kernels'
        // order (ascending channel, one pass for s1 and s2): the tiles go
        // through LDS so that one lane reads a pixel's channels in turn; then
        // every lane normalises the values it holds with the LayerNorm's
        // expression (mode 0), or writes the statistics (mode 1). A band's
        // G * TW channels are the tiles of G consecutive waves of one block
        // (G = lo.group; G = 1 with KS = 4).
        // With G = 1 the exchange stays within the wave (its own LDS rows)
        // and needs no block barrier; with G > 1 every wave of a block that
        // holds a group takes both barriers (block-uniform, and the host
        // launches whole blocks of tiles, so no wave has left early).
        const int G = KS == 1 ? a.lo.group : 1;
        bool any = lnw;
        if (KS == 1 && G > 1) {
            any = false;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int bw = ((unit * 4 + j) % nib) * TW;
                any = any || (bw >= a.lo.row0 && bw < a.lo.row0 + lnspan);
            }
        }
        if (any) {
            float *t;
            if constexpr (KS == 1) {
                t = lt + wave * PER;
            } else {
                static_assert(4 * PER <= 4 * NACC * 64, "the reduction buffer holds the exchange");
                __syncthreads();  // every wave has read its sums out of red
                t = red + wave * PER;
#pragma unroll
                for (int k = 0; k < NK; ++k) st4(t + (k * 16 + i) * LDT + 4 * g, vs[k]);
            }
            auto sync = [&]() {
                if (G > 1) {
                    __syncthreads();
                } else {
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                }
            };
            const int band = lnw ? (w0 - a.lo.row0) / (G * TW) : 0;
            const int lq = lnw ? (w0 - a.lo.row0) / TW - band * G : 0;  // place in the group
            // mode 0: this wave's values of the band, normalised with the
            // statistics at ts (mean row, then 1 / std row) and stored
            auto normalise = [&](const float *ts) {
                float lw[TMW], lb[TMW];
#pragma unroll
                for (int mt = 0; mt < TMW; ++mt) {
                    lw[mt] = a.lo.scale[lq * TW + mt * 16 + i];
                    lb[mt] = a.lo.bias[lq * TW + mt * 16 + i];
                }
                float *ly = a.lo.y - (int64_t)a.lo.row0 * N;  // indexed like Y (one batch)
#pragma unroll
                for (int k = 0; k < NK; ++k) {
                    const int mt = KS == 1 ? k / 4 : k, x = KS == 1 ? k % 4 : 0;
                    int64_t off;
                    if (!where(k, off)) continue;
                    const float4 m4 = ld4(ts + 16 * x + 4 * g);
                    const float4 r4 = ld4(ts + PC + 16 * x + 4 * g);
                    const float w = lw[mt], c = lb[mt];
                    float4 y = ld4(t + (mt * 16 + i) * LDT + 16 * x + 4 * g);
                    y.x = (y.x - m4.x) * r4.x * w + c;
                    y.y = (y.y - m4.y) * r4.y * w + c;
                    y.z = (y.z - m4.z) * r4.z * w + c;
                    y.w = (y.w - m4.w) * r4.w * w + c;
                    st4(ly + off, y);
                }
            };
            // (G TW is a power of two, so the product with its reciprocal is
            // the quotient to the bit; with the per-wave partial sums, whose
            // order already differs from the LayerNorm kernels', 1 / std is
            // the transcendental unit's reciprocal square root, 1 ulp)
            const float inv = 1.0f / (float)(G * TW);
            auto stats = [&](float s1, float s2, int n_at) {
                const float m = s1 * inv;
                const float var = s2 * inv - m * m;
                const float r = a.lo.order ? __builtin_amdgcn_rsqf(fmaxf(var, 0.0f) + a.lo.eps)
                                           : 1.0f / sqrtf(fmaxf(var, 0.0f) + a.lo.eps);
                if (a.lo.mode) {  // the statistics only, at the pixel's image position
                    const int n = s0 + n_at;
                    if (n < N) {
                        float *sy = a.lo.y + (int64_t)band * 2 * N;
                        const int64_t at = placed(n);
                        sy[at] = m;
                        sy[N + at] = r;
                    }
                } else {
                    t[TW * LDT + lane] = m;
                    t[TW * LDT + PC + lane] = r;
                }
            };
            if (KS == 1 && TW >= 32 && G > 1 && a.lo.order) {
                // Each wave of the group sums its own channels of a pixel
                // (its own LDS rows: a wave barrier), the partial sums meet
                // in LDS (one block barrier), and every wave adds the
                // group's partials in wave order and keeps the statistics
                // it needs (its own rows again). A wave's partial sums of
                // pixel p sit in its tile's row padding: s1 in rows 0..15,
                // s2 in rows 16..31, column PC + p % 4 of row p / 4 (the
                // padding holds 4 TW >= 2 PC floats and is read nowhere else).
                auto pad = [&](int which, int p) { return (which * 16 + (p >> 2)) * LDT + PC + (p & 3); };
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (lnw) {
                    float p1 = 0.0f, p2 = 0.0f;
#pragma unroll 8
                    for (int c = 0; c < TW; ++c) {
                        const float v = t[c * LDT + lane];
                        p1 += v;
                        p2 += v * v;
                    }
                    t[pad(0, lane)] = p1;
                    t[pad(1, lane)] = p2;
                }
                __syncthreads();
                if (lnw) {
                    const float *g0 = t - lq * PER;
                    float s1 = g0[pad(0, lane)], s2 = g0[pad(1, lane)];
                    for (int q = 1; q < G; ++q) {
                        s1 = s1 + g0[q * PER + pad(0, lane)];
                        s2 = s2 + g0[q * PER + pad(1, lane)];
                    }
                    if (!a.lo.mode || lq == 0) stats(s1, s2, KS == 1 ? lane : 16 * wave + lane);
                }
                if (!a.lo.mode) {
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                }
                if (lnw && !a.lo.mode) normalise(t + TW * LDT);
            } else {
                sync();
                if (lnw && lq == 0 && lane < PC) {
                    float s1 = 0.0f, s2 = 0.0f;
                    for (int q = 0; q < G; ++q) {
#pragma unroll 8
                        for (int c = 0; c < TW; ++c) {
                            const float v = t[q * PER + c * LDT + lane];
                            s1 += v;
                            s2 += v * v;
                        }
                    }
                    stats(s1, s2, KS == 1 ? lane : 16 * wave + lane);
                }
                if (!a.lo.mode) sync();
                if (lnw && !a.lo.mode) normalise(t - lq * PER + TW * LDT);  // the group's statistics
            }
        }
    }
}

}  // namespace pw

// mx_pw_{ch,rw}<TMW>[_k4|_s2|_s4][_ln|_xm|_mul][_f]: 256 threads; _k4 splits the
// reduction over the block's four waves, _s<SH> shares X between SH of them, _ln folds a channel LayerNorm into X
// (CH only), _xm reads X through a token map (GateMm over an elided forward
// permutation), _mul forms X as the product of two tensors (a folded Mul, CH
// only), _f applies the fused epilogue. mx_pw_ch<TMW>[_k4]_t: the transposed
// 2x2 stride-2 conv (rows ordered (ky, oc, kx), co and the input width in
// GemmArgs co / wd, wd % 4 == 0).
#define MXK_PWF(LNAME, LAYOUT, TMW, KS, LN, XM, XMUL, SH, SUF)                                     \
    extern "C" __global__ __launch_bounds__(256) void mx_pw_##LNAME##TMW##SUF##_f(GemmArgs a) {    \
        pw::body<pw::LAYOUT, TMW, KS, true, LN, XM, XMUL, false, false, -1, false, false, SH>(     \
            a, blockIdx.x, gridDim.x, blockIdx.y);                                                 \
    }
#define MXK_PW3(LNAME, LAYOUT, TMW, KS, LN, XM, XMUL, SH, SUF)                                     \
    extern "C" __global__ __launch_bounds__(256) void mx_pw_##LNAME##TMW##SUF(GemmArgs a) {        \
        pw::body<pw::LAYOUT, TMW, KS, false, LN, XM, XMUL, false, false, -1, false, false, SH>(    \
            a, blockIdx.x, gridDim.x, blockIdx.y);                                                 \
    }                                                                                              \
    MXK_PWF(LNAME, LAYOUT, TMW, KS, LN, XM, XMUL, SH, SUF)
#define MXK_PW2(LNAME, LAYOUT, TMW, KS, LN, XM, XMUL, SUF) MXK_PW3(LNAME, LAYOUT, TMW, KS, LN, XM, XMUL, 1, SUF)
#define MXK_PW1(LNAME, LAYOUT, TMW, KS, LN, XM, SUF) MXK_PW2(LNAME, LAYOUT, TMW, KS, LN, XM, false, SUF)
// _s<SH>: X shared by SH waves of a block
#define MXK_PW_S(LNAME, LAYOUT, TMW, SH)                                                           \
    MXK_PW3(LNAME, LAYOUT, TMW, 1, 0, false, false, SH, _s##SH)                                    \
    MXK_PW3(LNAME, LAYOUT, TMW, 1, 0, true, false, SH, _s##SH##_xm)
#define MXK_PW_CHS(TMW, SH)                                                                        \
    MXK_PW_S(ch, CH, TMW, SH)                                                                      \
    MXK_PW3(ch, CH, TMW, 1, 1, false, false, SH, _s##SH##_ln)                                      \
    MXK_PW3(ch, CH, TMW, 1, 0, false, true, SH, _s##SH##_mul)                                      \
    MXK_PW_CT(TMW, 1, SH, _s##SH)                                                                  \
    MXK_PWB1(TMW, 1, false, SH, _s##SH) MXK_PWB1(TMW, 1, true, SH, _s##SH##_xm)
#define MXK_PW(LNAME, LAYOUT, TMW)                                                                 \
    MXK_PW1(LNAME, LAYOUT, TMW, 1, false, false, ) MXK_PW1(LNAME, LAYOUT, TMW, 4, false, false, _k4) \
    MXK_PW1(LNAME, LAYOUT, TMW, 1, false, true, _xm) MXK_PW1(LNAME, LAYOUT, TMW, 4, false, true, _k4_xm)
#define MXK_PW_LN(TMW) MXK_PW1(ch, CH, TMW, 1, 1, false, _ln) MXK_PW1(ch, CH, TMW, 4, 1, false, _k4_ln)
// _k4_ln2: the LayerNorm statistics computed by the block itself (LN = 2)
MXK_PW1(ch, CH, 2, 4, 2, false, _k4_ln2)
#define MXK_PW_CT(TMW, KS, SH, SUF)                                                                \
    extern "C" __global__ __launch_bounds__(256) void mx_pw_ch##TMW##SUF##_t(GemmArgs a) {         \
        pw::body<pw::CH, TMW, KS, false, 0, false, false, true, false, -1, false, false, SH>(      \
            a, blockIdx.x, gridDim.x, blockIdx.y);                                                 \
    }
// mx_pw_ch<TMW>[_k4][_ln]_f_lo: with a LayerNorm of one wave-wide band of
// the output rows (GemmArgs lo).
#define MXK_PW_LO(TMW, KS, LN, SH, SUF)                                                            \
    extern "C" __global__ __launch_bounds__(256) void mx_pw_ch##TMW##SUF##_f_lo(GemmArgs a) {      \
        pw::body<pw::CH, TMW, KS, true, LN, false, false, false, true, -1, false, false, SH>(      \
            a, blockIdx.x, gridDim.x, blockIdx.y);                                                 \
    }
#define MXK_PW_MUL(TMW) \
    MXK_PW2(ch, CH, TMW, 1, false, false, true, _mul) MXK_PW2(ch, CH, TMW, 4, false, false, true, _k4_mul)
// mx_pw_chb<TMW>[_k4][_xm][_f]: channel-major over a folded batch (GemmArgs
// fold; GateMm mode 0, whose channels are the batch)
#define MXK_PWB1(TMW, KS, XM, SH, SUF)                                                             \
    extern "C" __global__ __launch_bounds__(256) void mx_pw_chb##TMW##SUF(GemmArgs a) {            \
        pw::body<pw::CH, TMW, KS, false, 0, XM, false, false, false, -1, true, false, SH>(         \
            a, blockIdx.x, gridDim.x, 0);                                                          \
    }                                                                                              \
    extern "C" __global__ __launch_bounds__(256) void mx_pw_chb##TMW##SUF##_f(GemmArgs a) {        \
        pw::body<pw::CH, TMW, KS, true, 0, XM, false, false, false, -1, true, false, SH>(          \
            a, blockIdx.x, gridDim.x, 0);                                                          \
    }
#define MXK_PWB(TMW)                                                                               \
    MXK_PWB1(TMW, 1, false, 1, ) MXK_PWB1(TMW, 4, false, 1, _k4)                                   \
    MXK_PWB1(TMW, 1, true, 1, _xm) MXK_PWB1(TMW, 4, true, 1, _k4_xm)
MXK_PW(ch, CH, 1)
MXK_PW(ch, CH, 2)
MXK_PW(ch, CH, 4)
MXK_PWB(1)
MXK_PWB(2)
MXK_PWB(4)
MXK_PW(rw, RW, 1)
MXK_PW(rw, RW, 2)
MXK_PW(rw, RW, 4)
MXK_PW_LN(1)
MXK_PW_LN(2)
MXK_PW_LN(4)
MXK_PW_MUL(1)
MXK_PW_MUL(2)
MXK_PW_MUL(4)
MXK_PW_CT(1, 1, 1, )
MXK_PW_CT(1, 4, 1, _k4)
MXK_PW_CT(2, 1, 1, )
MXK_PW_CT(2, 4, 1, _k4)
MXK_PW_CT(4, 1, 1, )
MXK_PW_CT(4, 4, 1, _k4)
// 16-wide tiles share X only where a step of 17 to 32 outputs with a residual
// takes them (with_epilogue): the fused forms of two waves
MXK_PWF(ch, CH, 1, 1, 0, false, false, 2, _s2)
MXK_PWF(ch, CH, 1, 1, 0, true, false, 2, _s2_xm)
MXK_PWF(ch, CH, 1, 1, 1, false, false, 2, _s2_ln)
MXK_PWF(ch, CH, 1, 1, 0, false, true, 2, _s2_mul)
MXK_PW_CHS(2, 2)
MXK_PW_CHS(2, 4)
MXK_PW_S(rw, RW, 2, 2)
MXK_PW_S(rw, RW, 2, 4)
MXK_PW_LO(1, 1, 0, 1, )
MXK_PW_LO(2, 1, 0, 1, )
MXK_PW_LO(2, 4, 0, 1, _k4)
MXK_PW_LO(2, 1, 1, 1, _ln)
MXK_PW_LO(2, 4, 1, 1, _k4_ln)
MXK_PW_LO(4, 1, 0, 1, )
MXK_PW_LO(4, 4, 0, 1, _k4)
MXK_PW_LO(4, 1, 1, 1, _ln)
MXK_PW_LO(4, 4, 1, 1, _k4_ln)
MXK_PW_LO(1, 1, 0, 2, _s2)
MXK_PW_LO(2, 1, 0, 2, _s2)
MXK_PW_LO(2, 1, 0, 4, _s4)
MXK_PW_LO(2, 1, 1, 2, _s2_ln)
MXK_PW_LO(2, 1, 1, 4, _s4_ln)

// mx_pw_..._f[_lo]_e<EP>: a fused streaming kernel specialised for one
// epilogue operand set (pw::EP_* mask), for the combinations the MAXIM
// program launches most; the host takes one when it exists and the generic
// _f kernel otherwise (the same arithmetic in the same order).
#define MXK_PW_ES(NAME, LAYOUT, TMW, KS, LN, XM, XMUL, LNO, FOLD, SH, EP)                          \
    extern "C" __global__ __launch_bounds__(256) void NAME##_e##EP(GemmArgs a) {                   \
        pw::body<pw::LAYOUT, TMW, KS, true, LN, XM, XMUL, false, LNO, EP, FOLD, false, SH>(        \
            a, blockIdx.x, gridDim.x, FOLD ? 0 : blockIdx.y);                                      \
    }
#define MXK_PW_E(NAME, LAYOUT, TMW, KS, LN, XM, XMUL, LNO, EP) \
    MXK_PW_ES(NAME, LAYOUT, TMW, KS, LN, XM, XMUL, LNO, false, 1, EP)
// NAME_e<EP>_x2: two independent launches of that kernel as one grid (the
// first d.na blocks run d.a, the rest d.b; one batch each), so that two
// steps too small to fill the chip share its CUs and one launch's tail. Both
// parts run the same function, so they share its LDS.
#define MXK_PW_X2S(NAME, LAYOUT, TMW, KS, LN, XM, XMUL, LNO, SH, EP)                               \
    extern "C" __global__ __launch_bounds__(256) void NAME##_e##EP##_x2(DualGemmArgs d) {          \
        if (blockIdx.x < d.na)                                                                     \
            pw::body<pw::LAYOUT, TMW, KS, true, LN, XM, XMUL, false, LNO, EP, false, false, SH>(   \
                d.a, blockIdx.x, d.na, 0);                                                         \
        else                                                                                       \
            pw::body<pw::LAYOUT, TMW, KS, true, LN, XM, XMUL, false, LNO, EP, false, false, SH>(   \
                d.b, blockIdx.x - d.na, gridDim.x - d.na, 0);                                      \
    }
#define MXK_PW_X2(NAME, LAYOUT, TMW, KS, LN, XM, XMUL, LNO, EP) \
    MXK_PW_X2S(NAME, LAYOUT, TMW, KS, LN, XM, XMUL, LNO, 1, EP)
MXK_PW_E(mx_pw_ch2_ln_f_lo, CH, 2, 1, 1, false, false, true, 72)
MXK_PW_E(mx_pw_ch4_k4_ln_f_lo, CH, 4, 4, 1, false, false, true, 72)
MXK_PW_E(mx_pw_ch2_ln_f, CH, 2, 1, 1, false, false, false, 72)
MXK_PW_E(mx_pw_ch2_k4_ln_f, CH, 2, 4, 1, false, false, false, 72)
MXK_PW_E(mx_pw_ch2_k4_ln2_f, CH, 2, 4, 2, false, false, false, 72)
MXK_PW_E(mx_pw_ch2_f_lo, CH, 2, 1, 0, false, false, true, 64)
MXK_PW_E(mx_pw_ch2_f_lo, CH, 2, 1, 0, false, false, true, 66)
MXK_PW_E(mx_pw_ch1_f_lo, CH, 1, 1, 0, false, false, true, 66)
MXK_PW_E(mx_pw_ch2_k4_f_lo, CH, 2, 4, 0, false, false, true, 64)
MXK_PW_E(mx_pw_ch2_k4_f_lo, CH, 2, 4, 0, false, false, true, 66)
MXK_PW_E(mx_pw_ch4_k4_f_lo, CH, 4, 4, 0, false, false, true, 64)
MXK_PW_E(mx_pw_ch4_k4_f_lo, CH, 4, 4, 0, false, false, true, 66)
MXK_PW_E(mx_pw_ch1_f, CH, 1, 1, 0, false, false, false, 226)
MXK_PW_E(mx_pw_ch2_f, CH, 2, 1, 0, false, false, false, 64)
MXK_PW_E(mx_pw_ch2_f, CH, 2, 1, 0, false, false, false, 226)
MXK_PW_E(mx_pw_ch2_k4_f, CH, 2, 4, 0, false, false, false, 64)
MXK_PW_E(mx_pw_ch2_k4_f, CH, 2, 4, 0, false, false, false, 65)
MXK_PW_E(mx_pw_ch2_k4_f, CH, 2, 4, 0, false, false, false, 66)
MXK_PW_E(mx_pw_ch2_k4_f, CH, 2, 4, 0, false, false, false, 226)
MXK_PW_E(mx_pw_ch1_mul_f, CH, 1, 1, 0, false, true, false, 66)
MXK_PW_E(mx_pw_ch1_mul_f, CH, 1, 1, 0, false, true, false, 70)
MXK_PW_E(mx_pw_ch2_mul_f, CH, 2, 1, 0, false, true, false, 66)
MXK_PW_E(mx_pw_ch2_mul_f, CH, 2, 1, 0, false, true, false, 70)
MXK_PW_E(mx_pw_ch2_k4_mul_f, CH, 2, 4, 0, false, true, false, 66)
MXK_PW_E(mx_pw_ch2_k4_mul_f, CH, 2, 4, 0, false, true, false, 70)
MXK_PW_E(mx_pw_rw2_k4_f, RW, 2, 4, 0, false, false, false, 65)
MXK_PW_ES(mx_pw_chb2_k4_f, CH, 2, 4, 0, false, false, false, true, 1, 65)
// with X shared by two or four waves
#define MXK_PW_ESS(SH)                                                                  \
    MXK_PW_ES(mx_pw_ch2_s##SH##_ln_f_lo, CH, 2, 1, 1, false, false, true, false, SH, 72) \
    MXK_PW_ES(mx_pw_ch2_s##SH##_ln_f, CH, 2, 1, 1, false, false, false, false, SH, 72)   \
    MXK_PW_ES(mx_pw_ch2_s##SH##_f_lo, CH, 2, 1, 0, false, false, true, false, SH, 64)    \
    MXK_PW_ES(mx_pw_ch2_s##SH##_f_lo, CH, 2, 1, 0, false, false, true, false, SH, 66)    \
    MXK_PW_ES(mx_pw_ch2_s##SH##_f, CH, 2, 1, 0, false, false, false, false, SH, 64)      \
    MXK_PW_ES(mx_pw_ch2_s##SH##_f, CH, 2, 1, 0, false, false, false, false, SH, 66)      \
    MXK_PW_ES(mx_pw_ch2_s##SH##_f, CH, 2, 1, 0, false, false, false, false, SH, 226)     \
    MXK_PW_ES(mx_pw_ch2_s##SH##_mul_f, CH, 2, 1, 0, false, true, false, false, SH, 66)   \
    MXK_PW_ES(mx_pw_ch2_s##SH##_mul_f, CH, 2, 1, 0, false, true, false, false, SH, 70)   \
    MXK_PW_ES(mx_pw_rw2_s##SH##_f, RW, 2, 1, 0, false, false, false, false, SH, 65)      \
    MXK_PW_ES(mx_pw_chb2_s##SH##_f, CH, 2, 1, 0, false, false, false, true, SH, 65)      \
    MXK_PW_X2S(mx_pw_ch2_s##SH##_ln_f_lo, CH, 2, 1, 1, false, false, true, SH, 72)       \
    MXK_PW_X2S(mx_pw_ch2_s##SH##_ln_f, CH, 2, 1, 1, false, false, false, SH, 72)         \
    MXK_PW_X2S(mx_pw_ch2_s##SH##_f, CH, 2, 1, 0, false, false, false, SH, 226)
MXK_PW_ESS(2)
MXK_PW_ESS(4)
MXK_PW_ES(mx_pw_ch1_s2_f_lo, CH, 1, 1, 0, false, false, true, false, 2, 66)
MXK_PW_ES(mx_pw_ch1_s2_f, CH, 1, 1, 0, false, false, false, false, 2, 226)
MXK_PW_ES(mx_pw_ch1_s2_mul_f, CH, 1, 1, 0, false, true, false, false, 2, 66)
MXK_PW_ES(mx_pw_ch1_s2_mul_f, CH, 1, 1, 0, false, true, false, false, 2, 70)
MXK_PW_X2S(mx_pw_ch1_s2_f, CH, 1, 1, 0, false, false, false, 2, 226)
MXK_PW_E(mx_pw_rw4_k4_f, RW, 4, 4, 0, false, false, false, 65)
MXK_PW_X2(mx_pw_ch2_ln_f_lo, CH, 2, 1, 1, false, false, true, 72)
MXK_PW_X2(mx_pw_ch1_f, CH, 1, 1, 0, false, false, false, 226)
MXK_PW_X2(mx_pw_ch2_f, CH, 2, 1, 0, false, false, false, 226)
MXK_PW_X2(mx_pw_ch2_k4_f, CH, 2, 4, 0, false, false, false, 226)
MXK_PW_X2(mx_pw_ch2_k4_ln2_f, CH, 2, 4, 2, false, false, false, 72)
// A__B_x2: two different split-reduction GEMMs, independent of each other,
// side by side in one grid (the first d.na blocks run A, the rest B) with one
// reduction buffer for both (each instance would otherwise bring its own and
// halve the blocks per CU): the grid and block branches' GateMms of a
// multi-axis gMLP block, mode 0 over a folded batch and mode 1.
extern "C" __global__ __launch_bounds__(256) void mx_pw_chb2_k4_xm__rw2_k4_xm_x2(DualGemmArgs d) {
    __shared__ float red[4 * 32 * 64];
    if (blockIdx.x < d.na)
        pw::body<pw::CH, 2, 4, false, 0, true, false, false, false, -1, true, true>(d.a, blockIdx.x, d.na, 0, red);
    else
        pw::body<pw::RW, 2, 4, false, 0, true, false, false, false, -1, false, true>(d.b, blockIdx.x - d.na,
                                                                                      gridDim.x - d.na, 0, red);
}
extern "C" __global__ __launch_bounds__(256) void mx_pw_chb2_k4_f_e65__rw2_k4_f_e65_x2(DualGemmArgs d) {
    __shared__ float red[4 * 32 * 64];
    if (blockIdx.x < d.na)
        pw::body<pw::CH, 2, 4, true, 0, false, false, false, false, 65, true, true>(d.a, blockIdx.x, d.na, 0, red);
    else
        pw::body<pw::RW, 2, 4, true, 0, false, false, false, false, 65, false, true>(d.b, blockIdx.x - d.na,
                                                                                      gridDim.x - d.na, 0, red);
}
// and with X shared by four waves
extern "C" __global__ __launch_bounds__(256) void mx_pw_chb2_s4_xm__rw2_s4_xm_x2(DualGemmArgs d) {
    __shared__ __align__(16) float pool[4 * 64 * 24];
    if (blockIdx.x < d.na)
        pw::body<pw::CH, 2, 1, false, 0, true, false, false, false, -1, true, true, 4>(d.a, blockIdx.x, d.na, 0, pool);
    else
        pw::body<pw::RW, 2, 1, false, 0, true, false, false, false, -1, false, true, 4>(d.b, blockIdx.x - d.na,
                                                                                         gridDim.x - d.na, 0, pool);
}
extern "C" __global__ __launch_bounds__(256) void mx_pw_chb2_s4_f_e65__rw2_s4_f_e65_x2(DualGemmArgs d) {
    __shared__ __align__(16) float pool[4 * 64 * 24];
    if (blockIdx.x < d.na)
        pw::body<pw::CH, 2, 1, true, 0, false, false, false, false, 65, true, true, 4>(d.a, blockIdx.x, d.na, 0, pool);
    else
        pw::body<pw::RW, 2, 1, true, 0, false, false, false, false, 65, false, true, 4>(d.b, blockIdx.x - d.na,
                                                                                         gridDim.x - d.na, 0, pool);
}
// the out-projections of the two branches at the smallest resolutions: a
// residual add (grid branch), and a residual add into a backward permutation
// (block branch)
extern "C" __global__ __launch_bounds__(256) void mx_pw_ch2_k4_f_e66__ch2_k4_f_e226_x2(DualGemmArgs d) {
    __shared__ float red[4 * 32 * 64];
    if (blockIdx.x < d.na)
        pw::body<pw::CH, 2, 4, true, 0, false, false, false, false, 66, false, true>(d.a, blockIdx.x, d.na, 0, red);
    else
        pw::body<pw::CH, 2, 4, true, 0, false, false, false, false, 226, false, true>(d.b, blockIdx.x - d.na,
                                                                                       gridDim.x - d.na, 0, red);
}
// the unfused split-reduction kernel (a GEMM with no epilogue), paired
extern "C" __global__ __launch_bounds__(256) void mx_pw_ch2_k4_x2(DualGemmArgs d) {
    if (blockIdx.x < d.na)
        pw::body<pw::CH, 2, 4, false, 0, false, false>(d.a, blockIdx.x, d.na, 0);
    else
        pw::body<pw::CH, 2, 4, false, 0, false, false>(d.b, blockIdx.x - d.na, gridDim.x - d.na, 0);
}

// The weights of every streaming GEMM in bf16 parts (SplitEntry): one block a
// 16-row tile, one wave a chunk of 32 k's, one launch per executor (a launch
// per matrix, 30 to 800 of them, took 3.4 us each).
extern "C" __global__ __launch_bounds__(256) void mx_split_w(SplitArgs s) {
    int lo = 0, hi = s.n;  // the last entry that starts at or before this block
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (s.table[mid].first <= (int)blockIdx.x) lo = mid;
        else hi = mid;
    }
    const SplitEntry a = s.table[lo];
    const float *w = (const float *)s.base + a.w;
    const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    const int tile = blockIdx.x - a.first;
    const int nC = (a.K + 31) / 32, row = tile * 16 + i;
    for (int c = threadIdx.x >> 6; c < nC; c += 4) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int k = 32 * c + 16 * (e >> 2) + 4 * g + (e & 3);
            v[e] = row < a.M && k < a.K ? w[(int64_t)row * a.K + k] : 0.0f;
        }
        u32x4 p[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t h, m, l;
            split2(v[2 * e] * kSplitScale, v[2 * e + 1] * kSplitScale, h, m, l);
            p[0][e] = h;
            p[1][e] = m;
            p[2][e] = l;
        }
        u32x4 *o = (u32x4 *)((unsigned char *)s.base + a.out) + ((int64_t)tile * nC + c) * 192 + lane;
        o[0] = p[0];
        o[64] = p[1];
        o[128] = p[2];
    }
}
