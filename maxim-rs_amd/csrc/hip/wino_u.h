// 3x3 convolution (pad 1) at any image width by Winograd's minimal filtering
// F(2x2, 3x3) (wino.h has the transforms and their matrices), its products
// formed from three-part bf16 operands (common.h; the halo is scaled as it is
// staged, U by the host).
//
// A block owns 32 output channels x 2 x 16 tiles (4 x 32 output pixels) and
// walks the input channels in chunks of 16. Per chunk the input halo (6 x 34
// per channel) is staged in LDS, read word by word with lanes along the row,
// since rows start on any word (two buffers, so one block barrier per chunk).
// Wave w owns the transform row xi = w (positions p = 4w + nu, nu = 0..3), and
// each of its lanes transforms exactly the patches whose V its MFMA B operand
// needs - channels lane / 32 + 2 e (e = 0..7) of tile lane % 32 - for that row
// only, so V never goes through LDS. The products are 32x32x16 bf16 MFMAs,
// whose one B operand is all 32 tiles: V is split in registers, the A operand,
// U_p[m][c], by the host (laid out lane by lane, read from memory straight into
// registers a position ahead). The output transform A^T . A runs in two halves:
// the column half (over nu) in registers, the row half (over xi, across the
// waves) after one exchange through LDS. A block with a non-finite sum (an
// infinite or NaN operand, one that bf16 parts cannot hold, or transforms that
// overflow) forms its outputs as direct sums of nine taps instead: the
// transforms would turn an infinity into inf - inf = NaN, and reach pixels that
// an output does not read.
//
// Bound by issue (the transforms and the split on the vector ALU, two waves a
// SIMD at 224 VGPRs) and its last round of blocks. 128 -> 128 channels at
// 225x319: 232 us as implicit GEMM on fp32 MFMAs, 126 here (110 of kernel
// time, 192 direct-equivalent TFLOP/s), error against 64 bits 6.1e-7 -> 2.9e-7.
// For the aligned widths the fp32 kernel of wino.h stays: with the same split
// they measured 37.4 us against its 36.2 (32 channels, 448x640), 34.7 against
// 34.8 (64, 224x320) and 41.3 against 37.4 (128, 112x160: 560 blocks over 512
// resident ones, where the fp32 form holds more blocks at once); a third block
// per CU would need 168 VGPRs and spills.
#pragma once

#include "common.h"

namespace wino_u {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int BM = 32;  // output channels per block
constexpr int CK = 16;  // input channels per chunk

// EP: -1 the generic fused epilogue, 16 a LeakyReLU only (the residual
// blocks' first conv; the same expression as the generic one).
template <bool FUSED, int EP = -1>
__device__ void body(const ConvArgs &a) {
    constexpr int NT = 32;               // tiles per block
    constexpr int TC = 16, TR = NT / TC; // tile columns and rows
    constexpr int OW = 2 * TC;           // output columns per block
    constexpr int HH = 2 * TR + 2;       // halo rows
    // halo LDS pitch: even, so a patch row is two aligned 64-bit reads, and
    // the two tile rows' 32 words on distinct banks (2 HP = 32 mod 64)
    constexpr int HP = 48;
    constexpr int MP = 36;  // M pitch: the 4-row steps of a half-wave's stores on distinct banks
    constexpr int NW = HH * (CK / 8);          // halo words per thread and chunk
    constexpr int ER = 256 / (CK * 2);         // halo rows its edge loads cover at once
    constexpr int NET = (HH + ER - 1) / ER;    // edge columns per thread and chunk
    constexpr int CS = HH * HP;                // channel pitch
    constexpr int HALO = CK * CS;
    constexpr int MS = 4 * 2 * BM * MP;
    constexpr int POOL = 2 * HALO > MS ? 2 * HALO : MS;
    static_assert(BM * NT / 256 * 4 * 256 <= POOL, "the direct sums");
    static_assert(CK == 16 && HP >= OW + 2 && HP % 2 == 0 && OW == 32, "eight rows of 32 words at a time");
    __shared__ __align__(16) float smem[POOL];
    __shared__ int bad[4];
    float *Ms = smem;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lt = lane & 31, lk = lane >> 5;
    const int tiles_x = (a.ow + OW - 1) / OW;
    int tile, mb;
    xcd_tile(tile, mb);
    const int oy0 = (tile / tiles_x) * (2 * TR), ox0 = (tile % tiles_x) * OW;
    const int m0 = mb * BM;
    // the bias of this thread's (output channel, tile) pairs of the
    // epilogue, fetched now so its latency hides behind the main loop
    constexpr int PAIRS = BM * NT / 256;
    float bsv[PAIRS];
#pragma unroll
    for (int q = 0; q < PAIRS; ++q) {
        const int m = m0 + (tid + q * 256) / NT;
        bsv[q] = a.bias && m < a.co ? a.bias[m] : 0.0f;
    }
    const int nchunk = (a.ci + CK - 1) / CK;
    // this block's transformed filters, [chunk][wave][nu][part][lane]
    const u32x4 *ublk = reinterpret_cast<const u32x4 *>(a.w) + ((int64_t)mb * nchunk) * (4 * 4 * 3 * 64);

    // The halo loads of this thread: column wk of channels wc and wc + 8, and
    // one edge column of channel ec in rows er0, er0 + ER, ... Addresses are
    // clamped into the image, and what lies outside it is multiplied by 0
    // instead of the operands' scale (an infinity read there is in the halo
    // itself, so the block takes the direct sums). The last chunk may hold
    // eight channels (c_in % 8 == 0): it reads them twice, the second time
    // against U's zeros.
    const int wc = tid >> 5, wk = tid & 31;
    const int ec = tid / 2 % CK, side = tid & 1, er0 = tid / (CK * 2);
    const uint32_t plane = (uint32_t)a.h * (uint32_t)a.wd;  // 16 planes < 2^32, checked by the host
    const uint32_t wd = (uint32_t)a.wd;
    const uint32_t woff = wc * plane + min(ox0 + wk, a.wd - 1);
    const int ecol = side ? ox0 + OW : ox0 - 1;
    float wsc[HH], esc[NET];
    uint32_t eoff[NET];
#pragma unroll
    for (int r = 0; r < HH; ++r)
        wsc[r] = (unsigned)(oy0 - 1 + r) < (unsigned)a.h && ox0 + wk < a.wd ? kSplitScale : 0.0f;
#pragma unroll
    for (int i = 0; i < NET; ++i) {
        const int iy = oy0 - 1 + er0 + ER * i;
        esc[i] = (unsigned)iy < (unsigned)a.h && (unsigned)ecol < (unsigned)a.wd ? kSplitScale : 0.0f;
        eoff[i] = (uint32_t)min(max(iy, 0), a.h - 1) * wd + min(max(ecol, 0), a.wd - 1);
    }
    const int wlds = wc * CS + 1 + wk, elds = ec * CS + er0 * HP + (side ? OW + 1 : 0);
    float qw[NW], er[NET];
    u32x4 ur[2][3];  // two positions' filters, one in use and one on its way
    auto fetch_halo = [&](int chunk) {
        const bool half = a.ci - chunk * CK < CK;
        const float *xc = a.x + (int64_t)chunk * CK * plane;
        const float *xw = xc + woff;
        const int64_t q1 = half ? 0 : 8 * (int64_t)plane;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int iy = min(max(oy0 - 1 + i % HH, 0), a.h - 1);
            qw[i] = xw[i / HH * q1 + (int64_t)iy * a.wd];
        }
        const uint32_t ep = (half ? ec & 7 : ec) * plane;
#pragma unroll
        for (int i = 0; i < NET; ++i) er[i] = xc[ep + eoff[i]];
    };
    auto stage_halo = [&](float *Hs) {
#pragma unroll
        for (int i = 0; i < NW; ++i) Hs[wlds + 8 * (i / HH) * CS + i % HH * HP] = qw[i] * wsc[i % HH];
#pragma unroll
        for (int i = 0; i < NET; ++i)
            if (er0 + ER * i < HH) Hs[elds + ER * i * HP] = er[i] * esc[i];
    };
    auto fetch_u = [&](int chunk, int nu) {
        const u32x4 *u = ublk + ((int64_t)(chunk * 4 + wave) * 4 + nu) * (3 * 64) + lane;
#pragma unroll
        for (int p = 0; p < 3; ++p) ur[nu & 1][p] = u[p * 64];
    };

    // This wave's row of B^T d: T = d[r0] + sgn d[r1] (d0 - d2, d1 + d2,
    // d2 - d1, d1 - d3 for xi = 0..3), of this lane's patches: channels
    // lk + 2 e of tile lt.
    const int r0 = wave == 0 ? 0 : wave == 3 ? 1 : wave == 1 ? 1 : 2;
    const int r1 = wave == 0 ? 2 : wave == 3 ? 3 : wave == 1 ? 2 : 1;
    const float sgn = wave == 1 ? 1.0f : -1.0f;
    const int pofs = lk * CS + (lt / TC) * 2 * HP + (lt % TC) * 2;

    f32x16 acc[4];

#pragma unroll
    for (int nu = 0; nu < 4; ++nu)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[nu][r] = 0.0f;
    // this wave's row of B^T d of this lane's patches
    auto rows = [&](const float *Hs, float (&t)[8][4]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float *h = Hs + pofs + 2 * e * CS;
            const float2 p0 = *reinterpret_cast<const float2 *>(h + r0 * HP);
            const float2 p1 = *reinterpret_cast<const float2 *>(h + r0 * HP + 2);
            const float2 q0 = *reinterpret_cast<const float2 *>(h + r1 * HP);
            const float2 q1 = *reinterpret_cast<const float2 *>(h + r1 * HP + 2);
            t[e][0] = __builtin_fmaf(sgn, q0.x, p0.x);
            t[e][1] = __builtin_fmaf(sgn, q0.y, p0.y);
            t[e][2] = __builtin_fmaf(sgn, q1.x, p1.x);
            t[e][3] = __builtin_fmaf(sgn, q1.y, p1.y);
            // four channels' patches in flight, not all (registers)
            if (e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
    };
    // ... and V's position nu
    auto col = [](const float (&t)[4], int nu) {
        return nu == 0 ? t[0] - t[2] : nu == 1 ? t[1] + t[2] : nu == 2 ? t[2] - t[1] : t[1] - t[3];
    };

    fetch_halo(0);
    fetch_u(0, 0);
    for (int chunk = 0; chunk < nchunk; ++chunk) {
        float *Hs = smem + (chunk & 1) * HALO;
        // (every wave finished reading this buffer two chunks ago, before
        // the previous chunk's barrier)
        stage_halo(Hs);
        __syncthreads();
        if (chunk + 1 < nchunk) fetch_halo(chunk + 1);
        float t[8][4];
        rows(Hs, t);
#pragma unroll
        for (int nu = 0; nu < 4; ++nu) {
            if (nu < 3)
                fetch_u(chunk, nu + 1);
            else if (chunk + 1 < nchunk)
                fetch_u(chunk + 1, 0);
            u32x4 vp[3];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t h, m, l;
                split2(col(t[2 * e], nu), col(t[2 * e + 1], nu), h, m, l);
                vp[0][e] = h;
                vp[1][e] = m;
                vp[2][e] = l;
            }
            // the six products, the smallest first
            constexpr int PU[6] = {2, 1, 0, 1, 0, 0}, PV[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
            for (int k = 0; k < 6; ++k)
                acc[nu] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ur[nu & 1][PU[k]]),
                                                                  __builtin_bit_cast(bf16x8, vp[PV[k]]), acc[nu], 0, 0, 0);
        }
    }
    // (2^8 below the largest float, so that the output transform stays finite)
    float top = 0.0f;
#pragma unroll
    for (int nu = 0; nu < 4; ++nu)
#pragma unroll
        for (int r = 0; r < 16; ++r) top = __builtin_elementwise_maximum(top, __builtin_fabsf(acc[nu][r]));
    const bool over = __builtin_amdgcn_ballot_w64(!(top < 0x1p120f)) != 0;
    if (lane == 0) bad[wave] = over;
    __syncthreads();
    const bool direct = (bad[0] | bad[1] | bad[2] | bad[3]) != 0;

    // (.) A over nu in registers: u[dx] for this wave's transform row xi;
    // then the rows of all four waves meet in LDS as Ms[xi][dx][m][t].
    if (!direct) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float a0 = acc[0][r], a1 = acc[1][r], a2 = acc[2][r], a3 = acc[3][r];
            const int m = r / 4 * 8 + 4 * lk + r % 4;
            Ms[((wave * 2 + 0) * BM + m) * MP + lt] = a0 + a1 + a2;
            Ms[((wave * 2 + 1) * BM + m) * MP + lt] = a1 - a2 - a3;
        }
        __syncthreads();
    } else {
        // the 2x2 outputs of this thread's (output channel, tile) pairs, each
        // its own sum in fp32 over the image and the untransformed filters,
        // left in LDS for itself (tap by tap, channels innermost)
#pragma nounroll
        for (int q = 0; q < PAIRS; ++q) {
            const int e = tid + q * 256, m = m0 + e / NT, t = e % NT;
#pragma nounroll
            for (int d = 0; d < 4; ++d) {
                const int oy = oy0 + 2 * (t / TC) + d / 2, ox = ox0 + 2 * (t % TC) + d % 2;
                float s = 0.0f;
                if (m < a.co && oy < a.oh && ox < a.ow) {
#pragma nounroll
                    for (int tap = 0; tap < 9; ++tap) {
                        const int iy = oy + tap / 3 - 1, ix = ox + tap % 3 - 1;
                        if (iy < 0 || iy >= a.h || ix < 0 || ix >= a.wd) continue;
                        const float *xi = a.x + (int64_t)iy * a.wd + ix;
                        const float *wi = a.wo + (int64_t)m * a.ci * 9 + tap;
#pragma nounroll
                        for (int c = 0; c < a.ci; ++c) s = __builtin_fmaf(wi[c * 9], xi[(int64_t)c * plane], s);
                    }
                }
                Ms[(q * 4 + d) * 256 + tid] = s;
            }
        }
    }
    // A^T . over xi, bias, epilogue, stores: thread -> (m, tile), tiles fastest
    // rows and columns may end inside the block
    const int64_t oplane = (int64_t)a.oh * a.ow;
    const bool vec = a.cvec != 0;
    const float us = direct ? 1.0f : kUnsplit;
#pragma unroll
    for (int q = 0; q < PAIRS; ++q) {
        const int e = tid + q * 256, m = e / NT, t = e % NT;
        if (m0 + m >= a.co) continue;
        float y[2][2];
        if (!direct) {
            float u[4][2];
#pragma unroll
            for (int xi = 0; xi < 4; ++xi)
#pragma unroll
                for (int dx = 0; dx < 2; ++dx) u[xi][dx] = Ms[((xi * 2 + dx) * BM + m) * MP + t];
#pragma unroll
            for (int dx = 0; dx < 2; ++dx) {
                y[0][dx] = u[0][dx] + u[1][dx] + u[2][dx];
                y[1][dx] = u[1][dx] - u[2][dx] - u[3][dx];
            }
        } else {
#pragma unroll
            for (int d = 0; d < 4; ++d) y[d / 2][d % 2] = Ms[(q * 4 + d) * 256 + tid];
        }
        const int oy = oy0 + 2 * (t / TC), ox = ox0 + 2 * (t % TC);
        if (ox >= a.ow) continue;
        const int64_t ib = (int64_t)(m0 + m) * oplane + ox;
        const float bb = bsv[q];
#pragma unroll
        for (int dy = 0; dy < 2; ++dy) {
            if (oy + dy >= a.oh) continue;
            const int64_t idx = ib + (int64_t)(oy + dy) * a.ow;
            float v0 = __builtin_fmaf(y[dy][0], us, bb), v1 = __builtin_fmaf(y[dy][1], us, bb);
            if (EP == 16) {
                v0 = v0 >= 0.0f ? v0 : a.e.slope * v0;
                v1 = v1 >= 0.0f ? v1 : a.e.slope * v1;
            }
            if (vec) {
                if (FUSED && EP < 0) epilogue2(a.e, v0, v1, idx);
                *reinterpret_cast<float2 *>(a.y + idx) = make_float2(v0, v1);
            } else {
                const bool two = ox + 1 < a.ow;
                if (FUSED && EP < 0) {
                    v0 = epilogue(a.e, v0, idx);
                    if (two) v1 = epilogue(a.e, v1, idx + 1);
                }
                a.y[idx] = v0;
                if (two) a.y[idx + 1] = v1;
            }
        }
    }
}

}  // namespace wino_u

// mx_wino3_t16_u[_f[_e16]]: 3x3 pad 1, any width and alignment, 32 output
// channels x 4 x 32 pixels per block; cvec (even widths): the output and every
// epilogue operand 8-byte aligned (paired loads and stores). _f applies the
// fused epilogue, _f_e16 one that is a LeakyReLU alone.
extern "C" __global__ __launch_bounds__(256, 2) void mx_wino3_t16_u(ConvArgs a) { wino_u::body<false>(a); }
extern "C" __global__ __launch_bounds__(256, 2) void mx_wino3_t16_u_f(ConvArgs a) { wino_u::body<true>(a); }
extern "C" __global__ __launch_bounds__(256, 2) void mx_wino3_t16_u_f_e16(ConvArgs a) { wino_u::body<true, 16>(a); }
