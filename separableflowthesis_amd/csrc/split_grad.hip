// Feature gradients on the 16-bit matrix units, at fp32 accuracy.
//
//   d_f1[p,:] = sum_q G[p,q] f2[q,:]      d_f2[q,:] = sum_p G[p,q] f1[p,:]      G = dL/dS, formed on the way
//
// the same sums as df1_kernel and df2_tiled_kernel in sepcorr.hip, for G of the attention compression, alone or with the
// max/average terms.  C <= 256.
//
// Halves.  Both operands of a product are written as h + l, h = fp16(x), l = fp16(x - h), and multiplied as h h + h l + l h
// with v_mfma_f32_32x32x16_f16, accumulated in fp32.  The contraction runs over pixels, so a scale may depend on anything
// that is not summed over, or be split between the two factors:
//   features   a power of two per image and channel, largest value into [2^14, 2^15);
//   G, d_f1    a power of two per pixel p from a bound of |G[p,:]|;
//   G, d_f2    a power of two per position q of image 2 and FLUSH steps of pixels, from bounds of |G[p,q]| over 16 pixels each
//              (grad_prepare_kernel): a row of d_f2 that all attention avoids, or that only pixels of small gradients reach,
//              has its own.  (Summed over p with one factor per pixel, rows 2^-17, 2^-23, 2^-29 of the largest were off by
//              2e-6, 2e-4, 8e-3.)
// 22 bits are held down to 2^-17 of the largest value a scale stands for, 2^-39 of that below.  Operands without such a form
// (inf, NaN, more than one feature in 2048 below 2^-17 of its channel's largest) are found on the way, and the contractions
// then run in fp32 from the inputs instead (contract_fp32).
// Relative error against 64 bits, d_f1 / d_f2, fp32 kernels -> halves: B=2, 55x128, K=4 2.2e-7 / 6.9e-7 -> 1.7e-7 / 3.0e-7;
// B=4, 48x64 2.2e-7 / 4.5e-7 -> 1.5e-7 / 2.5e-7; 136x240 2.4e-7 / 9.0e-7 -> 1.8e-7 / 3.3e-7; B=2, 47x61, C=100, K=2 2.1e-7 / 3.5e-7 ->
// 1.3e-7 / 2.0e-7.  Of single rows at B=2, 40x56, with attention that is flat, peaked or avoids half of image 2 by up to 40 in
// the logits and gradients of one size or of 2^-40..1, at the most 2.8e-7 / 4.4e-7 -> 1.7e-7 / 3.4e-7.
//
// Work split.  A workgroup of eight waves, one per compute unit, owns 128 pixels x all channels of d_f1, or 8 rows x 32
// columns x all channels of d_f2 (64 or 128 accumulator registers a lane), and takes a step at a time: 32 columns of a row of
// fmap2, or 16 pixels of image 1, whose halves are DMA'd into LDS two steps ahead.  G of the next step is formed once per
// workgroup, 8 elements a lane, its halves put into LDS in operand order; d_f1 keeps the v-indexed weights of its columns in
// registers over the rows, d_f2 has them in LDS and transposes G with ds_read_b64_tr_b16.  The steps of all tiles are dealt
// out evenly; pieces of tiles are put together by grad_finish_kernel in the order of their steps.
//
// Measured at B=2, 55x128, C=256, K=4 (fp32 kernels, then here): d_f1 507 us and 14 before it, 195 + 16; d_f2 517 + 14, 220 + 19;
// the operands 54 on top.  Backward call 1.28 -> 0.73 ms, 136x240 20.9 -> 7.2 ms.  The matrix instructions alone take 123 us
// each at the 1.24 PFLOP/s that a large fp16 product reaches here.  What the rest is, in d_f1 (variants with a part left out,
// results then wrong): without forming G 148 us, without the DMA 182 of then 209; in d_f2 the factors by positions are 18 of it,
// 6 to find them, 3 to take them back, the rest beside forming G.
#include "split_grad.h"

#include <math.h>

#include <algorithm>

#include "sepcorr.h"
#include "sepcorr_internal.h"
#include "split_grad_deal.h"

#ifndef GRAD_PART
#define GRAD_PART (-1)
#endif
#define GRAD_IN_PART(n) (GRAD_PART < 0 || GRAD_PART == (n))

namespace {
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr int TPX = 128;      // pixels of a d_f1 tile
constexpr int ROWS = 8;       // rows of fmap2 of a d_f2 tile
constexpr unsigned OOB = 0x80000000u;   // a byte offset above every buffer size used here: reads as zero
// One feature in so many may be below 2^-17 of its channel's largest.  (Of normal ones one in 37 000 is; beside a single one
// of 2^17 times the rest a whole channel, one in 256 at the most.)
constexpr unsigned SMALL_SHARE = 2048;

constexpr int SLABS = 16;     // blocks per image and tensor that look for the largest channels

// Fields of the v-indexed weights of a pixel and column: a_u[k], g_cv[k] (, g_v[max], g_v[avg], argmax_v), as they are.
__host__ __device__ constexpr int vfields(bool both, int kc) { return 2 * kc + (both ? 3 : 0); }
// Of the u-indexed ones: g_cu[k], a_v[k] (, g_u[max] + g_u[avg] / W2, g_u[avg] / W2, argmax_u).
__host__ __device__ constexpr int ufields(bool both, int kc) { return (2 * kc + (both ? 3 : 0) + 3) & ~3; }
// Bounds of a block of 16 pixels, by columns and by rows (grad_prepare_kernel).
__host__ __device__ constexpr int nbounds(bool both) { return both ? 3 : 2; }

// floats between the u-indexed rows of a pixel in LDS (16 bytes aligned, banks apart)
__host__ __device__ __forceinline__ int u_row(int H2) { return (H2 + ROWS - 1) / ROWS * ROWS + 4; }
__host__ __device__ __forceinline__ size_t prepare_lds(bool both, int kc, int H2) { return (size_t)16 * (2 * kc + (both ? 3 : 0)) * u_row(H2) * sizeof(float); }

__device__ __forceinline__ int vmap(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }
__device__ __forceinline__ unsigned magnitude(float x) { return __float_as_uint(x) & 0x7fffffffu; }
__device__ __forceinline__ int xcd_contiguous(int bid, int n) {
    const int c = bid & 7, slot = bid >> 3, q = n >> 3, r = n & 7;
    return c * q + (c < r ? c : r) + slot;
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *p, unsigned bytes) {
    const uint64_t addr = reinterpret_cast<uint64_t>(p);
    const uint64_t lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)addr);
    const uint64_t hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(addr >> 32));
    const int n = __builtin_amdgcn_readfirstlane((int)bytes);
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>((hi << 32) | lo), 0, n, 0x00020000);
}
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rs, void *lds, unsigned lane_off, unsigned off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)lds, 16, lane_off, off, 0, 0);
}
// largest magnitude -> the power of two that brings it into [2^14, 2^15), at most 2^126 (below 2^-112 it stays smaller: a bit
// of the halves is then one of the smallest numbers there are)
__device__ __forceinline__ int scale_exponent(float m) { return 141 - (int)max(magnitude(m) >> 23, 15u); }
__device__ __forceinline__ float power(int e) { return __uint_as_float((unsigned)(e + 127) << 23); }
__device__ __forceinline__ int exponent_of(float p) { return (int)(__float_as_uint(p) >> 23) - 127; }
// the largest of 16 lanes in a row, for all of them
__device__ __forceinline__ unsigned max16(unsigned x) {
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xf, 0xf, true));   // (row_ror)
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x124, 0xf, 0xf, true));
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x122, 0xf, 0xf, true));
    return max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x121, 0xf, 0xf, true));
}
__device__ __forceinline__ float max16(float x) { return __uint_as_float(max16(__float_as_uint(x))); }   // (none negative)
// x, y -> their high halves in one register, their low halves in another: x - h is exact and rounded once
__device__ __forceinline__ void split2(float x, float y, unsigned &h, unsigned &l) {
    asm("v_cvt_pk_f16_f32 %0, %2, %3\n\t"
        "v_fma_mixlo_f16 %1, %0, -1.0, %2 op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixhi_f16 %1, %0, -1.0, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "=&v"(h), "=&v"(l) : "v"(x), "v"(y));
}
// the same of x s, y t, s and t powers of two
__device__ __forceinline__ void split2(float x, float y, float s, float t, unsigned &h, unsigned &l) {
    asm("v_fma_mixlo_f16 %0, %2, %4, 0\n\t"
        "v_fma_mixhi_f16 %0, %3, %5, 0\n\t"
        "v_fma_mixlo_f16 %1, %2, %4, -%0 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %1, %3, %5, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
        : "=&v"(h), "=&v"(l) : "v"(x), "v"(y), "v"(s), "v"(t));
}
__device__ __forceinline__ void phase_end() { asm volatile("s_barrier" ::: "memory"); }
__device__ __forceinline__ v16f mfma(v8h a, v8h b, v16f c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }

__device__ __forceinline__ bool unsuitable(const GradArgs &a) {
    return a.count[2] != 0 || a.count[0] > (unsigned)((size_t)a.B * a.N1 * a.C / SMALL_SHARE) ||
           a.count[1] > (unsigned)((size_t)a.B * a.H2 * a.W2 * a.C / SMALL_SHARE);
}

// Four consecutive columns from v on of a row of W2, zeros beyond it.
__device__ __forceinline__ v4f columns4(const float *row, int v, int W2, bool ok) {
    v4f y = {0.f, 0.f, 0.f, 0.f};
    if (ok && v + 4 <= W2) {
        __builtin_memcpy(&y, row + v, 16);
    } else if (ok) {
#pragma unroll
        for (int e = 0; e < 3; ++e)
            if (v + e < W2) y[e] = row[v + e];
    }
    return y;
}
// The v-indexed weights, field f, of pixel bp.
template <int KC>
__device__ __forceinline__ const float *vrow(const GradArgs &a, int f, size_t bp) {
    if (f < KC) return a.a_u + (bp * a.KT + a.k0 + f) * a.W2;
    if (f < 2 * KC) return a.g_cv + (bp * a.KT + a.k0 + f - KC) * a.W2;
    if (f < 2 * KC + 2) return a.g_v + (2 * bp + f - 2 * KC) * a.W2;
    return reinterpret_cast<const float *>(a.am_v) + bp * a.W2;
}

// What both contractions need beforehand, bound by its traffic: 82 MB read and 31 written in 37 us at B=2, 55x128, K=4 (32 without
// the bounds; 44 with the v-indexed rows read twice for them; 14 more with the channels' blocks behind the others and one channel a
// lane, 59 more with atomics for the channels' maxima).
// Blocks [0, 2 B SLABS): the largest magnitude of every channel of a slab of f1 or f2.
// The blocks behind them: the weights of 16 pixels, and what bounds |G| there,
//   |G[p,u,v]| <= sum_k |a_u[k,v] g_cu[k,u]| + sum_k |a_v[k,u] g_cv[k,v]| (+ the max/average gradients):
//   the pixel's factor (d_f1) brings beta = sum_k max|a_u| max|g_cu| + max|a_v| max|g_cv| (+ ..) into [2^14, 2^15);
//   the factors of d_f2 go by positions of image 2 (split_d2_kernel) and need, of the 16 pixels together, for every column
//     X = max_p sum_k |a_u[k,v]| max_u |g_cu[k]|,  X' = max_p sum_k |g_cv[k,v]| max_u |a_v[k]|  (, |g_v[max]| + |g_v[avg]| / H2),
//   for every row Y and Y' likewise (, |g_u[max]| + |g_u[avg]| / W2): |G| <= min(X, Y) + min(X', Y') (+ both others).
template <bool BOTH, int KC>
__global__ void __launch_bounds__(256) grad_prepare_kernel(const GradArgs a) {
    constexpr int NF = vfields(BOTH, KC), NU = ufields(BOTH, KC), NR = 2 * KC + (BOTH ? 3 : 0), NX = nbounds(BOTH);
    constexpr int NM = 2 * KC + (BOTH ? 2 : 0);
    __shared__ unsigned smv[NM][16], smu[NM][16];   // [field][pixel]: the largest magnitude of a row
    extern __shared__ float sh[];   // [pixel][row of u-indexed weights][urow]
    const int urow = u_row(a.H2);
    const int ntile = a.N1p / 16;
    const int N1 = a.N1, H2 = a.H2, W2 = a.W2;
    const int nslab = 2 * a.B * SLABS;
    if ((int)blockIdx.x < nslab) {   // (first: each takes longer than a block of weights)
        const int slab = blockIdx.x % SLABS, t = blockIdx.x / SLABS, cp = 32 * a.ncb;   // t: tensor * B + image
        const bool second = t >= a.B, vec = (a.C & 3) == 0;
        const int n = second ? H2 * W2 : N1, per = vec ? 4 : 1, lanes = cp / per, step = 256 / lanes;
        const int c = per * (threadIdx.x & (lanes - 1)), pl = threadIdx.x / lanes;
        const float *src = (second ? a.f2 : a.f1) + (size_t)(second ? t - a.B : t) * n * a.C;
        const int p0 = (int)((long)slab * n / SLABS), p1 = (int)((long)(slab + 1) * n / SLABS);
        unsigned m[4] = {0, 0, 0, 0};
        if (vec && c < a.C) {
#pragma unroll 8
            for (int p = p0 + pl; p < p1; p += step) {
                v4f x;
                __builtin_memcpy(&x, src + (size_t)p * a.C + c, 16);
#pragma unroll
                for (int e = 0; e < 4; ++e) m[e] = max(m[e], magnitude(x[e]));
            }
        } else if (c < a.C) {
#pragma unroll 8
            for (int p = p0 + pl; p < p1; p += step) m[0] = max(m[0], magnitude(src[(size_t)p * a.C + c]));
        }
        unsigned *red = reinterpret_cast<unsigned *>(sh);   // [step][cp]
        for (int e = 0; e < per; ++e) red[pl * cp + c + e] = m[e];
        __syncthreads();
        if ((int)threadIdx.x < cp) {
            unsigned top = 0;
            for (int i = 0; i < step; ++i) top = max(top, red[i * cp + threadIdx.x]);
            a.pmax[((size_t)t * SLABS + slab) * 256 + threadIdx.x] = top;
        }
        return;
    }
    const int blk = blockIdx.x - nslab;
    const int b = blk / ntile, t16 = blk - b * ntile;
    const float inv_w2 = 1.f / (float)W2, inv_h2 = 1.f / (float)H2;
    if (blk == 0 && threadIdx.x < 3) a.count[threadIdx.x] = 0;
    if ((int)threadIdx.x < NM * 16) smv[threadIdx.x / 16][threadIdx.x % 16] = 0;
    {   // u-indexed rows: their largest magnitudes; they stay in LDS
        const int i = threadIdx.x >> 4, j = threadIdx.x & 15, pix = 16 * t16 + i;
        const bool ok = pix < N1;
        const size_t bp = (size_t)b * N1 + (ok ? pix : N1 - 1);
        const float *ur[NR];
#pragma unroll
        for (int f = 0; f < NR; ++f)
            ur[f] = f < KC ? a.g_cu + (bp * a.KT + a.k0 + f) * H2 : f < 2 * KC ? a.a_v + (bp * a.KT + a.k0 + f - KC) * H2
                  : f < 2 * KC + 2 ? a.g_u + (2 * bp + f - 2 * KC) * H2 : reinterpret_cast<const float *>(a.am_u) + bp * H2;
        unsigned mu[NM] = {};
        for (int x = 4 * j; x < a.H2p; x += 64) {
            v4f z[NR];
#pragma unroll
            for (int f = 0; f < NR; ++f) z[f] = columns4(ur[f], x, H2, x < H2 && ok);
#pragma unroll
            for (int f = 0; f < NR; ++f) *reinterpret_cast<v4f *>(sh + (i * NR + f) * urow + x) = z[f];
#pragma unroll
            for (int f = 0; f < NM; ++f)
#pragma unroll
                for (int e = 0; e < 4; ++e) mu[f] = max(mu[f], magnitude(z[f][e]));
        }
#pragma unroll
        for (int f = 0; f < NM; ++f) {
            mu[f] = max16(mu[f]);
            if (j == f) smu[f][i] = mu[f];
        }
    }
    __syncthreads();
    const int i = threadIdx.x & 15, pix = 16 * t16 + i;
    const bool ok = pix < N1;
    {   // v-indexed rows: 64 lanes have the four columns each of 16 pixels
        const size_t bp = (size_t)b * N1 + (ok ? pix : N1 - 1);
        unsigned mv[NM] = {};
        float wu[2 * KC];
#pragma unroll
        for (int f = 0; f < 2 * KC; ++f) wu[f] = __uint_as_float(smu[f][i]);
        for (int vg = threadIdx.x >> 4; vg < 8 * a.nvc; vg += 16) {
            v4f y[NF], x[NX] = {};
            if (a.direct) {   // (argmax_v is only copied)
#pragma unroll
                for (int f = 0; f < NM; ++f) y[f] = columns4(vrow<KC>(a, f, bp), 4 * vg, W2, ok);
            } else {
#pragma unroll
                for (int f = 0; f < NF; ++f) y[f] = columns4(vrow<KC>(a, f, bp), 4 * vg, W2, ok);
                float *dst = a.pv + (((size_t)b * a.nvc + (vg >> 3)) * ntile + t16) * NF * 512 + ((vg & 7) * 16 + i) * 4;   // (1 KB a wave)
#pragma unroll
                for (int f = 0; f < NF; ++f) *reinterpret_cast<v4f *>(dst + f * 512) = y[f];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma unroll
                for (int f = 0; f < NM; ++f) mv[f] = max(mv[f], magnitude(y[f][e]));
#pragma unroll
                for (int f = 0; f < 2 * KC; ++f) x[f / KC][e] = fmaf(fabsf(y[f][e]), wu[f], x[f / KC][e]);
                if constexpr (BOTH) x[NX - 1][e] = fmaf(fabsf(y[2 * KC + 1][e]), inv_h2, fabsf(y[2 * KC][e]));
            }
#pragma unroll
            for (int n = 0; n < NX; ++n) {
#pragma unroll
                for (int e = 0; e < 4; ++e) x[n][e] = max16(x[n][e]);
                if (i == n) *reinterpret_cast<v4f *>(a.bound_v + (((size_t)b * a.nvc + (vg >> 3)) * ntile + t16) * NX * 32 + n * 32 + 4 * (vg & 7)) = x[n];
            }
        }
#pragma unroll
        for (int f = 0; f < NM; ++f) atomicMax(&smv[f][i], mv[f]);
    }
    __syncthreads();
    float wv[2 * KC];
#pragma unroll
    for (int f = 0; f < 2 * KC; ++f) wv[f] = __uint_as_float(smv[f][i]);
    if (threadIdx.x < 64) {
        float beta = 0.f;
#pragma unroll
        for (int f = 0; f < 2 * KC; ++f) beta += wv[f] * __uint_as_float(smu[f][i]);
        if constexpr (BOTH) {
            beta += __uint_as_float(smu[2 * KC][i]) + __uint_as_float(smu[2 * KC + 1][i]) * inv_w2;
            beta += __uint_as_float(smv[2 * KC][i]) + __uint_as_float(smv[2 * KC + 1][i]) * inv_h2;
        }
        const bool good = beta < 0x1p126f;   // (not where an operand is inf or NaN)
        if (threadIdx.x < 16) a.pscale[(size_t)b * a.N1p + pix] = good ? power(scale_exponent(beta)) : 1.f;
        const unsigned long long bad = __ballot(ok && !good);
        if (threadIdx.x == 0) a.block_bad[blk] = bad != 0;
    }
    for (int u = threadIdx.x >> 4; u < a.H2p; u += 16) {
        const float *r = sh + i * NR * urow + u;
        float y[NX] = {};
#pragma unroll
        for (int f = 0; f < 2 * KC; ++f) y[f / KC] = fmaf(fabsf(r[f * urow]), wv[f], y[f / KC]);
        if constexpr (BOTH) y[NX - 1] = fmaf(fabsf(r[(2 * KC + 1) * urow]), inv_w2, fabsf(r[2 * KC * urow]));
#pragma unroll
        for (int n = 0; n < NX; ++n) {
            y[n] = max16(y[n]);
            if (i == n) a.bound_u[((size_t)b * ntile + t16) * NX * a.H2p + n * a.H2p + u] = y[n];
        }
    }
    // u-indexed weights: a pixel's fields of a row together
    for (int n = threadIdx.x; n < a.H2p * 16 * (NU / 4); n += 256) {
        const int f4 = 4 * (n % (NU / 4)), pi = n / (NU / 4) % 16, u = n / (16 * (NU / 4));
        const float *r = sh + pi * NR * urow + u;
        v4f y;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int f = f4 + e;
            if (f < 2 * KC) y[e] = r[f * urow];
            else if (!BOTH || f > 2 * KC + 2) y[e] = 0.f;
            else if (f == 2 * KC) y[e] = r[f * urow] + r[(f + 1) * urow] * inv_w2;
            else y[e] = f == 2 * KC + 1 ? r[f * urow] * inv_w2 : r[f * urow];
        }
        *reinterpret_cast<v4f *>(a.pu + (((size_t)b * a.H2p + u) * a.N1p + 16 * t16 + pi) * NU + f4) = y;
    }
}

#if GRAD_IN_PART(0)
// Halves of 32 pixels of a row of fmap2, or of 16 pixels of image 1, in operand order: one KB per (16 pixels, 32 channels,
// half) holding the 16 bytes of each lane in lane order (lane 32 g + i: channel i, pixels 8 g + 0..7).  A channel is scaled
// by a power of two that brings the largest of the image into [2^14, 2^15).
template <int NCB>
__global__ void __launch_bounds__(256) grad_split_kernel(const GradArgs a) {
    constexpr int CP = 32 * NCB;
    const bool second = (int)blockIdx.x < a.B * a.nvc * a.H2;
    int b, n, p0;
    const float *src;
    char *dst;
    bool leads;   // the block that writes down the scales of its image
    bool bad = false;
    if (second) {
        const int u = blockIdx.x % a.H2, bc = blockIdx.x / a.H2, vc = bc % a.nvc;
        b = bc / a.nvc;
        n = a.W2;
        p0 = 32 * vc;
        leads = u == 0 && vc == 0;
        src = a.f2 + ((size_t)b * a.H2 + u) * a.W2 * a.C;
        dst = a.f2h + (size_t)blockIdx.x * NCB * 4096;
    } else {
        const int blk = blockIdx.x - a.B * a.nvc * a.H2, ntile = a.N1p / 16;
        b = blk / a.npx;
        n = a.N1;
        p0 = 16 * (blk - b * a.npx);
        leads = p0 == 0;
        src = a.f1 + (size_t)b * a.N1 * a.C;
        dst = a.f1h + (size_t)blk * NCB * 2048;
        if (leads)
            for (int i = threadIdx.x; i < ntile; i += 256) bad |= a.block_bad[b * ntile + i] != 0;
    }
    if (blockIdx.x == 0) {   // (from where they are: an assignment would move them to the stack)
        const unsigned *args = (const unsigned *)__builtin_amdgcn_kernarg_segment_ptr();
        for (int i = threadIdx.x; i < (int)(sizeof(GradArgs) / 4); i += 256) reinterpret_cast<unsigned *>(a.self)[i] = args[i];
    }
    const int c = threadIdx.x & (CP - 1);
    unsigned top = 0;
    {
        const unsigned *pm = a.pmax + (size_t)(second ? a.B + b : b) * SLABS * 256 + c;
#pragma unroll
        for (int i = 0; i < SLABS; ++i) top = max(top, pm[i * 256]);
    }
    bad |= top >= 0x7f800000u;
    const int fe = scale_exponent(__uint_as_float(top));
    float fwd = power(fe);
    if (leads && (int)threadIdx.x < CP) a.cback[((second ? a.B : 0) + b) * 256 + c] = -fe;
    if (second ? (blockIdx.x % a.H2) & 1 : (p0 / 16 / FLUSH) & 1) fwd = -fwd;   // (see block_sign)
    const unsigned least = top > (17u << 23) ? (top & 0x7f800000u) - (17u << 23) : 0;
    unsigned small = 0;
    for (int i = threadIdx.x; i < (second ? 4 : 2) * CP; i += 256) {
        const int g = i / CP;
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int p = p0 + 8 * g + e;
            x[e] = c < a.C && p < n ? src[(size_t)p * a.C + c] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            small += magnitude(x[e]) - 1u < least - 1u && least > 0;
            x[e] *= fwd;
        }
        v4u h, l;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            unsigned hh, ll;
            split2(x[2 * e], x[2 * e + 1], hh, ll);
            h[e] = hh;
            l[e] = ll;
        }
        char *d = dst + (((g >> 1) * NCB + (c >> 5)) * 2) * 1024 + (32 * (g & 1) + (c & 31)) * 16;
        *reinterpret_cast<v4u *>(d) = h;
        *reinterpret_cast<v4u *>(d + 1024) = l;
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) small += (unsigned)__shfl_xor((int)small, d);
    if ((threadIdx.x & 63) == 0 && small) atomicAdd(a.count + (second ? 1 : 0), small);
    if (bad) a.count[2] = 1;
}
#endif

// Finished 32 x 32 block of d_f1 (rows: pixels of image b) or d_f2 (rows: columns of row u of fmap2), accumulator layout.
// (d_f1 may still carry the factors of its channel and pixels: SCALED)
template <bool FIRST, bool SCALED>
__device__ __forceinline__ void store_block(const GradArgs &a, int b, int u, int p0, int c0, const float (&x)[16]) {
    const int lane = threadIdx.x & 63, c = c0 + (lane & 31), h = lane >> 5;
    if (c >= a.C) return;
    const int ce = SCALED ? a.cback[(a.B + b) * 256 + c] : 0;
    const int n = FIRST ? a.N1 : a.W2, add = FIRST ? a.add1 : a.add2;
    float *dst = (FIRST ? a.d1 + (size_t)b * a.N1 * a.C : a.d2 + ((size_t)b * a.H2 + u) * a.W2 * a.C) + c;
    float old[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int p = p0 + vmap(r, h);
        old[r] = add && p < n ? dst[(size_t)p * a.C] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int p = p0 + vmap(r, h);
        float y = x[r];
        if constexpr (SCALED) y = ldexpf(y, ce - exponent_of(a.pscale[(size_t)b * a.N1p + p]));
        if (p < n) dst[(size_t)p * a.C] = add ? old[r] + y : y;
    }
}

// Adds up what the pieces of a tile left in their slots, in the order of their steps.  One wave per 32 x 32 block.
template <bool FIRST, bool BOTH, int KC>
__global__ void __launch_bounds__(256) grad_finish_kernel(const GradArgs a) {
    const int ncb = a.ncb, per = (FIRST ? 4 : ROWS) * ncb, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int unit = blockIdx.x * 4 + wave, tile = unit / per, sub = unit - tile * per, cb = sub % ncb, row = sub / ncb;
    const int nug = a.H2p / ROWS, npt = a.N1p / TPX;
    const int tiles = FIRST ? a.B * npt : a.B * nug * a.nvc, spt = FIRST ? a.nvc * a.H2 : a.npx, G = FIRST ? a.G1 : a.G2;
    if (tile >= tiles) return;
    const long T = (long)tiles * spt, t0 = (long)tile * spt;
    int w0, w1;
    pieces_of(t0, t0 + spt, G, T, w0, w1);
    if (w0 == w1) return;   // (its workgroup has written it)
    const int ug = tile % nug, bv = tile / nug, u = ROWS * ug + row;   // (d_f2)
    if (!FIRST && u >= a.H2) return;
    const size_t slot = (size_t)per * 1024;
    // four pieces in flight, summed before they join the rest: a short tile in hundreds of pieces makes no long chain
    v4f x[4] = {};
    for (int wb = w0; wb <= w1; wb += 4) {
        v4f y[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int w = min(wb + i, w1);
            const v4f *src = reinterpret_cast<const v4f *>(a.slots + slot_of(w, tile, first_step(w, G, T) > t0, tiles, G) * slot + sub * 1024) + lane;
#pragma unroll
            for (int q = 0; q < 4; ++q) y[i][q] = src[q * 64];
        }
#pragma unroll
        for (int i = 1; i < 4; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) y[i][q] = wb + i <= w1 ? y[i][q] : v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] += (y[0][q] + y[1][q]) + (y[2][q] + y[3][q]);
    }
    float z[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) z[r] = x[r >> 2][r & 3];
    const bool scaled = FIRST && !unsuitable(a);
    if (scaled) store_block<true, true>(a, tile / npt, 0, TPX * (tile % npt) + 32 * row, 32 * cb, z);
    else if (FIRST) store_block<true, false>(a, tile / npt, 0, TPX * (tile % npt) + 32 * row, 32 * cb, z);
    else store_block<false, false>(a, bv / a.nvc, u, 32 * (bv % a.nvc), 32 * cb, z);
}

// The 16-bit matrix instructions round their sums down, not to nearest: with every product of one sign convention the
// mean error of d_f1 at 136x240 is -0.72 of its root mean square.  Odd rows of fmap2, and every other FLUSH pixel tiles of
// image 1, have their sign turned in the halves, and their sums are subtracted: what is rounded down there raises the
// result (d_f1 at 136x240, error against 64 bits: 2.66e-7 as products of one sign).
__device__ __forceinline__ float block_sign(int odd) { return odd & 1 ? -1.f : 1.f; }

// A piece's sums of a lane's block: what earlier flushes left of it in its slot (none if `first`), and x.
__device__ __forceinline__ void sums_of_piece(const v4f *slot, bool first, const float (&x)[16], float (&y)[16]) {
    v4f old[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) old[q] = first ? v4f{0.f, 0.f, 0.f, 0.f} : slot[q * 64];
#pragma unroll
    for (int r = 0; r < 16; ++r) y[r] = old[r >> 2][r & 3] + x[r];
}
__device__ __forceinline__ v4f *block_of(float *slot, int sub) { return reinterpret_cast<v4f *>(slot + sub * 1024) + (threadIdx.x & 63); }
// Leaves them in the slot; a later flush of the same piece adds to it.
__device__ __forceinline__ void put_block(v4f *slot, const float (&y)[16]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) slot[q * 64] = v4f{y[4 * q], y[4 * q + 1], y[4 * q + 2], y[4 * q + 3]};
}

// The contraction in fp32 straight from the inputs, for operands that have no halves: the same tiles, pieces and slots.  A
// workgroup goes through its steps of a tile for 64 of the pixels (FIRST) or two of the rows at a time: a wave has both
// blocks of 32 of them for 32 channels, or, with 128 channels and fewer, one.  dL/dS is formed in LDS, 32 columns and pixels
// of each block, while the features and weights of the next step are on their way; a register sum takes 128 products.
// Call of the compression's backward with one NaN in it, the fp32 kernels of sepcorr.hip -> here: B=2, 55x128, C=256, K=4 1172 -> 1693
// us; B=4, 48x64 503 -> 708; B=2, 47x61, C=100, K=2 221 -> 275; 55x128 on 27x64 234 -> 347.  (Tasks of 32 pixels or columns of a
// workgroup's own, nothing on its way: 3414, 1472, 430, 1263; half of the waves forming the next dL/dS while the others multiply: 1628,
// 706, 300, 351; four rows at a time: 1722, 733, 265, 353, the combined call 1.2 times as long.)
// (A function of its own, its arguments in memory: with a copy on the stack the kernels don't keep theirs in registers.)
template <bool FIRST, bool BOTH, int KC>
__device__ __attribute__((noinline)) void contract_fp32(const GradArgs *args, float *lds) {
    // (the arguments of a function are a lane's own, and what is loaded through them may lie anywhere: told here that they are not)
    typedef const __attribute__((address_space(1))) float *Floats;
    typedef v4f __attribute__((aligned(4))) u4f;
    GradArgs a;
    {
        const uint64_t at = reinterpret_cast<uint64_t>(args);
        const uint64_t lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)at), hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(at >> 32));
        const __attribute__((address_space(4))) unsigned *words = reinterpret_cast<const __attribute__((address_space(4))) unsigned *>((hi << 32) | lo);
        unsigned copy[sizeof(a) / 4];
#pragma unroll
        for (int i = 0; i < (int)(sizeof(a) / 4); ++i) copy[i] = words[i];
        __builtin_memcpy(&a, copy, sizeof(a));
    }
    constexpr int NF = vfields(BOTH, KC), GP = 36, GBLK = 32 * GP;        // floats of a pixel's row of dL/dS, of a block of it
    const int tid = threadIdx.x, lane = tid & 63, pl = lane & 31, h = lane >> 5, ncb = a.ncb;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), cb = wave % ncb, part = wave / ncb;
    const int gb = tid >> 8, gp = tid >> 3 & 31, gv = 4 * (tid & 7);      // dL/dS: this thread's block, pixel and four columns
    const int N1 = a.N1, H2 = a.H2, W2 = a.W2, C = a.C;
    const unsigned lane_off = 32 * cb + pl < C ? (unsigned)(16 * h * C + 32 * cb + pl) * 4 : OOB;
    const int npt = a.N1p / TPX, nug = a.H2p / ROWS, tiles = FIRST ? a.B * npt : a.B * nug * a.nvc;
    const int spt = FIRST ? a.nvc * H2 : a.npx, G = FIRST ? a.G1 : a.G2, wg = xcd_contiguous(blockIdx.x, gridDim.x);
    const long T = (long)tiles * spt;
    const int g0 = (int)first_step(wg, G, T), g1 = (int)first_step(wg + 1, G, T);
    const float inv_w2 = 1.f / (float)W2, inv_h2 = 1.f / (float)H2;
    const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int g = g0; g < g1;) {
        const int tile = g / spt, bv = FIRST ? 0 : tile / nug, b = FIRST ? tile / npt : bv / a.nvc;
        const Piece piece = piece_of(tile, g0, g1, spt);
        g = tile * spt + piece.end;
        const int p_end = FIRST ? N1 : min(N1, 16 * piece.end);           // pixels that are not this piece's count as none
        const int steps = FIRST ? piece.end - piece.begin : (piece.end - piece.begin + 1) / 2;
        for (int pair = 0; pair < (FIRST ? 2 : 4); ++pair) {              // of the tile's blocks of 32 pixels, or of its rows
            const int p0 = FIRST ? TPX * (tile % npt) + 64 * pair : 0, u0 = FIRST ? 0 : ROWS * (tile % nug) + 2 * pair;
            if (FIRST ? p0 >= N1 : u0 >= H2) break;
            v4f w[NF];
            float gu[KC], av[KC], mx = 0.f, mean = 0.f, fn[16];
            int am = -1;
            // weights of this thread's pixel, and features, of a step: column chunk vc and row u (FIRST), 32 pixels from p on
            // (those past an end are others', and not used)
            auto load = [&](int vc, int u, int p, bool all) __attribute__((always_inline)) {
                const size_t bp = (size_t)b * N1 + min(p + gp, N1 - 1);
                const int row = min(u, H2 - 1), v = 32 * vc + gv;
                if (!FIRST || all) {
                    if (32 * vc + 32 <= W2) {
#pragma unroll
                        for (int f = 0; f < NF; ++f) w[f] = *(const __attribute__((address_space(1))) u4f *)((Floats)vrow<KC>(a, f, bp) + v);
                    } else {
#pragma unroll
                        for (int f = 0; f < NF; ++f)
#pragma unroll
                            for (int e = 0; e < 4; ++e) w[f][e] = ((Floats)vrow<KC>(a, f, bp))[min(v + e, W2 - 1)];
                    }
                }
#pragma unroll
                for (int k = 0; k < KC; ++k) {
                    gu[k] = ((Floats)a.g_cu)[(bp * a.KT + a.k0 + k) * H2 + row];
                    av[k] = ((Floats)a.a_v)[(bp * a.KT + a.k0 + k) * H2 + row];
                }
                if constexpr (BOTH) {
                    mean = ((Floats)a.g_u)[(2 * bp + 1) * H2 + row];
                    mx = ((Floats)a.g_u)[2 * bp * H2 + row];
                    am = __float_as_int(((Floats)a.am_u)[bp * H2 + row]);
                }
                const float *src = FIRST ? a.f2 + (((size_t)b * H2 + u) * W2 + 32 * vc) * C : a.f1 + ((size_t)b * N1 + p) * C;
                const int n = min(32, FIRST ? W2 - 32 * vc : p_end - p);  // rows of the other operand there are: zeros behind them
                const __amdgpu_buffer_rsrc_t rs = make_rsrc(src, (unsigned)(n * C) * 4);
#pragma unroll
                for (int s = 0; s < 16; ++s) fn[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, lane_off + (unsigned)(s * C * 4), 0, 0));
            };
            v16f sum[2] = {zero, zero}, acc[2] = {zero, zero};
            int vc = FIRST ? piece.begin / H2 : bv % a.nvc, u = FIRST ? piece.begin - vc * H2 : u0 + gb, p = FIRST ? p0 + 32 * gb : 16 * piece.begin;
            load(vc, u, p, true);
            for (int i = 0; i < steps; ++i) {
                float *gl = lds + (i & 1) * 2 * GBLK;                     // [block][pixel][36]
                float f[16];
#pragma unroll
                for (int s = 0; s < 16; ++s) f[s] = fn[s];
                v4f x;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float y = 0.f;
                    if constexpr (BOTH) {
                        const float m = w[2 * KC + 1][e] * inv_h2, mu = mean * inv_w2;
                        y = (am == 32 * vc + gv + e ? mx + mu : mu) + (__float_as_int(w[2 * KC + 2][e]) == u ? m + w[2 * KC][e] : m);
                    }
#pragma unroll
                    for (int k = 0; k < KC; ++k) {
                        y = fmaf(w[k][e], gu[k], y);
                        y = fmaf(av[k], w[KC + k][e], y);
                    }
                    x[e] = p + gp < p_end && 32 * vc + gv + e < W2 ? y : 0.f;
                }
                *reinterpret_cast<v4f *>(gl + gb * GBLK + gp * GP + gv) = x;
                __syncthreads();
                if constexpr (FIRST) {
                    if (++u == H2) u = 0, ++vc;
                } else p += 32;
                if (i + 1 < steps) load(vc, u, p, u == 0);
                // (the contraction's index runs 16 h + s, so that a lane's part of a pixel's row lies together)
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    if (ncb == 8 || m == part) {
                        const float *gm = gl + m * GBLK;
                        float y[16];
                        if constexpr (FIRST) {
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const v4f z = *reinterpret_cast<const v4f *>(gm + pl * GP + 16 * h + 4 * q);
#pragma unroll
                                for (int e = 0; e < 4; ++e) y[4 * q + e] = z[e];
                            }
                        } else {
#pragma unroll
                            for (int s = 0; s < 16; ++s) y[s] = gm[(16 * h + s) * GP + pl];
                        }
#pragma unroll
                        for (int s = 0; s < 16; ++s) acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(y[s], f[s], acc[m], 0, 0, 0);
                        if ((i & 3) == 3 || i == steps - 1) {
                            sum[m] += acc[m];
                            acc[m] = zero;
                        }
                    }
                }
            }
            __syncthreads();
            float *slot = a.slots + (size_t)slot_of(wg, tile, piece.begin > 0, tiles, G) * (FIRST ? 4 : ROWS) * ncb * 1024;
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                if (ncb == 8 || m == part) {
                    float z[16];
#pragma unroll
                    for (int r = 0; r < 16; ++r) z[r] = sum[m][r];
                    if (!piece.whole(spt)) put_block(block_of(slot, (2 * pair + m) * ncb + cb), z);
                    else if (FIRST || u0 + m < H2) store_block<FIRST, false>(a, b, u0 + m, FIRST ? p0 + 32 * m : 32 * (bv % a.nvc), 32 * cb, z);
                }
            }
        }
    }
}

// dL/dS of one column at the pixel whose u-indexed weights are wu; wv(f): its v-indexed weights, the max/average ones as
// ma = max + average, mean = average.
template <bool BOTH, int KC, typename WV>
__device__ __forceinline__ float gval(const float *wu, WV wv, int amu_rel, int col, int u, float ma, float mean, int amv) {
    float g = 0.f;
    if constexpr (BOTH) g = (amu_rel == col ? wu[2 * KC] : wu[2 * KC + 1]) + (amv == u ? ma : mean);
#pragma unroll
    for (int k = 0; k < KC; ++k) {
        g = fmaf(wv(k), wu[k], g);
        g = fmaf(wv(KC + k), wu[KC + k], g);
    }
    return g;
}

template <bool BOTH, int KC, int NCB>
struct D1Shape {
    static constexpr int MP = NCB == 2 ? 1 : 2, MC = NCB == 8 ? 2 : 1;   // 32 x 32 blocks of a wave
    static constexpr int NB = BOTH && NCB == 8 ? 2 : 3;                  // row blocks in LDS
    static constexpr int VLDS = BOTH ? 3 * 8 * 512 * 4 : 0;              // max/average weights of the v-indexed kind
    static constexpr int BLK = NCB * 4096;
    static constexpr size_t LDS = (size_t)NB * BLK + 2 * 16384 + VLDS;
};

// Bound by what its waves wait for each other: matrix units 45 % busy (36 with the max/average terms), vector units 50 %, of the
// time a compute unit is.  With all waves in the same phase
// (operands from LDS, G, products) 209 us at B=2, 55x128, K=4, with every second wave a phase behind 195; with the other
// order of G and products in half of the waves, but one barrier a step, 213; at a raised priority around the products 214.
template <bool BOTH, int KC, int NCB>
__global__ void __launch_bounds__(512) split_d1_kernel(const GradArgs a) {
    typedef D1Shape<BOTH, KC, NCB> S;
    constexpr int NU = ufields(BOTH, KC), NF = vfields(BOTH, KC), MP = S::MP, MC = S::MC, NB = S::NB, BLK = S::BLK;
    extern __shared__ char smem[];
    char *gbuf = smem + NB * BLK;
    if (unsuitable(a)) {
        contract_fp32<true, BOTH, KC>(a.self, reinterpret_cast<float *>(smem));
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, pl = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pg = wave & 3, sh = wave >> 2;                              // dL/dS: pixels 32 pg.., columns 16 sh..
    const int mp0 = NCB == 2 ? wave & 3 : 2 * (wave & 1);                 // products: pixel groups mp0.., channel blocks mc0..
    const int mc0 = NCB == 2 ? wave >> 2 : MC * (wave >> 1);
    const int wg = xcd_contiguous(blockIdx.x, gridDim.x), npt = a.N1p / TPX, H2 = a.H2;
    const int spt = a.nvc * H2, tiles = a.B * npt;
    const long T = (long)tiles * spt;
    const int g0 = (int)first_step(wg, a.G1, T), g1 = (int)first_step(wg + 1, a.G1, T);
    v16f acc[MP][MC];
    int held = 0;              // steps in acc
    bool first = true;         // nothing of this piece is in its slot yet
    for (int g = g0; g < g1;) {
        const int tile = g / spt, r0 = g - tile * spt, vc = r0 / H2, ua = r0 - vc * H2;
        const int b = tile / npt, pt = tile - b * npt;
        const int ub = min(min(H2, ua + g1 - g), ua + FLUSH - held);
        const Piece piece = piece_of(tile, g0, g1, spt);
        g += ub - ua;
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.f2h + (size_t)(b * a.nvc + vc) * H2 * BLK, (unsigned)H2 * BLK);
        auto dma = [&](int u, int buf) __attribute__((always_inline)) {
            if constexpr (NB == 3) {
#pragma unroll
                for (int i = 0; i < NCB / 2; ++i) dma16(rs, smem + buf * BLK + (8 * i + wave) * 1024, lane * 16, (unsigned)min(u, H2 - 1) * BLK + (8 * i + wave) * 1024);
            } else if (wave < 4) {   // (a step ahead only: the waves that are a phase behind would ask too late)
#pragma unroll
                for (int i = 0; i < NCB; ++i) dma16(rs, smem + buf * BLK + (4 * i + wave) * 1024, lane * 16, (unsigned)min(u, H2 - 1) * BLK + (4 * i + wave) * 1024);
            }
        };
        const int pix = TPX * pt + 32 * pg + pl;
        const float *pu = a.pu + ((size_t)b * a.H2p * a.N1p + pix) * NU;
        const size_t pu_row = (size_t)a.N1p * NU;
        v4f pn[NU / 4];
        auto load_pu = [&](int u) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NU / 4; ++i) pn[i] = *reinterpret_cast<const v4f *>(pu + min(u, H2 - 1) * pu_row + 4 * i);
        };
        dma(ua, 0);
        if (NB == 3) dma(ua + 1, 1);
        load_pu(ua);
        const int col0 = 32 * vc + 16 * sh + 8 * h;
        const float sc = a.pscale[(size_t)b * a.N1p + pix];
        float wv[2 * KC][8];
        {
            v4f y[NF][2];
            if (a.direct) {
                const bool pok = pix < a.N1;
                const size_t bp = (size_t)b * a.N1 + (pok ? pix : 0);
#pragma unroll
                for (int f = 0; f < NF; ++f)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        y[f][q] = v4f{0.f, 0.f, 0.f, 0.f};
                        if (pok && col0 + 4 * q < a.W2) y[f][q] = *reinterpret_cast<const v4f *>(vrow<KC>(a, f, bp) + col0 + 4 * q);
                    }
            } else {
                const float *src = a.pv + (((size_t)b * a.nvc + vc) * (a.N1p / 16) + (pix >> 4)) * NF * 512 + ((4 * sh + 2 * h) * 16 + (pix & 15)) * 4;
#pragma unroll
                for (int f = 0; f < NF; ++f)
#pragma unroll
                    for (int q = 0; q < 2; ++q) y[f][q] = *reinterpret_cast<const v4f *>(src + f * 512 + q * 64);
            }
#pragma unroll
            for (int f = 0; f < 2 * KC; ++f)
#pragma unroll
                for (int e = 0; e < 8; ++e) wv[f][e] = y[f][e / 4][e % 4];
            if constexpr (BOTH) {   // kept in LDS: each thread reads its own again
                const float inv_h2 = 1.f / (float)H2;
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    v4f ma, mean;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float m = y[2 * KC + 1][q][e] * inv_h2;
                        mean[e] = m;
                        ma[e] = m + y[2 * KC][q][e];
                    }
                    char *d = gbuf + 32768 + q * 24576 + tid * 16;
                    *reinterpret_cast<v4f *>(d) = ma;
                    *reinterpret_cast<v4f *>(d + 8192) = mean;
                    *reinterpret_cast<v4f *>(d + 16384) = y[2 * KC + 2][q];
                }
            }
        }
        // halves of dL/dS of row u at this lane's pixel and eight columns, into buffer gi
        auto make_g = [&](int u, int gi) __attribute__((always_inline)) {
            float wu[NU];
#pragma unroll
            for (int i = 0; i < NU; ++i) wu[i] = pn[i / 4][i % 4];
            const int rel = BOTH ? __float_as_int(wu[BOTH ? 2 * KC + 2 : 0]) - col0 : 0;
            v4u hi, lo;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                v4f ma = {0.f, 0.f, 0.f, 0.f}, mean = ma, am = ma;
                if constexpr (BOTH) {
                    const char *d = gbuf + 32768 + q * 24576 + tid * 16;
                    ma = *reinterpret_cast<const v4f *>(d);
                    mean = *reinterpret_cast<const v4f *>(d + 8192);
                    am = *reinterpret_cast<const v4f *>(d + 16384);
                }
                float x[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    x[e] = gval<BOTH, KC>(wu, [&](int f) { return wv[f][4 * q + e]; }, rel, 4 * q + e, u, ma[e], mean[e], __float_as_int(am[e]));
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    unsigned hh, ll;
                    split2(x[2 * e], x[2 * e + 1], sc, sc, hh, ll);
                    hi[2 * q + e] = hh;
                    lo[2 * q + e] = ll;
                }
            }
            char *d = gbuf + gi * 16384 + (pg * 2 + sh) * 2048 + lane * 16;
            *reinterpret_cast<v4u *>(d) = hi;
            *reinterpret_cast<v4u *>(d + 1024) = lo;
        };
        if (held == 0) {
#pragma unroll
            for (int i = 0; i < MP; ++i)
#pragma unroll
                for (int j = 0; j < MC; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
        }
        make_g(ua, 0);
        load_pu(ua + 1);
        // (the builtin: the compiler then knows that nothing is outstanding, and waits for no requests in the loop)
        __builtin_amdgcn_s_waitcnt(0x0F70);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        // Two phases a step: operands are read and the next row's dL/dS is formed in one, multiplied in the other.  Of the two
        // waves that share a SIMD (w and w + 4) one is a phase behind: it reads and forms while the other multiplies.
        if (wave >= 4) phase_end();
        int buf = 0;
        for (int u = ua; u < ub; ++u) {
            const int gi = (u - ua) & 1;
            const int far = NB == 3 ? (buf == 0 ? 2 : buf - 1) : buf ^ 1;   // the block of the step before
            const float sign = block_sign(u);
            const char *fb = smem + buf * BLK + lane * 16, *gb = gbuf + gi * 16384 + lane * 16;
            v8h F[MC][2][2], G[MP][2][2];
#pragma unroll
            for (int j = 0; j < MC; ++j)
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int q = 0; q < 2; ++q) F[j][s][q] = *reinterpret_cast<const v8h *>(fb + ((s * NCB + mc0 + j) * 2 + q) * 1024);
#pragma unroll
            for (int i = 0; i < MP; ++i)
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int q = 0; q < 2; ++q) G[i][s][q] = *reinterpret_cast<const v8h *>(gb + ((mp0 + i) * 4 + s * 2 + q) * 1024);
            __builtin_amdgcn_sched_barrier(0);
            make_g(u + 1, gi ^ 1);
            load_pu(u + 2);
            __builtin_amdgcn_sched_barrier(0);   // (ahead of the requests: waiting for one is then not waiting for those)
            dma(u + NB - 1, far);
            __builtin_amdgcn_sched_barrier(0);
            // the row block of the next step has to be there: with three of them all but this step's requests
            if constexpr (NB == 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NCB / 2 + NU / 4) : "memory");
            else asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MP; ++i) {
                // the products with a low half first, then those of the high ones: a step's sum is rounded twice at its full
                // size, and once more when it is added to the steps before
                v16f t[MC];
#pragma unroll
                for (int j = 0; j < MC; ++j) t[j] = v16f{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 2; ++s) {
#pragma unroll
                    for (int j = 0; j < MC; ++j) t[j] = mfma(G[i][s][1], F[j][s][0], t[j]);
#pragma unroll
                    for (int j = 0; j < MC; ++j) t[j] = mfma(G[i][s][0], F[j][s][1], t[j]);
                }
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int j = 0; j < MC; ++j) t[j] = mfma(G[i][s][0], F[j][s][0], t[j]);
#pragma unroll
                for (int j = 0; j < MC; ++j) acc[i][j] += sign * t[j];
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (NB == 3) phase_end();
            else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            buf = NB == 3 ? (buf == 2 ? 0 : buf + 1) : buf ^ 1;
        }
        if (wave < 4) phase_end();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (what was requested past the last row, before the buffers are used again)
        held += ub - ua;
        const int rend = r0 + ub - ua;
        const bool ends = rend == piece.end;
        if (!ends && held < FLUSH) continue;
        float *slot = a.slots + (size_t)slot_of(wg, tile, piece.begin > 0, tiles, a.G1) * 4 * NCB * 1024;
        const bool out = ends && piece.whole(spt);
#pragma unroll
        for (int i = 0; i < MP; ++i)
#pragma unroll
            for (int j = 0; j < MC; ++j) {
                float x[16], y[16];
                v4f *block = block_of(slot, (mp0 + i) * NCB + mc0 + j);
#pragma unroll
                for (int r = 0; r < 16; ++r) x[r] = acc[i][j][r];
                sums_of_piece(block, first, x, y);
                if (out) store_block<true, true>(a, b, 0, TPX * pt + 32 * (mp0 + i), 32 * (mc0 + j), y);
                else put_block(block, y);
            }
        held = 0;
        first = ends;
    }
}

template <bool BOTH, int KC, int NCB>
struct D2Shape {
    static constexpr int MC = NCB / 2;                                   // channel blocks of a wave (and two rows)
    static constexpr int FB = NCB * 2048, VB = vfields(BOTH, KC) * 2048; // a step's f1 and v-indexed weights
    static constexpr int RS = 72, GB = ROWS * 2 * 16 * RS;               // dL/dS: [row][half][16 pixels][32 columns]
    static constexpr size_t LDS = 3 * (size_t)(FB + VB) + 2 * GB + ROWS * 32 * 4 + 1024;
};

// Bound like split_d1_kernel: matrix units 38 % busy (30 with the max/average terms), vector units 38 %.
// DIRECT: the v-indexed weights come into LDS from the tensors themselves (rows of a multiple of 4 floats, 16-byte aligned),
// otherwise from a copy laid out for it, 58 MB more written and read back at B=2, 55x128, K=4.  While the compiler waited for
// the requests of a step before the transposed reads, 260 us; with those in one block of assembly 222; with every second
// wave a phase behind 216 (all three before the factors by positions).  Row groups of one column chunk follow each other, so that an XCD's workgroups read the same weights.
template <bool BOTH, int KC, int NCB, bool DIRECT>
__global__ void __launch_bounds__(512) split_d2_kernel(const GradArgs a) {
    typedef D2Shape<BOTH, KC, NCB> S;
    constexpr int NU = ufields(BOTH, KC), NF = vfields(BOTH, KC), NX = nbounds(BOTH), MC = S::MC, FB = S::FB, VB = S::VB, RS = S::RS, GB = S::GB;
    extern __shared__ char smem[];
    char *gbuf = smem + 3 * (FB + VB);
    float *tq = reinterpret_cast<float *>(gbuf + 2 * GB);                // factors of the tile's positions, [row][column]
    int *ce = reinterpret_cast<int *>(tq + ROWS * 32);                   // what takes the channels' back
    if (unsuitable(a)) {
        contract_fp32<false, BOTH, KC>(a.self, reinterpret_cast<float *>(smem));
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rp = wave & 3, half = wave >> 2;                           // rows 2 rp, 2 rp + 1; columns 16 half.. / channels
    const int wg = xcd_contiguous(blockIdx.x, gridDim.x), nug = a.H2p / ROWS, spt = a.npx, tiles = a.B * nug * a.nvc;
    const long T = (long)tiles * spt;
    const int g0 = (int)first_step(wg, a.G2, T), g1 = (int)first_step(wg + 1, a.G2, T);
    const float inv_h2 = 1.f / (float)a.H2;
    bool first = true;
    for (int g = g0; g < g1;) {
        const int tile = g / spt, ta = g - tile * spt, tb = min(min(spt, ta + g1 - g), (ta / FLUSH + 1) * FLUSH);
        // (row groups of one column chunk follow each other: the workgroups of an XCD then read the same weights)
        const int ug = tile % nug, bv = tile / nug, vc = bv % a.nvc, b = bv / a.nvc;
        const Piece piece = piece_of(tile, g0, g1, spt);
        g += tb - ta;
        // A step's requests: f1 of that step and the weights of the one after it, whose dL/dS is formed during it.  This
        // wave's i-th one is KB 8 i + wave of the two together; every wave makes the same number of them.
        constexpr int ND = (2 * NCB + 2 * NF + 7) / 8;
        uint64_t src[ND];
        unsigned bytes[ND], off[ND], step[ND], lane_off[ND];
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const int kb = 8 * i + wave < 2 * (NCB + NF) ? 8 * i + wave : 2 * (NCB + NF) - 2 + (wave & 1);   // (one there is, once more)
            const bool is_f1 = 8 * i + 7 < 2 * NCB || (8 * i < 2 * NCB && kb < 2 * NCB);
            const int f = is_f1 ? 0 : (kb - 2 * NCB) >> 1;
            if (DIRECT) {
                const VField &v = a.self->vfield[f];   // (from memory: chosen from the arguments it would come from a copy of them on the stack)
                const int rows = __builtin_amdgcn_readfirstlane(v.rows), row = __builtin_amdgcn_readfirstlane(v.row), q = 4 * (kb & 1) + (lane >> 4);
                bytes[i] = (unsigned)a.N1 * rows * a.W2 * 4u;
                src[i] = reinterpret_cast<uint64_t>(v.src) + (size_t)b * bytes[i];
                step[i] = 16u * rows * a.W2 * 4u;
                off[i] = ((unsigned)row * a.W2 + 32 * vc) * 4u;
                lane_off[i] = 32 * vc + 4 * q < a.W2 ? ((lane & 15) * rows * a.W2 + 4 * q) * 4u : OOB;
            } else {
                bytes[i] = (unsigned)(a.N1p / 16) * VB;
                src[i] = reinterpret_cast<uint64_t>(a.pv) + ((size_t)b * a.nvc + vc) * bytes[i];
                step[i] = VB;
                off[i] = (kb - 2 * NCB) * 1024;
                lane_off[i] = lane * 16;
            }
            if (is_f1) {
                bytes[i] = (unsigned)a.npx * FB;
                src[i] = reinterpret_cast<uint64_t>(a.f1h) + (size_t)b * bytes[i];
                step[i] = FB;
                off[i] = kb * 1024;
                lane_off[i] = lane * 16;
            }
        }
        auto dma = [&](int t, int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                const int kb = 8 * i + wave < 2 * (NCB + NF) ? 8 * i + wave : 2 * (NCB + NF) - 2 + (wave & 1);
                const int at = max(0, min(kb < 2 * NCB ? t : t + 1, spt - 1));   // (past either end: not used, but read)
                dma16(make_rsrc(reinterpret_cast<const void *>(src[i]), bytes[i]), smem + buf * (FB + VB) + kb * 1024, lane_off[i],
                      __builtin_amdgcn_readfirstlane(off[i] + at * step[i]));
            }
        };
        const int p16 = lane & 15, vg = 4 * half + (lane >> 4), u0 = ROWS * ug + 2 * rp;
        const float *pu = a.pu + (((size_t)b * a.H2p + u0) * a.N1p + p16) * NU;
        v4f pn[2][NU / 4];
        auto load_pu = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int i = 0; i < NU / 4; ++i)
                    pn[r][i] = *reinterpret_cast<const v4f *>(pu + ((size_t)r * a.N1p + 16 * min(t, spt - 1)) * NU + 4 * i);
        };
        // halves of dL/dS of this lane's pixel, four columns and two rows, from weight block buf into buffer gi
        auto load_tr = [&](v4f (&tr)[2]) __attribute__((always_inline)) {   // the factors of its positions
#pragma unroll
            for (int r = 0; r < 2; ++r) tr[r] = *reinterpret_cast<const v4f *>(tq + (2 * rp + r) * 32 + 4 * vg);
        };
        // (tr: its factors, read first: the compiler waits for everything else before it when it is read where it is needed)
        auto make_g = [&](int buf, int gi, const v4f (&tr)[2]) __attribute__((always_inline)) {
            const char *wb = smem + buf * (FB + VB) + FB + (vg * 16 + p16) * 16;
            v4f m[NF], ma = {0.f, 0.f, 0.f, 0.f}, mean = ma, am = ma;
#pragma unroll
            for (int f = 0; f < NF; ++f) m[f] = *reinterpret_cast<const v4f *>(wb + f * 2048);
            if constexpr (BOTH) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    mean[e] = m[2 * KC + 1][e] * inv_h2;
                    ma[e] = m[2 * KC][e] + mean[e];
                }
                am = m[2 * KC + 2];
            }
            float x[2][4];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                float wu[NU];
#pragma unroll
                for (int i = 0; i < NU; ++i) wu[i] = pn[r][i / 4][i % 4];
                const int rel = BOTH ? __float_as_int(wu[BOTH ? 2 * KC + 2 : 0]) - (32 * vc + 4 * vg) : 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) x[r][e] = gval<BOTH, KC>(wu, [&](int f) { return m[f][e]; }, rel, e, u0 + r, ma[e], mean[e], __float_as_int(am[e]));
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                v2u hi, lo;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    unsigned hh, ll;
                    split2(x[r][2 * e], x[r][2 * e + 1], tr[r][2 * e], tr[r][2 * e + 1], hh, ll);
                    hi[e] = hh;
                    lo[e] = ll;
                }
                char *d = gbuf + gi * GB + (2 * rp + r) * 2 * 16 * RS + p16 * RS + vg * 8;
                *reinterpret_cast<v2u *>(d) = hi;
                *reinterpret_cast<v2u *>(d + 16 * RS) = lo;
            }
        };
        v16f acc[2][MC];
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int j = 0; j < MC; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[r][j][e] = 0.f;
        load_pu(ta);
        dma(ta - 1, 2);   // (for the weights; of f1 the step before, or nothing)
        dma(ta, 0);
        dma(ta + 1, 1);
        {   // factors of the tile's positions for these steps: eight waves take every eighth block of 16 pixels
            const float *bx = a.bound_v + ((size_t)b * a.nvc + vc) * (a.N1p / 16) * NX * 32 + 4 * (lane & 7);
            const float *by = a.bound_u + (size_t)b * (a.N1p / 16) * NX * a.H2p + ROWS * ug + (lane >> 3);
            const int channel = a.cback[b * 256 + (tid & 255)];
            v4f top = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < FLUSH / 8; ++i) {
                const int t = min(ta + 8 * i + wave, tb - 1);
                v4f x[NX];
                float y[NX];
#pragma unroll
                for (int n = 0; n < NX; ++n) {
                    x[n] = *reinterpret_cast<const v4f *>(bx + ((size_t)t * NX + n) * 32);
                    y[n] = by[((size_t)t * NX + n) * a.H2p];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float m = fminf(x[0][e], y[0]) + fminf(x[1][e], y[1]);
                    if constexpr (BOTH) m += x[NX - 1][e] + y[NX - 1];
                    top[e] = fmaxf(top[e], m);
                }
            }
            float *red = reinterpret_cast<float *>(gbuf);   // [wave][row][column]
            *reinterpret_cast<v4f *>(red + wave * 256 + lane * 4) = top;
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (tid < 256) {
                float m = 0.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) m = fmaxf(m, red[i * 256 + tid]);
                tq[tid] = power(scale_exponent(m));
            } else {
                ce[tid - 256] = channel;
            }
        }
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * ND) : "memory");
        {
            v4f tr[2];
            load_tr(tr);
            make_g(2, 0, tr);
        }
        load_pu(ta + 1);
        // (the builtin: the compiler then knows that nothing is outstanding, and waits for no requests in the loop)
        __builtin_amdgcn_s_waitcnt(0x0F70);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (wave >= 4) phase_end();   // (two phases a step, as in split_d1_kernel)
        int buf = 0;
        for (int t = ta; t < tb; ++t) {
            const int gi = (t - ta) & 1, far = buf == 0 ? 2 : buf - 1;
            const char *fb = smem + buf * (FB + VB) + half * MC * 2048 + lane * 16;
            v4f tr[2];
            v8h F[MC][2];
            auto load_f = [&]() __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < MC; ++j)
#pragma unroll
                    for (int q = 0; q < 2; ++q) F[j][q] = *reinterpret_cast<const v8h *>(fb + j * 2048 + q * 1024);
            };
            constexpr bool LATE = NCB == 8;   // (there are not the registers to have them while dL/dS is formed)
            if (!LATE) load_f();
            load_tr(tr);
            __builtin_amdgcn_sched_barrier(0);
            make_g(buf, gi ^ 1, tr);
            load_pu(t + 2);
            __builtin_amdgcn_sched_barrier(0);
            dma(t + 2, far);
            __builtin_amdgcn_sched_barrier(0);
            if (LATE) load_f();
            __builtin_amdgcn_sched_barrier(0);
            // lane 16 (2 h + w) + 4 r + q asks for columns 16 w + 4 q.. of pixel 8 h + r and gets column 16 w + 4 r + q of four pixels
            const char *gb = gbuf + gi * GB + (8 * h + ((lane >> 2) & 3)) * RS + ((lane >> 4) & 1) * 32 + (lane & 3) * 8 + 2 * rp * 2 * 16 * RS;
            v2u g[4][2];
            // (one block with its wait: behind the builtin the compiler waits for the requests to LDS as well)
            asm volatile(
                "ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:%c9\n\t"
                "ds_read_b64_tr_b16 %2, %8 offset:%c10\n\tds_read_b64_tr_b16 %3, %8 offset:%c11\n\t"
                "ds_read_b64_tr_b16 %4, %8 offset:%c12\n\tds_read_b64_tr_b16 %5, %8 offset:%c13\n\t"
                "ds_read_b64_tr_b16 %6, %8 offset:%c14\n\tds_read_b64_tr_b16 %7, %8 offset:%c15\n\t"
                "s_waitcnt lgkmcnt(0)"
                : "=&v"(g[0][0]), "=&v"(g[0][1]), "=&v"(g[1][0]), "=&v"(g[1][1]), "=&v"(g[2][0]), "=&v"(g[2][1]), "=&v"(g[3][0]), "=&v"(g[3][1])
                : "v"((unsigned)(uintptr_t)(__attribute__((address_space(3))) const char *)gb), "n"(4 * RS), "n"(16 * RS), "n"(20 * RS), "n"(32 * RS),
                  "n"(36 * RS), "n"(48 * RS), "n"(52 * RS)
                : "memory");
            v8h G[2][2];
#pragma unroll
            for (int i = 0; i < 4; ++i) G[i >> 1][i & 1] = __builtin_bit_cast(v8h, __builtin_shufflevector(g[i][0], g[i][1], 0, 1, 2, 3));
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(ND + NU / 2) : "memory");
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < MC; ++j) {
#pragma unroll
                for (int r = 0; r < 2; ++r) acc[r][j] = mfma(G[r][1], F[j][0], acc[r][j]);
#pragma unroll
                for (int r = 0; r < 2; ++r) acc[r][j] = mfma(G[r][0], F[j][1], acc[r][j]);
#pragma unroll
                for (int r = 0; r < 2; ++r) acc[r][j] = mfma(G[r][0], F[j][0], acc[r][j]);
            }
            __builtin_amdgcn_sched_barrier(0);
            phase_end();
            __builtin_amdgcn_sched_barrier(0);
            buf = buf == 2 ? 0 : buf + 1;
        }
        if (wave < 4) phase_end();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (what was requested past the last step, before the buffers are used again)
        const bool ends = tb == piece.end;
        float *slot = a.slots + (size_t)slot_of(wg, tile, piece.begin > 0, tiles, a.G2) * ROWS * NCB * 1024;
        const bool out = ends && piece.whole(spt);
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int j = 0; j < MC; ++j) {
                float x[16], y[16];
                v4f *block = block_of(slot, (2 * rp + r) * NCB + half * MC + j);
                const int back = ce[32 * (half * MC + j) + (lane & 31)];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const v4f t = *reinterpret_cast<const v4f *>(tq + (2 * rp + r) * 32 + 8 * q + 4 * h);
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[4 * q + e] = ldexpf(block_sign(ta / FLUSH) * acc[r][j][4 * q + e], back - exponent_of(t[e]));
                }
                sums_of_piece(block, first, x, y);
                if (!out) put_block(block, y);
                else if (u0 + r < a.H2) store_block<false, false>(a, b, u0 + r, 32 * vc, 32 * (half * MC + j), y);
            }
        first = ends;
    }
}

template <typename K>
int reserve(K k, size_t lds) {
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return sepcorr_set_error(SEPCORR_ELAUNCH, "sepcorr: cannot reserve the feature gradients' LDS");
    return 0;
}
template <bool BOTH, int KC, int NCB>
int launch_contraction(const GradArgs &a, hipStream_t s, bool first) {
    if (first) {
        if (int rc = reserve(split_d1_kernel<BOTH, KC, NCB>, D1Shape<BOTH, KC, NCB>::LDS)) return rc;
        hipLaunchKernelGGL((split_d1_kernel<BOTH, KC, NCB>), dim3(a.G1), dim3(512), (D1Shape<BOTH, KC, NCB>::LDS), s, a);
    } else {
        auto k = a.direct ? split_d2_kernel<BOTH, KC, NCB, true> : split_d2_kernel<BOTH, KC, NCB, false>;
        if (int rc = reserve(k, D2Shape<BOTH, KC, NCB>::LDS)) return rc;
        hipLaunchKernelGGL(k, dim3(a.G2), dim3(512), (D2Shape<BOTH, KC, NCB>::LDS), s, a);
    }
    return 0;
}
}  // namespace
int grad_split_operands(const GradArgs &, hipStream_t);
namespace {
template <bool BOTH, int KC>
int launch_all(const GradArgs &a, hipStream_t s) {
    {
        void *prof = sepcorr_prof_begin("grad_split_operands", s);
        const size_t lds = std::max((size_t)4096, prepare_lds(BOTH, KC, a.H2));
        int rc = reserve(grad_prepare_kernel<BOTH, KC>, lds);
        if (!rc) hipLaunchKernelGGL((grad_prepare_kernel<BOTH, KC>), dim3(a.B * (a.N1p / 16 + 2 * SLABS)), dim3(256), lds, s, a);
        if (!rc) rc = grad_split_operands(a, s);
        sepcorr_prof_end(prof);
        if (rc) return rc;
    }
    for (int first = 1; first >= 0; --first) {
        void *prof = sepcorr_prof_begin(first ? (BOTH ? "df1_both_split" : "df1_comp_split") : (BOTH ? "df2_both_split" : "df2_comp_split"), s);
        const int rc = a.ncb == 2 ? launch_contraction<BOTH, KC, 2>(a, s, first)
                     : a.ncb == 4 ? launch_contraction<BOTH, KC, 4>(a, s, first) : launch_contraction<BOTH, KC, 8>(a, s, first);
        if (first) hipLaunchKernelGGL((grad_finish_kernel<true, BOTH, KC>), dim3(a.B * (a.N1p / TPX) * a.ncb), dim3(256), 0, s, a);
        else hipLaunchKernelGGL((grad_finish_kernel<false, BOTH, KC>), dim3(a.B * (a.H2p / ROWS) * a.nvc * 2 * a.ncb), dim3(256), 0, s, a);
        sepcorr_prof_end(prof);
        if (rc) return rc;
    }
    return 0;
}
}  // namespace

#define GRAD_LAUNCHER(name, BOTH, KC) int name(const GradArgs &a, hipStream_t s) { return launch_all<BOTH, KC>(a, s); }
#define GRAD_DECL(name) int name(const GradArgs &, hipStream_t)
GRAD_DECL(grad_launch_c1); GRAD_DECL(grad_launch_c2); GRAD_DECL(grad_launch_c3); GRAD_DECL(grad_launch_c4);
GRAD_DECL(grad_launch_b1); GRAD_DECL(grad_launch_b2); GRAD_DECL(grad_launch_b3); GRAD_DECL(grad_launch_b4);
#if GRAD_IN_PART(1)
GRAD_LAUNCHER(grad_launch_c1, false, 1)
GRAD_LAUNCHER(grad_launch_c2, false, 2)
#endif
#if GRAD_IN_PART(2)
GRAD_LAUNCHER(grad_launch_c3, false, 3)
GRAD_LAUNCHER(grad_launch_c4, false, 4)
#endif
#if GRAD_IN_PART(3)
GRAD_LAUNCHER(grad_launch_b1, true, 1)
GRAD_LAUNCHER(grad_launch_b2, true, 2)
#endif
#if GRAD_IN_PART(4)
GRAD_LAUNCHER(grad_launch_b3, true, 3)
GRAD_LAUNCHER(grad_launch_b4, true, 4)
#endif

#if GRAD_IN_PART(0)
namespace {
constexpr int kMinChannels = 32;
constexpr int kPlaces = 256;   // compute units

struct GradPlan {
    bool ok, direct;
    int ncb, nvc, H2p, N1p, npx, G1, G2;
    size_t pv, pu, pscale, block_bad, bound_v, bound_u, pmax, cback, f1h, f2h, slots;
    size_t bytes() const { return pv + pu + pscale + block_bad + bound_v + bound_u + pmax + cback + f1h + f2h + slots + 1024; }
};
size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// aligned: the tensors of the v-indexed weights begin at multiples of 16 bytes.
GradPlan plan(int B, int N1, int H2, int W2, int C, int both, int kc, int KT, bool aligned) {
    GradPlan p = {};
    if (C < kMinChannels || C > 256 || kc < 1 || kc > 4) return p;
    if ((double)B * N1 * H2 * W2 * (C + 64) < SPLIT_GRAD_LEAST) return p;
    p.ncb = C <= 64 ? 2 : C <= 128 ? 4 : 8;
    p.nvc = (W2 + 31) / 32;
    p.H2p = (H2 + ROWS - 1) / ROWS * ROWS;
    p.N1p = (N1 + TPX - 1) / TPX * TPX;
    p.npx = (N1 + 15) / 16;
    const int nf = vfields(both, kc);
    const long tiles1 = (long)B * (p.N1p / TPX), tiles2 = (long)B * (p.H2p / ROWS) * p.nvc;
    const long T1 = tiles1 * p.nvc * H2, T2 = tiles2 * p.npx;
    if (T1 > (1L << 30) || T2 > (1L << 30) || prepare_lds(true, 4, H2) > 150 * 1024) return p;
    if ((size_t)H2 * p.ncb * 4096 >= (1u << 30) || (size_t)p.npx * p.ncb * 2048 >= (1u << 30) || (size_t)(p.N1p / 16) * nf * 2048 >= (1u << 30)) return p;
    p.direct = aligned && W2 % 4 == 0 && (size_t)p.N1p * (KT > 2 ? KT : 2) * W2 * 4 < (1u << 30);
    p.G1 = (int)(T1 < kPlaces ? T1 : kPlaces);
    p.G2 = (int)(T2 < kPlaces ? T2 : kPlaces);
    p.pv = p.direct ? 0 : align256((size_t)B * p.nvc * (p.N1p / 16) * nf * 2048);
    p.pu = align256((size_t)B * p.H2p * p.N1p * ufields(both, kc) * 4);
    p.pscale = align256((size_t)B * p.N1p * 4);
    p.block_bad = align256((size_t)B * (p.N1p / 16) * 4);
    p.bound_v = align256((size_t)B * p.nvc * (p.N1p / 16) * nbounds(both) * 128);
    p.bound_u = align256((size_t)B * (p.N1p / 16) * nbounds(both) * p.H2p * 4);
    p.pmax = align256((size_t)2 * B * SLABS * 256 * 4);
    p.cback = align256((size_t)2 * B * 256 * 4);
    p.f1h = align256((size_t)B * p.npx * p.ncb * 2048);
    p.f2h = align256((size_t)B * p.nvc * H2 * p.ncb * 4096);
    const size_t s1 = slots_of(tiles1, p.G1) * 4 * p.ncb * 4096, s2 = slots_of(tiles2, p.G2) * ROWS * p.ncb * 4096;
    p.slots = s1 > s2 ? s1 : s2;
    p.ok = true;
    return p;
}
}  // namespace

int grad_split_operands(const GradArgs &a, hipStream_t s) {
    auto k = a.ncb == 2 ? grad_split_kernel<2> : a.ncb == 4 ? grad_split_kernel<4> : grad_split_kernel<8>;
    hipLaunchKernelGGL(k, dim3(a.B * (a.nvc * a.H2 + a.npx)), dim3(256), 0, s, a);
    return 0;
}

size_t split_grad_bytes(int B, int N1, int H2, int W2, int C) {
    // (the most channels of one launch; 16-byte aligned weights, as every allocation is)
    const GradPlan p = plan(B, N1, H2, W2, C, 1, 4, 8, true);
    return p.ok ? p.bytes() : 0;
}

namespace {
GradPlan plan_of(int both, int kc, const GradArgs &a) {
    uintptr_t bits = reinterpret_cast<uintptr_t>(a.a_u) | reinterpret_cast<uintptr_t>(a.g_cv);
    if (both) bits |= reinterpret_cast<uintptr_t>(a.g_v) | reinterpret_cast<uintptr_t>(a.am_v);
    return plan(a.B, a.N1, a.H2, a.W2, a.C, both, kc, a.KT, bits % 16 == 0);
}
}  // namespace

bool split_grad_fits(int both, int kc, const GradArgs &a, size_t ws_bytes) {
    const GradPlan p = plan_of(both, kc, a);
    return p.ok && ws_bytes >= p.bytes();
}

int split_grad(int both, int kc, GradArgs a, void *ws, size_t ws_bytes, hipStream_t s) {
    const GradPlan p = plan_of(both, kc, a);
    if (!p.ok || ws == nullptr || ws_bytes < p.bytes()) return sepcorr_set_error(SEPCORR_EWORKSPACE, "sepcorr: feature gradients: scratch does not suffice");
    a.ncb = p.ncb; a.nvc = p.nvc; a.H2p = p.H2p; a.N1p = p.N1p; a.npx = p.npx; a.G1 = p.G1; a.G2 = p.G2; a.direct = p.direct;
    char *base = static_cast<char *>(ws);
    auto take = [&](size_t n) { char *r = base; base += n; return r; };
    a.slots = reinterpret_cast<float *>(take(p.slots));
    a.pv = reinterpret_cast<float *>(take(p.pv));
    a.pu = reinterpret_cast<float *>(take(p.pu));
    a.pscale = reinterpret_cast<float *>(take(p.pscale));
    a.block_bad = reinterpret_cast<int *>(take(p.block_bad));
    a.bound_v = reinterpret_cast<float *>(take(p.bound_v));
    a.bound_u = reinterpret_cast<float *>(take(p.bound_u));
    a.pmax = reinterpret_cast<unsigned *>(take(p.pmax));
    a.cback = reinterpret_cast<int *>(take(p.cback));
    a.f1h = take(p.f1h);
    a.f2h = take(p.f2h);
    a.count = reinterpret_cast<unsigned *>(take(256));
    static_assert(sizeof(GradArgs) <= 768, "room for the arguments");
    a.self = reinterpret_cast<GradArgs *>(take(768));
    for (int f = 0; f < vfields(both, kc); ++f) {
        VField &v = a.vfield[f];
        if (f < 2 * kc) v.src = f < kc ? a.a_u : a.g_cv, v.rows = a.KT, v.row = a.k0 + f % kc;
        else if (f < 2 * kc + 2) v.src = a.g_v, v.rows = 2, v.row = f - 2 * kc;
        else v.src = reinterpret_cast<const float *>(a.am_v), v.rows = 1, v.row = 0;
    }
    auto launch = both ? (kc == 1 ? grad_launch_b1 : kc == 2 ? grad_launch_b2 : kc == 3 ? grad_launch_b3 : grad_launch_b4)
                       : (kc == 1 ? grad_launch_c1 : kc == 2 ? grad_launch_c2 : kc == 3 ? grad_launch_c3 : grad_launch_c4);
    if (int rc = launch(a, s)) return rc;
    if (hipGetLastError() != hipSuccess) return sepcorr_set_error(SEPCORR_ELAUNCH, "sepcorr: feature gradients: launch failed");
    return 0;
}
#endif
