// Forward-type sweeps on the 16-bit matrix units, at fp32 accuracy.
//
// The same sums as the fp32 sweep (fwd_kernel in sepcorr.hip): S[p,q] = <f1[p,:], f2[q,:]> is made 32x32 pixels at a
// time and reduced at once, over the columns v of fmap2 into out_u and over its rows u into out_v.
//
// Contraction.  A pixel's channels are scaled by a power of two that brings the largest of them into [2^14, 2^15) and
// each is written as h + 2^-11 l, h = fp16(x), l = fp16(2^11 (x - h)): 22 significant bits down to 2^-28 of the pixel's
// largest channel (both halves of a smaller one are subnormal), 2^-50 of it below.  A product is h h + 2^-11 (h l + l h):
// three v_mfma_f32_32x32x16_f16, which accumulate in fp32, in place of eight v_mfma_f32_32x32x2_f32 of twice the length.
// What is left out (l l) and what the halves do not hold are below the rounding of the fp32 sum, and a sum of 256
// products is rounded 16 times instead of 128 (the sum of the cross terms, 2^-11 of it, 32 times).
// Scaling by powers of two is exact and taken back in fp32.  A pixel that has no such form (a channel that is inf or
// NaN, a largest channel outside [2^-60, 2^61), max(2, C / 32) channels below 2^-28 of it that are not zero) is marked,
// and 32x32 blocks with a marked pixel are multiplied with fp32 MFMAs straight from the inputs.
//
// Work split.  A step = 128 pixels p x 32 columns v of one row u: the workgroup's four waves own 32 pixels each, whose
// halves stay in registers for the whole sweep (128 registers at C = 256), and share the row block of fmap2 (33 KB at
// C = 256), which is DMA'd into LDS while the step before is multiplied.  Per step and compute unit that is 33 KB from
// the L2 and 132 KB from LDS (198 where the high halves are read twice) for 1536 cycles of matrix work of each wave.
// The steps of all tiles (levels, images, column chunks, pixel tiles, rows) are dealt out evenly.  Results of the other
// chunks and of other pieces of a tile are left in scratch and put together by split_finish_kernel in a fixed order.
#include "split_sweep.h"

#include <math.h>

#include <type_traits>

#include "sepcorr.h"
#include "sepcorr_internal.h"

#ifndef SPLIT_PART
#define SPLIT_PART (-1)
#endif
#define SPLIT_IN_PART(n) (SPLIT_PART < 0 || SPLIT_PART == (n))

namespace {
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int TPX = 128;          // pixels of a step
// A row block: one KB per (16-channel step, half) holding the 16 bytes of each lane in lane order (lane 32 g + i:
// column i, channels 16 s + 8 g + 0..7), then one KB with the 32 factors that take the scaling back and a mark.
__host__ __device__ constexpr int block_bytes(int nk) { return (2 * nk + 1) * 1024; }
constexpr int MARK = 32;          // index of the mark among the floats of the last KB

__device__ __forceinline__ int vmap(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *p, unsigned bytes) {
    const uint64_t addr = reinterpret_cast<uint64_t>(p);
    const uint64_t lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)addr);
    const uint64_t hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(addr >> 32));
    const int n = __builtin_amdgcn_readfirstlane((int)bytes);
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>((hi << 32) | lo), 0, n, 0x00020000);
}
__device__ __forceinline__ void wave_halves(float x, float &lo, float &hi) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    lo = __uint_as_float(r[0]);
    hi = __uint_as_float(r[1]);
}
// max(a, b) as a > b ? a : b of a running maximum a that is never NaN: one instruction, a NaN in b is passed over
__device__ __forceinline__ float maxnum(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// Pins the computation of x to where it is written: the compiler otherwise sinks it behind the matrix work it is
// meant to run beside.
template <typename T>
__device__ __forceinline__ void keep_here(T &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ int xcd_contiguous(int bid, int n) {
    const int c = bid & 7, slot = bid >> 3, q = n >> 3, r = n & 7;
    return c * q + (c < r ? c : r) + slot;
}
// bits of the largest magnitude of a pixel -> factor into [2^14, 2^15) and the factor back; false: no such form
__device__ __forceinline__ bool pixel_scale(unsigned m, float &fwd, float &back) {
    const unsigned e = m >> 23;
    if (m == 0) { fwd = 1.f; back = 1.f; return true; }
    if (e < 67 || e > 187) { fwd = 0.f; back = 1.f; return false; }
    fwd = __uint_as_float((268u - e) << 23);
    back = __uint_as_float((e - 14u) << 23);
    return true;
}
// low halves are held times 2^11: they are as far from the subnormals as high ones
constexpr float LOW_UNIT = 1.f / 2048.f;
// (a marked pixel has factor 0 and may hold inf: its halves are zeros, not NaN)
__device__ __forceinline__ void split8(const float (&x)[8], float f, v8h &h, v8h &l) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float y = f == 0.f ? 0.f : x[e] * f;
        const _Float16 hh = (_Float16)y;
        h[e] = hh;
        l[e] = (_Float16)((y - (float)hh) * (1.f / LOW_UNIT));
    }
}
constexpr unsigned OOB = 0x80000000u;   // a byte offset above every buffer size used here: reads as zero
// channels c .. c+7 of the pixel that begins at byte `off` of the buffer, zero from channel C on
__device__ __forceinline__ void load8(__amdgpu_buffer_rsrc_t r, unsigned off, int c, int C, bool vec, float (&x)[8]) {
    if (vec) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const v4f y = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, c + 4 * g < C ? off + (c + 4 * g) * 4u : OOB, 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) x[4 * g + e] = y[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            x[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, c + e < C ? off + (c + e) * 4u : OOB, 0, 0));
    }
}
__device__ __forceinline__ unsigned magnitude(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// A block with a marked pixel: fp32 products straight from the inputs, this lane's pixel of image 1 at byte o1 of n1, of
// fmap2 at byte o2 of n2 (OOB: none), the first `cols` columns of this lane's half.  16 channels a turn; a lane's eight are
// contiguous, and the next turn's are on their way.  A function of its own: its registers would otherwise be taken from
// the sweep's.
// B=2, 55x128, max/average: 0.18 ms without a marked pixel, 0.44 with one in image 1, 0.86 with all of them marked; with one
// channel a turn 0.88 and 2.78 ms, the fp32 sweep 0.44.
__device__ __attribute__((noinline)) v16f products_fp32(const float *f1, unsigned n1, unsigned o1, const float *f2, unsigned n2, unsigned o2,
                                                        int C_in, int cols) {
    const int C = __builtin_amdgcn_readfirstlane(C_in), h = (threadIdx.x >> 5) & 1;
    const __amdgpu_buffer_rsrc_t r1 = make_rsrc(f1, n1), r2 = make_rsrc(f2, n2);
    const bool vec = (C & 3) == 0;
    v16f acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float y[8], z[8];
    load8(r2, o2, 8 * h, C, vec, y);
    load8(r1, o1, 8 * h, C, vec, z);
#pragma unroll 1
    for (int c = 16; c < C + 16; c += 16) {
        float yn[8], zn[8];
        load8(r2, o2, c + 8 * h, C, vec, yn);
        load8(r1, o1, c + 8 * h, C, vec, zn);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(y[e], z[e], acc, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = yn[e], z[e] = zn[e];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = vmap(r, 0) < cols ? acc[r] : 0.f;   // (an inf of image 1 times nothing is no NaN)
    return acc;
}

// The workgroups that hold the steps [t0, t1) when T steps are dealt out evenly to G workgroups.
__device__ __forceinline__ void pieces_of(long t0, long t1, int G, long T, int &w0, int &w1) {
    w0 = (int)((t0 * G) / T);
    while (w0 > 0 && ((long)w0 * T) / G > t0) --w0;
    while (((long)(w0 + 1) * T) / G <= t0) ++w0;
    w1 = w0;
    while (((long)(w1 + 1) * T) / G < t1) ++w1;
}

// Finished columns v .. v+3 of out_v (weighted: channel q; max/avg: q = 0 max, 1 sum, 2 argmax) of pixel bp.
template <int MODE>
__device__ __forceinline__ void store_v(const SplitArgs &a, const SplitLevel &L, size_t bp, int q, int v, v4f x) {
    const int W2 = L.W2;
    float *dst;
    if constexpr (MODE == SPLIT_WEIGHTED) {
        const size_t row = bp * a.KT + a.k0 + q;
        dst = L.out_v + row * W2 + v;
        if (a.dlog) {
            const float m = L.st_ov[2 * row], il = 1.f / L.st_ov[2 * row + 1], dot = L.dot_ov[row];
            v4f z = {0.f, 0.f, 0.f, 0.f};
            if (v + 4 <= W2) {
                __builtin_memcpy(&z, L.z_ov + row * W2 + v, 16);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (v + e < W2) z[e] = L.z_ov[row * W2 + v + e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = __expf(z[e] - m) * il * (x[e] - dot);
        }
    } else if (MODE == SPLIT_ARGMAX && q == 2) {
        dst = reinterpret_cast<float *>(L.am_v + bp * W2 + v);
    } else {
        dst = L.out_v + (bp * 2 + q) * W2 + v;
        if (q == 1) x = x / (float)L.H2;
    }
    // (16 bytes at a 4-byte aligned address: rows of any length.  Four stores of 4 bytes in rows that are not a multiple of 4 long
    // cost a piece some 10 us: B=3, four levels of 47x115, C=56, K=4 450 us, 410 us like this, 350 with the fp32 sweep; C=256,
    // K=2 over four levels of 47x156 229 and 217.)
    if (v + 4 <= W2) {
        __builtin_memcpy(dst, &x, 16);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (v + e < W2) dst[e] = x[e];
    }
}

#if SPLIT_IN_PART(0)
// Splits the levels of fmap2 into row blocks, and image 1 into blocks of 32 consecutive pixels: one workgroup per
// block, eight lanes per pixel.  Bound by its traffic (4 bytes read and written per value).
template <int NK>
__global__ void __launch_bounds__(256) split_prepare_kernel(const SplitArgs a) {
    const int i = threadIdx.x >> 3, j = threadIdx.x & 7;
    int n, v;                                            // pixels from `src` on, this lane's among them
    const float *src;
    char *dst;
    if ((int)blockIdx.x < a.blocks) {
        int l = a.nlev - 1;
        while (l > 0 && (int)blockIdx.x < a.lev[l].block0) --l;
        const SplitLevel &L = a.lev[l];
        const int blk = blockIdx.x - L.block0;           // (b * nvc + vc) * H2 + u
        const int u = blk % L.H2, bc = blk / L.H2, vc = bc % L.nvc, b = bc / L.nvc;
        n = L.W2;
        v = 32 * vc + i;
        src = L.f2 + ((size_t)b * L.H2 + u) * L.W2 * a.C;
        dst = L.planes + (size_t)blk * block_bytes(NK);
    } else {
        const int blk = blockIdx.x - a.blocks, nb = (a.N1 + 31) / 32, b = blk / nb, k = blk - b * nb;   // b * nb + k
        n = min(32, a.N1 - 32 * k);
        v = i;
        src = a.f1 + ((size_t)b * a.N1 + 32 * k) * a.C;
        dst = a.f1_planes + (size_t)blk * block_bytes(NK);
    }
    const bool ok = v < n, vec = (a.C & 3) == 0;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(src, (unsigned)n * a.C * 4u);
    constexpr int M = NK / 4;                            // 8 lanes x 8 channels = 4 channel steps
    float x[M][8];
    unsigned m = 0, tiny = 0;
#pragma unroll
    for (int t = 0; t < M; ++t) {
        load8(rs, ok ? (unsigned)v * a.C * 4u : OOB, 64 * t + 8 * j, a.C, vec, x[t]);
#pragma unroll
        for (int e = 0; e < 8; ++e) m = max(m, magnitude(x[t][e]));
    }
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) m = max(m, (unsigned)__shfl_xor((int)m, d));
    // Non-zero channels below 2^-28 of the largest: a few are let pass, each with an error below 2^-50 of the largest.
    // (Among 256 normal ones a single one is found once in some 600 000 pixels; beside one channel of 2^14 times the
    // others two are found in one pixel of 12 000, beside one of 2^20 eight in one of a million.)
    const unsigned least = m > (28u << 23) ? (m & 0x7f800000u) - (28u << 23) : 0;
#pragma unroll
    for (int t = 0; t < M; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e) tiny += magnitude(x[t][e]) - 1u < least - 1u && least > 0;
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) tiny += (unsigned)__shfl_xor((int)tiny, d);
    float f, back;
    const bool good = pixel_scale(m, f, back) && tiny < max(2u, (unsigned)a.C / 32);
    if (!good) f = 0.f, back = 1.f;
#pragma unroll
    for (int t = 0; t < M; ++t) {
        v8h h, lo;
        split8(x[t], f, h, lo);
        char *d = dst + (4 * t + (j >> 1)) * 2048 + (32 * (j & 1) + i) * 16;
        *reinterpret_cast<v8h *>(d) = h;
        *reinterpret_cast<v8h *>(d + 1024) = lo;
    }
    float *tail = reinterpret_cast<float *>(dst + 2 * NK * 1024);
    if (j == 0) tail[i] = back;
    const int bad = __syncthreads_or(!good);
    if (threadIdx.x < 4) tail[MARK + threadIdx.x] = bad ? 1.f : 0.f;
}

// Puts together what the sweep left in scratch.  Blocks [0, 4 tiles): columns of out_v of tiles that were dealt out in
// pieces, one block per group of four accumulator registers, pieces in row order (equal maxima keep the lower row).
// The blocks behind them: out_u, 64 pixels x 32 rows each, chunks in column order.
template <int MODE, int Q>
__global__ void __launch_bounds__(256) split_finish_kernel(const SplitArgs a) {
    if ((int)blockIdx.x < 4 * a.tiles) {
        const int tile = blockIdx.x >> 2, rg = blockIdx.x & 3;
        int l = a.nlev - 1;
        while (l > 0 && tile < a.lev[l].tile0) --l;
        const SplitLevel &L = a.lev[l];
        const int t = tile - L.tile0, pt = t % a.npt, bc = t / a.npt, vc = bc % L.nvc, b = bc / L.nvc;
        const long t0 = L.step0 + (long)t * L.H2, T = a.steps;
        int w0, w1;
        pieces_of(t0, t0 + L.H2, a.G, T, w0, w1);
        if (w0 == w1) return;
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        const int pix = (a.pt0 + pt) * TPX + 32 * wave + (lane & 31), v = 32 * vc + vmap(4 * rg, lane >> 5);
        v4f x[Q];
        constexpr int FL = Q > 2 ? 3 : 4;   // pieces in flight
        for (int wb = w0; wb <= w1; wb += FL) {
            v4f y[FL][Q];
#pragma unroll
            for (int i = 0; i < FL; ++i) {
                const int w = min(wb + i, w1), slot = 2 * w + ((long)w * T / a.G > t0 ? 0 : 1);
                const v4f *src = reinterpret_cast<const v4f *>(a.slots + (size_t)slot * Q * 4096) + (wave * 4 + rg) * 64 + lane;
#pragma unroll
                for (int q = 0; q < Q; ++q) y[i][q] = src[q * 1024];
            }
#pragma unroll
            for (int i = 0; i < FL; ++i) {
                if (wb + i > w1) break;
                if (wb + i == w0) {
#pragma unroll
                    for (int q = 0; q < Q; ++q) x[q] = y[i][q];
                } else if constexpr (MODE == SPLIT_WEIGHTED) {
#pragma unroll
                    for (int q = 0; q < Q; ++q) x[q] += y[i][q];
                } else {
                    x[1] += y[i][1];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (y[i][0][e] > x[0][e]) {
                            x[0][e] = y[i][0][e];
                            if constexpr (MODE == SPLIT_ARGMAX) x[2][e] = y[i][2][e];
                        }
                }
            }
        }
        if (pix < a.N1 && v < L.W2) {
#pragma unroll
            for (int q = 0; q < Q; ++q) store_v<MODE>(a, L, (size_t)b * a.N1 + pix, q, v, x[q]);
        }
        return;
    }
    __shared__ float sh[Q][64][33];
    const int fb = blockIdx.x - 4 * a.tiles;
    int l = a.nlev - 1;
    while (l > 0 && fb < a.lev[l].fin0) --l;
    const SplitLevel &L = a.lev[l];
    const int nuc = (L.H2 + 31) / 32;
    const int k = fb - L.fin0, uc = k % nuc, r = k / nuc, ph = r % (2 * a.npt), b = r / (2 * a.npt);
    const int N1p = a.npt * TPX, H2 = L.H2, nvc = L.nvc;
    {
        const int p = threadIdx.x & 63;
#pragma unroll 2
        for (int i = threadIdx.x >> 6; i < 32; i += 4) {
            const int u = 32 * uc + i;
            if (u >= H2) break;
            float x[Q];
            for (int vb = 0; vb < nvc; vb += 4) {   // four chunks in flight
                float y[4][Q];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float *src = L.part + (((size_t)(b * nvc + min(vb + j, nvc - 1)) * H2 + u) * Q) * N1p + 64 * ph + p;
#pragma unroll
                    for (int q = 0; q < Q; ++q) y[j][q] = src[(size_t)q * N1p];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (vb + j >= nvc) break;
                    if (vb + j == 0) {
#pragma unroll
                        for (int q = 0; q < Q; ++q) x[q] = y[j][q];
                    } else if constexpr (MODE == SPLIT_WEIGHTED) {
#pragma unroll
                        for (int q = 0; q < Q; ++q) x[q] += y[j][q];
                    } else {
                        x[1] += y[j][1];
                        if (y[j][0] > x[0]) {
                            x[0] = y[j][0];
                            if constexpr (MODE == SPLIT_ARGMAX) x[2] = y[j][2];
                        }
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < Q; ++q) sh[q][p][i] = x[q];
        }
    }
    __syncthreads();
    const int u = 32 * uc + (threadIdx.x & 31);
    if (u >= H2) return;
    for (int p = threadIdx.x >> 5; p < 64; p += 8) {
        const int pix = a.pt0 * TPX + 64 * ph + p;
        if (pix >= a.N1) break;
        const size_t bp = (size_t)b * a.N1 + pix;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            float x = sh[q][p][threadIdx.x & 31];
            if constexpr (MODE == SPLIT_WEIGHTED) {
                const size_t row = bp * a.KT + a.k0 + q;
                if (a.dlog) x = __expf(L.z_ou[row * H2 + u] - L.st_ou[2 * row]) / L.st_ou[2 * row + 1] * (x - L.dot_ou[row]);
                L.out_u[row * H2 + u] = x;
            } else if (MODE == SPLIT_ARGMAX && q == 2) {
                L.am_u[bp * H2 + u] = __float_as_int(x);
            } else {
                L.out_u[(bp * 2 + q) * H2 + u] = q == 1 ? x / (float)L.W2 : x;
            }
        }
    }
}
#endif

// The max/avg modes and one weight channel fit 256 registers, and so do two channels where a pixel's halves take few
// (C <= 64): two workgroups per compute unit, one wave's reductions run beside the other's matrix work.  More channels
// take the whole register file, and a wave reduces one row while it multiplies the next.  Both ways measured (two
// workgroups / one): C=256 max/avg, B=2, 55x128 0.149 / 0.166 ms, two channels over the four levels of 47x156 0.225 / 0.212;
// C=64 two channels B=4, 80x120 0.270 / 0.342, four 0.895 / 0.521; C=100 two channels B=2, 47x61 0.054 / 0.046.
__host__ __device__ constexpr bool pipelined(int mode, int kc, int nk) { return mode == SPLIT_WEIGHTED && kc > 1 && !(kc == 2 && nk == 4); }

// NK: channel steps of 16 (C <= 16 NK, the rest zeros).  Measured at B=2, 55x128, C=256: max/avg/argmax 0.454 ms with the
// fp32 sweep, 0.158 ms here (+ 0.014 split_prepare_kernel, 0.033 split_finish_kernel); four weighted sums 0.474 and
// 0.203 ms (+ 0.014 and 0.034).  The matrix instructions alone take 0.061 ms at 2.4 GHz; the clock falls to 1.5 to 1.7 GHz
// under them (matrix units 53 and 34 % busy), the rest is the vector work of the reductions, the reads of the row block
// from LDS and the beginning and end of every step.
template <int MODE, int KC, int NK>
__global__ void __launch_bounds__(256, pipelined(MODE, KC, NK) ? 1 : 2) split_sweep_kernel(const SplitArgs a) {
    constexpr bool WT = MODE == SPLIT_WEIGHTED;
    constexpr bool PIPE = pipelined(MODE, KC, NK);
    constexpr int Q = WT ? KC : (MODE == SPLIT_ARGMAX ? 3 : 2);
    constexpr int BLK = block_bytes(NK), BF = BLK / 4, NBUF = PIPE ? 3 : 2;
    // The low halves' products are summed apart, in units of LOW_UNIT.  The max/avg modes have no registers left for a second
    // accumulator at NK = 16 (argmax would spill 29): they sum the products of the low halves first, scale the sum and read
    // the high halves from LDS once more for the rest.  Measured at B=2, 55x128, C=256 (whole call; one accumulator with low
    // halves in units of 1, which loses bits of small channels, first): argmax 185 us, 189 as it is, 197 with two
    // accumulators; max/average 169, 178, 174 (kept like argmax, so that both give the same bits); one channel 166, 175, 168;
    // four channels 215, 229 and 223.
    constexpr bool TWO_ACC = WT || NK < 16;
    extern __shared__ float smem[];                       // NBUF row blocks, then the u-indexed weights of each wave
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    float *wus = smem + NBUF * BF + wave * (KC * 128);       // [k][row & 3][pixel]
    const int wg = xcd_contiguous(blockIdx.x, gridDim.x);
    const long T = a.steps;
    const int g0 = (int)(wg * T / a.G), g1 = (int)((wg + 1) * T / a.G);
    const int N1 = a.N1, C = a.C, N1p = a.npt * TPX;

    for (int g = g0; g < g1;) {
        // (max/avg modes: derived afresh for every piece.  What follows from them is otherwise worked out ahead of the loop over
        // the pieces, spilled and read back one by one where a piece begins; argmax, B=2, 55x128: 192 -> 189 us.  One weight
        // channel has the registers for it: 168 us as it is, 175 afresh.)
        int tid = threadIdx.x;
        if constexpr (!WT) keep_here(tid);
        const int lane = tid & 63, pl = lane & 31, h = lane >> 5;
        int l = a.nlev - 1;
        while (l > 0 && g < a.lev[l].step0) --l;
        const SplitLevel &L = a.lev[l];
        const int H2 = L.H2, W2 = L.W2, nvc = L.nvc;
        const int t = (g - L.step0) / H2, ua = (g - L.step0) - t * H2, ub = min(H2, ua + g1 - g);
        const int pt = t % a.npt, bc = t / a.npt, vc = bc % nvc, b = bc / nvc;
        g += ub - ua;
        const int cols = W2 - 32 * vc - 4 * h;   // register r holds column vmap(r, 0) of this half: one of the image if below
        const int pix = (a.pt0 + pt) * TPX + 32 * wave + pl;
        const bool pok = pix < N1;
        const size_t bp = (size_t)b * N1 + (pok ? pix : 0);
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(L.planes + (size_t)bc * H2 * BLK, (unsigned)H2 * BLK);
        constexpr int NDMA = (2 * NK + 4) / 4;   // KBs of a row block per wave
        auto dma = [&](int u, int buf, int i) {
            const int kb = 4 * i + wave;
            if (4 * i + 3 < 2 * NK + 1 || kb < 2 * NK + 1)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)(smem + buf * BF + kb * 256), 16,
                                                         lane * 16, u * BLK + kb * 1024, 0, 0);
        };
#pragma unroll
        for (int i = 0; i < NDMA; ++i) dma(ua, 0, i);
        if constexpr (PIPE) {
#pragma unroll
            for (int i = 0; i < NDMA; ++i) dma(ua + 1, 1, i);
        }
        // Everything a piece begins with is requested before any of it is waited for (in turn it takes 10 us).
        float vmax[16], vsum[16], wvr[KC][16], rv[KC][16];   // running state over u, accumulator layout
        int vidx[16];
        float wpre[KC][2], wm[KC], wil[KC], vm[KC], vil[KC];
        if constexpr (WT) {
#pragma unroll
            for (int k = 0; k < KC; ++k) {
                const size_t row = bp * a.KT + a.k0 + k;
                vm[k] = 0.f; vil[k] = 1.f; wm[k] = 0.f; wil[k] = 1.f;
                if (a.logits) { vm[k] = L.st_wv[2 * row]; vil[k] = L.st_wv[2 * row + 1]; wm[k] = L.st_wu[2 * row]; wil[k] = L.st_wu[2 * row + 1]; }
            }
            const __amdgpu_buffer_rsrc_t rw = make_rsrc(L.wv + ((size_t)b * N1 + min((a.pt0 + pt) * TPX, N1 - 1)) * a.KT * W2,
                                                        (unsigned)min(TPX, N1 - (a.pt0 + pt) * TPX) * a.KT * W2 * 4u);
            const unsigned row0 = ((32 * wave + pl) * a.KT + a.k0) * W2;
            if ((W2 & 3) == 0 || 32 * vc + 32 <= W2) {   // (loads of 16 bytes need 4-byte alignment only)
#pragma unroll
                for (int k = 0; k < KC; ++k)
#pragma unroll
                    for (int g4 = 0; g4 < 4; ++g4) {
                        const int v = 32 * vc + vmap(4 * g4, h);
                        const v4f y = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rw, v < W2 ? (row0 + k * W2 + v) * 4u : OOB, 0, 0));
#pragma unroll
                        for (int e = 0; e < 4; ++e) wvr[k][4 * g4 + e] = y[e];
                    }
            } else {
#pragma unroll
                for (int k = 0; k < KC; ++k)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int v = 32 * vc + vmap(r, h);
                        wvr[k][r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rw, v < W2 ? (row0 + k * W2 + v) * 4u : OOB, 0, 0));
                    }
            }
        }
        // this wave's pixels: halves of all channels, in operand layout
        v8h fh[NK], fl[NK];
        float back;
        bool fbad;
        {
            const int nb = (N1 + 31) / 32, k = (a.pt0 + pt) * 4 + wave;   // (a block past the image is read as zeros)
            const __amdgpu_buffer_rsrc_t r1 = make_rsrc(a.f1_planes + ((size_t)b * nb + min(k, nb - 1)) * BLK, k < nb ? BLK : 0);
            back = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r1, pl * 4, 2 * NK * 1024, 0));
            fbad = __builtin_amdgcn_readfirstlane(__builtin_amdgcn_raw_buffer_load_b32(r1, MARK * 4, 2 * NK * 1024, 0)) != 0;
#pragma unroll
            for (int s = 0; s < NK; ++s) {
                fh[s] = __builtin_bit_cast(v8h, __builtin_amdgcn_raw_buffer_load_b128(r1, lane * 16, s * 2048, 0));
                fl[s] = __builtin_bit_cast(v8h, __builtin_amdgcn_raw_buffer_load_b128(r1, lane * 16, s * 2048 + 1024, 0));
            }
        }
        // the u-indexed weights of four rows at a time: a lane reads two rows of its pixel, which lie in one line
        auto wu_load = [&](int grp) {
#pragma unroll
            for (int k = 0; k < KC; ++k)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int u = 4 * grp + 2 * h + j;
                    wpre[k][j] = (pok && u < H2) ? L.wu[(bp * a.KT + a.k0 + k) * H2 + u] : 0.f;
                }
        };
        auto wu_put = [&](int grp) {
#pragma unroll
            for (int k = 0; k < KC; ++k)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    float x = wpre[k][j];
                    if (a.logits) x = (pok && 4 * grp + 2 * h + j < H2) ? __expf(x - wm[k]) * wil[k] : 0.f;
                    wus[k * 128 + (2 * h + j) * 32 + pl] = x;
                }
            __builtin_amdgcn_wave_barrier();
        };
        if constexpr (WT) {
            wu_load(ua >> 2);
#pragma unroll
            for (int k = 0; k < KC; ++k) {
                wil[k] = 1.f / wil[k];
                const float il = 1.f / vil[k];
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    rv[k][r] = 0.f;
                    if (a.logits) wvr[k][r] = (pok && 32 * vc + vmap(r, h) < W2) ? __expf(wvr[k][r] - vm[k]) * il : 0.f;
                }
            }
            wu_put(ua >> 2);
            wu_load((ua >> 2) + 1);
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                vmax[r] = -INFINITY;
                vsum[r] = 0.f;
                vidx[r] = 0;
            }
        }
        // kept in the accumulator half of the register file, from where the matrix instructions read them; the other
        // half is for what the vector instructions work on
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            if (PIPE) asm volatile("" : "+a"(fh[s]));
            if (PIPE) asm volatile("" : "+a"(fl[s]));
        }
        float *part = L.part + (((size_t)bc * H2) * Q) * N1p + pt * TPX + 32 * wave + pl;
        // What a lane holds of a row, scaled back, goes into the running state and into out_u's parts:
        // begin(u), the registers one by one, finish(u).
        float red[KC], redw[KC], red_m = 0.f, red_s = 0.f;
        int red_i = 0, red_u = 0;
        auto begin = [&](int u) {
            red_u = u;
            if constexpr (WT) {
#pragma unroll
                for (int k = 0; k < KC; ++k) {
                    redw[k] = wus[k * 128 + (u & 3) * 32 + pl];
                    red[k] = 0.f;
                }
            } else {
                red_m = -INFINITY;
                red_s = 0.f;
                red_i = 0;   // (a row without a value above -inf ends up with its first column)
            }
        };
        auto take = [&](auto edge, int r, float y) {
            if constexpr (WT) {
#pragma unroll
                for (int k = 0; k < KC; ++k) {
                    red[k] += y * wvr[k][r];
                    rv[k][r] += y * redw[k];
                    keep_here(rv[k][r]);
                }
            } else {
                red_s += y;
                vsum[r] += y;
                if constexpr (MODE == SPLIT_ARGMAX) vidx[r] = y > vmax[r] ? red_u : vidx[r];
                vmax[r] = maxnum(vmax[r], y);
                const float z = (edge && vmap(r, 0) >= cols) ? -INFINITY : y;
                if constexpr (MODE == SPLIT_ARGMAX) red_i = z > red_m ? vmap(r, 0) : red_i;
                red_m = maxnum(red_m, z);
                keep_here(vmax[r]);
                keep_here(vsum[r]);
                if constexpr (MODE == SPLIT_ARGMAX) keep_here(vidx[r]);
            }
        };
        // What finish() leaves in `pend` is stored by flush(), at the beginning of the next step: the barrier at the end of
        // a step waits for all memory operations of the wave, and a store issued just before it holds up the workgroup for
        // as long as it takes to reach the L2 (most of 2 us a step at B=2, 55x128).
        float pend[KC > 2 ? 2 : MODE == SPLIT_ARGMAX ? 2 : 1];
        auto finish = [&] {
            if constexpr (WT) {
                float sk[KC];
#pragma unroll
                for (int k = 0; k < KC; ++k) {
                    float lo, hi;
                    wave_halves(red[k], lo, hi);
                    sk[k] = lo + hi;
                }
#pragma unroll
                for (int k = 0; k < KC; k += 2)   // lanes of half 0 store the even channels, of half 1 the odd ones
                    pend[k / 2] = k + 1 < KC ? (h ? sk[k + 1 < KC ? k + 1 : k] : sk[k]) : sk[k];
                if ((red_u & 3) == 3) {
                    __builtin_amdgcn_wave_barrier();
                    wu_put((red_u >> 2) + 1);
                }
            } else {
                float m_lo, m_hi, s_lo, s_hi;
                wave_halves(red_m, m_lo, m_hi);
                wave_halves(red_s, s_lo, s_hi);
                if constexpr (MODE == SPLIT_ARGMAX) {
                    red_i += 32 * vc + 4 * h;
                    float i_lo, i_hi;
                    wave_halves(__int_as_float(red_i), i_lo, i_hi);
                    const bool take_hi = m_hi > m_lo || (m_hi == m_lo && __float_as_int(i_hi) < __float_as_int(i_lo));
                    pend[0] = h ? (take_hi ? i_hi : i_lo) : (take_hi ? m_hi : m_lo);
                    pend[Q - 2] = s_lo + s_hi;
                } else {
                    pend[0] = h ? s_lo + s_hi : maxnum(m_lo, m_hi);
                }
            }
        };
        auto flush = [&] {
            float *dst = part + (size_t)red_u * Q * N1p;
            if constexpr (WT) {
#pragma unroll
                for (int k = 0; k < KC; k += 2)
                    if (k + 1 < KC || h == 0) dst[(k + (k + 1 < KC ? h : 0)) * N1p] = pend[k / 2];
                if ((red_u & 3) == 3) wu_load((red_u >> 2) + 2);
            } else if constexpr (MODE == SPLIT_ARGMAX) {
                dst[h ? 2 * N1p : 0] = pend[0];
                if (h == 0) dst[N1p] = pend[1];
            } else {
                dst[h ? N1p : 0] = pend[0];
            }
        };
        // The products of a row block; `beside(s)` is what the vector units do beside the matrix work of channel step s.
        // Operands are read two channel steps before they are used.  The order is fixed here: left to itself the
        // compiler either reads everything at once (and spills) or waits for every read, and puts the vector work last.
        // Row `next` is requested into row block nbuf a KB at a time between the matrix instructions (all requests at once
        // hold the wave up for 700 cycles; behind a piece's last row they fetch what follows it in the scratch, which is
        // not used).  The factors that scale row u back are in `fac` at the end and the block's mark in `mark`.
        v4f fac[4];
        int mark = 0;
        auto multiply = [&](int next, int buf, int nbuf, auto beside) {
            const char *blk = reinterpret_cast<const char *>(smem + buf * BF) + lane * 16;
            const float *tail = smem + buf * BF + 2 * NK * 256;
            v16f acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, cross = acc;
            v8h ah[3], al[3];
            auto fetch = [&](int t) {   // step t: channel step t mod NK; the second pass over them needs no low halves
                ah[t % 3] = *reinterpret_cast<const v8h *>(blk + (t % NK) * 2048);
                if (t < NK) al[t % 3] = *reinterpret_cast<const v8h *>(blk + t * 2048 + 1024);
            };
            constexpr int NT = TWO_ACC ? NK : 2 * NK;
            fetch(0);
            fetch(1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (t + 2 < NT) fetch(t + 2);
                if (t == NT - 2) {
#pragma unroll
                    for (int g4 = 0; g4 < 4; ++g4) fac[g4] = *reinterpret_cast<const v4f *>(tail + 8 * g4 + 4 * h);
                    mark = __float_as_int(tail[MARK]);
                }
                if (t == NK) acc = cross * LOW_UNIT;
                if (TWO_ACC || t >= NK) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[t % 3], fh[t % NK], acc, 0, 0, 0);
                if (t < NDMA) dma(next, nbuf, t);
                if (t < NK) {
                    cross = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[t % 3], fh[t], cross, 0, 0, 0);
                    cross = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[t % 3], fl[t], cross, 0, 0, 0);
                }
                beside(t);
                __builtin_amdgcn_sched_barrier(0);
            }
            return TWO_ACC ? acc + cross * LOW_UNIT : acc;
        };
        constexpr int PER = 16 / NK;   // accumulator registers reduced beside one channel step
        auto multiply_fp32 = [&](int u, float (&x)[16]) {
            const int v = 32 * vc + pl, first = (a.pt0 + pt) * TPX;
            const v16f acc = products_fp32(a.f1 + ((size_t)b * N1 + first) * C, (unsigned)min(TPX, N1 - first) * C * 4u,
                                           pok ? (unsigned)(32 * wave + pl) * C * 4u : OOB, L.f2 + ((size_t)b * H2 + u) * W2 * C,
                                           (unsigned)W2 * C * 4u, v < W2 ? (unsigned)v * C * 4u : OOB, C, cols);
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = acc[r];
        };
        // (both factors here, so that the running state is in the units of the results: a state that `back` is applied to at
        // the end overflows for products of marked blocks and for weights that the results themselves have room for)
        auto products = [&](const v16f &acc, int u, float (&x)[16]) {
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * g4 + e] = acc[4 * g4 + e] * fac[g4][e] * back;
            if (fbad || __builtin_amdgcn_readfirstlane(mark) != 0) multiply_fp32(u, x);
        };
        __syncthreads();
        float x[16];
        auto nothing = [](int) {};
        // (edge: the chunk has columns beyond the image, which the maxima over a row leave out)
        auto sweep = [&](auto edge) {
            if constexpr (PIPE) {
                // Rows are requested two steps ahead, into three blocks: a step (1600 cycles and more) is too short for
                // what the last requests of the step before take.  At the end of a step all but this step's requests
                // have to be there: of the wave's outstanding memory operations the latest 2 NK / 4 are among those.
                auto step_end = [] { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NK / 2) : "memory"); };
                products(multiply(ua + 2, 0, 2, nothing), ua, x);
                step_end();
                int buf = 1;
                for (int u = ua + 1; u < ub; ++u) {
                    const int nbuf = buf == 0 ? 2 : buf - 1;   // the block of row u - 1, which every wave is done with
                    if (u > ua + 1) flush();
                    begin(u - 1);
                    const v16f acc = multiply(u + 2, buf, nbuf, [&](int s) {
#pragma unroll
                        for (int e = 0; e < PER; ++e) take(edge, PER * s + e, x[PER * s + e]);
                    });
                    finish();
                    products(acc, u, x);
                    step_end();
                    buf = buf == 2 ? 0 : buf + 1;
                }
                if (ub > ua + 1) flush();
                begin(ub - 1);
#pragma unroll
                for (int r = 0; r < 16; ++r) take(edge, r, x[r]);
                finish();
                flush();
            } else {
                for (int u = ua; u < ub; ++u) {
                    const int buf = (u - ua) & 1;
                    if (u > ua) flush();
                    products(multiply(u + 1, buf, buf ^ 1, nothing), u, x);
                    begin(u);
#pragma unroll
                    for (int r = 0; r < 16; ++r) take(edge, r, x[r]);
                    finish();
                    __syncthreads();
                }
                flush();
            }
        };
        if (WT || 32 * vc + 32 <= W2) sweep(std::false_type{});
        else sweep(std::true_type{});
        // the columns of this piece
        const bool whole = ua == 0 && ub == H2;
        float *slot = a.slots + (size_t)(2 * wg + (ua > 0 ? 0 : 1)) * Q * 4096 + (wave * 4 * 64 + lane) * 4;
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                v4f x;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (WT) x[e] = rv[q][4 * g4 + e];
                    else x[e] = q == 0 ? vmax[4 * g4 + e] : q == 1 ? vsum[4 * g4 + e] : __int_as_float(vidx[4 * g4 + e]);
                }
                const int v = 32 * vc + vmap(4 * g4, h);
                if (!whole) *reinterpret_cast<v4f *>(slot + (q * 16 + g4) * 256) = x;
                else if (pok && v < W2) store_v<MODE>(a, L, bp, q, v, x);
            }
    }
}

template <int MODE, int KC>
int launch_sweep(const SplitArgs &a, int nk, hipStream_t s) {
    const size_t lds = (pipelined(MODE, KC, nk) ? 3 : 2) * (size_t)block_bytes(nk) + (MODE == SPLIT_WEIGHTED ? 4 * KC * 128 * sizeof(float) : 0);
    auto k = nk == 4 ? split_sweep_kernel<MODE, KC, 4> : nk == 8 ? split_sweep_kernel<MODE, KC, 8> : split_sweep_kernel<MODE, KC, 16>;
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return sepcorr_set_error(SEPCORR_ELAUNCH, "sepcorr: cannot reserve the sweep's LDS");
    hipLaunchKernelGGL(k, dim3(a.G), dim3(256), lds, s, a);
    return 0;
}
}  // namespace

#define SPLIT_LAUNCHER(name, MODE, KC) \
    int name(const SplitArgs &a, int nk, hipStream_t s) { return launch_sweep<MODE, KC>(a, nk, s); }
int split_launch_maxavg(const SplitArgs &, int, hipStream_t);
int split_launch_argmax(const SplitArgs &, int, hipStream_t);
int split_launch_w1(const SplitArgs &, int, hipStream_t);
int split_launch_w2(const SplitArgs &, int, hipStream_t);
int split_launch_w3(const SplitArgs &, int, hipStream_t);
int split_launch_w4(const SplitArgs &, int, hipStream_t);
#if SPLIT_IN_PART(1)
SPLIT_LAUNCHER(split_launch_maxavg, SPLIT_MAXAVG, 1)
#endif
#if SPLIT_IN_PART(2)
SPLIT_LAUNCHER(split_launch_argmax, SPLIT_ARGMAX, 1)
#endif
#if SPLIT_IN_PART(3)
SPLIT_LAUNCHER(split_launch_w1, SPLIT_WEIGHTED, 1)
#endif
#if SPLIT_IN_PART(4)
SPLIT_LAUNCHER(split_launch_w2, SPLIT_WEIGHTED, 2)
#endif
#if SPLIT_IN_PART(5)
SPLIT_LAUNCHER(split_launch_w3, SPLIT_WEIGHTED, 3)
#endif
#if SPLIT_IN_PART(6)
SPLIT_LAUNCHER(split_launch_w4, SPLIT_WEIGHTED, 4)
#endif

#if SPLIT_IN_PART(0)
namespace {
constexpr size_t kPartLimit = (size_t)96 << 20;   // out_u's parts of one launch: what the 256 MB cache still holds
constexpr int kMinChannels = 32;
constexpr int kPlaces = 256;                      // compute units

struct SplitPlan {
    bool ok;
    int nk, q, npt, slabs, npt_slab;
    size_t planes, part, slots;
    size_t bytes() const { return planes + part + slots; }
};
size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
int places(int mode, int kc, int nk) { return pipelined(mode, kc, nk) ? kPlaces : 2 * kPlaces; }

SplitPlan plan(int B, int N1, const int *h2, const int *w2, int nlev, int C, int mode, int kc) {
    SplitPlan p = {};
    if (C < kMinChannels || C > 256 || nlev < 1 || nlev > 4) return p;
    p.nk = C <= 64 ? 4 : C <= 128 ? 8 : 16;
    p.q = mode == SPLIT_WEIGHTED ? kc : mode == SPLIT_ARGMAX ? 3 : 2;
    p.npt = (N1 + TPX - 1) / TPX;
    long blocks = 0;
    double pairs = 0;
    for (int l = 0; l < nlev; ++l) {
        blocks += (long)B * ((w2[l] + 31) / 32) * h2[l];
        pairs += (double)B * N1 * h2[l] * w2[l];
    }
    const size_t per_pt = (size_t)blocks * p.q * TPX * sizeof(float);
    long fit = (long)(kPartLimit / per_pt);
    if (fit < 1) fit = 1;
    p.slabs = (int)((p.npt + fit - 1) / fit);
    p.npt_slab = (p.npt + p.slabs - 1) / p.slabs;
    const long steps = blocks * p.npt_slab;
    // The three launches and the hand-over through scratch take 26 us at the least, the fp32 sweep two launches and its
    // matrix work.  This sweep's time over the fp32 sweep's, three shapes each, at pairs (C + 64) = 0.4e9, 0.8e9, 1.3e9:
    // max/average C=32 0.84-1.06, 0.76-0.88, 0.73-0.85; C=128 0.64-0.84, 0.72-0.75, 0.57-0.65; C=256 0.89-1.12, 0.67-0.81,
    // 0.65-0.75; four channels C=32 0.98-1.08, 0.83-0.92, 0.82-1.01; C=128 0.70-0.84, 0.80-0.86, 0.65-0.76; C=256
    // 0.97-1.24, 0.76-0.94, 0.81-0.87; four levels are 0.3 to 0.9 from 0.7e9 on.  Above the line, in 402 shapes of up to 64
    // channels with two to four weight channels the median is 0.66; slower by more than 2 % are three or four channels
    // of some pyramids (16 of 190, at the most 1.21: B=12, 29x41, C=32, K=3: pieces of few rows) and, on a single level, three
    // channels at C=32 (0.89 to 1.13, on average 1.0): these stay with the fp32 sweep.
    if (pairs * (C + 64) < 1e9) return p;
    if (mode == SPLIT_WEIGHTED && kc == 3 && C % 32 == 0 && C < 64 && nlev == 1) return p;
    for (int l = 0; l < nlev; ++l)
        if ((size_t)h2[l] * block_bytes(p.nk) >= (1u << 30)) return p;
    if (steps > (1L << 30) || blocks > (1L << 24)) return p;
    p.planes = align256((size_t)B * ((N1 + 31) / 32) * block_bytes(p.nk));
    for (int l = 0; l < nlev; ++l) p.planes += align256((size_t)B * ((w2[l] + 31) / 32) * h2[l] * block_bytes(p.nk));
    p.part = align256(per_pt * p.npt_slab) + 4 * 256;
    p.slots = (size_t)2 * places(mode, kc, p.nk) * p.q * 4096 * sizeof(float);
    p.ok = true;
    return p;
}
}  // namespace

size_t sepcorr_split_sweep_bytes(int B, int N1, const int *h2, const int *w2, int nlev, int C, int mode, int kc) {
    const SplitPlan p = plan(B, N1, h2, w2, nlev, C, mode, kc);
    return p.ok ? p.bytes() : 0;
}

int split_sweep(int mode, int kc, SplitArgs a, void *ws, size_t ws_bytes, hipStream_t s) {
    int h2[4], w2[4];
    for (int l = 0; l < a.nlev && l < 4; ++l) { h2[l] = a.lev[l].H2; w2[l] = a.lev[l].W2; }
    const SplitPlan p = plan(a.B, a.N1, h2, w2, a.nlev, a.C, mode, kc);
    if (!p.ok || ws == nullptr || ws_bytes < p.bytes()) return 1;
    char *base = static_cast<char *>(ws);
    int blocks = 0;
    for (int l = 0; l < a.nlev; ++l) {
        SplitLevel &L = a.lev[l];
        L.nvc = (L.W2 + 31) / 32;
        L.block0 = blocks;
        L.planes = base;
        base += align256((size_t)a.B * L.nvc * L.H2 * block_bytes(p.nk));
        blocks += a.B * L.nvc * L.H2;
    }
    a.blocks = blocks;
    a.f1_planes = base;
    base += align256((size_t)a.B * ((a.N1 + 31) / 32) * block_bytes(p.nk));
    float *part = reinterpret_cast<float *>(base);
    a.slots = reinterpret_cast<float *>(base + p.part);
    auto pk = p.nk == 4 ? split_prepare_kernel<4> : p.nk == 8 ? split_prepare_kernel<8> : split_prepare_kernel<16>;
    hipLaunchKernelGGL(pk, dim3(blocks + a.B * ((a.N1 + 31) / 32)), dim3(256), 0, s, a);
    for (a.pt0 = 0; a.pt0 < p.npt; a.pt0 += p.npt_slab) {
        a.npt = p.npt - a.pt0 < p.npt_slab ? p.npt - a.pt0 : p.npt_slab;
        a.tiles = 0; a.steps = 0; a.fin_blocks = 0;
        float *pp = part;
        for (int l = 0; l < a.nlev; ++l) {
            SplitLevel &L = a.lev[l];
            L.tile0 = a.tiles; L.step0 = a.steps; L.fin0 = a.fin_blocks;
            L.part = pp;
            const int t = a.B * L.nvc * a.npt;
            a.tiles += t;
            a.steps += t * L.H2;
            a.fin_blocks += a.B * 2 * a.npt * ((L.H2 + 31) / 32);
            pp += ((size_t)a.B * L.nvc * L.H2 * p.q * a.npt * TPX + 63) & ~(size_t)63;
        }
        const int G = places(mode, kc, p.nk);
        a.G = a.steps < G ? a.steps : G;
        int rc;
        if (mode == SPLIT_MAXAVG) rc = split_launch_maxavg(a, p.nk, s);
        else if (mode == SPLIT_ARGMAX) rc = split_launch_argmax(a, p.nk, s);
        else rc = kc == 1 ? split_launch_w1(a, p.nk, s) : kc == 2 ? split_launch_w2(a, p.nk, s)
                  : kc == 3 ? split_launch_w3(a, p.nk, s) : split_launch_w4(a, p.nk, s);
        if (rc) return rc;
        auto fk = mode == SPLIT_MAXAVG ? split_finish_kernel<SPLIT_MAXAVG, 2> : mode == SPLIT_ARGMAX ? split_finish_kernel<SPLIT_ARGMAX, 3>
                  : kc == 1 ? split_finish_kernel<SPLIT_WEIGHTED, 1> : kc == 2 ? split_finish_kernel<SPLIT_WEIGHTED, 2>
                  : kc == 3 ? split_finish_kernel<SPLIT_WEIGHTED, 3> : split_finish_kernel<SPLIT_WEIGHTED, 4>;
        hipLaunchKernelGGL(fk, dim3(4 * a.tiles + a.fin_blocks), dim3(256), 0, s, a);
    }
    if (hipGetLastError() != hipSuccess) return sepcorr_set_error(SEPCORR_ELAUNCH, "sepcorr: split sweep: launch failed");
    return 0;
}
#endif
