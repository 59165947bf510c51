// Feature gradients (d_f1, d_f2) of the compression and of the combined backward with every fp32 operand split into two
// 16-bit halves (split_grad.hip): what sepcorr.hip hands over.  Internal to libsepcorr.
#ifndef SEPCORR_SPLIT_GRAD_H
#define SEPCORR_SPLIT_GRAD_H
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

struct VField {
    const float *src;      // a tensor of `rows` rows of W2 per pixel of image 1
    int rows, row;         // the field's among them
};
struct GradArgs {
    const float *f1, *f2;
    const float *a_u, *a_v, *g_cu, *g_cv;     // (B,N1,KT,W2), (B,N1,KT,H2), (B,N1,KT,H2), (B,N1,KT,W2)
    const int *am_u, *am_v;                   // with the max/average terms: (B,N1,H2), (B,N1,W2)
    const float *g_u, *g_v;                   //                             (B,N1,2,H2), (B,N1,2,W2)
    float *d1, *d2;                           // (B,N1,C), (B,H2 W2,C)
    int B, N1, H2, W2, C;
    int KT, k0;                               // weight channels in all, first one of this launch
    int add1, add2;                           // add to d1 / d2 instead of overwriting
    // filled by split_grad()
    int ncb, nvc;                             // channel blocks of 32 (2, 4, 8), column chunks of 32
    int H2p, N1p;                             // rows padded to 8, pixels padded to 128
    int npx;                                  // pixel tiles of 16 that hold pixels
    int direct;                               // the v-indexed weights are read where they are, not from pv
    float *pv;                                // [B][nvc][N1p / 16][field][8 groups of columns][16 pixels][4 columns]
    float *pu;                                // [B][H2p][N1p][u-indexed fields]
    float *pscale;                            // [B][N1p] power of two that dL/dS of a pixel is multiplied by in d_f1
    int *block_bad;                           // whether one of 16 pixels has none
    float *bound_v, *bound_u;                 // [B][nvc][N1p / 16][bounds][32], [B][N1p / 16][bounds][H2p]: see grad_prepare_kernel
    unsigned *pmax;                           // [2][B][slab][256] largest |f1|, |f2| of a channel
    int *cback;                               // [2][B][256] the power of two that takes a channel's factor back
    unsigned *count;                          // small values of f1, of f2; whether anything else is unsuitable
    char *f1h, *f2h;                          // halves of f1 [B][npx], of f2 [B][nvc][H2]
    VField vfield[11];                        // the v-indexed weights
    GradArgs *self;                           // these arguments, on the device
    float *slots;
    int G1, G2;                               // workgroups of the two contractions
};

// Below this many pairs of pixels times (channels + 64) split_grad() takes nothing.
#define SPLIT_GRAD_LEAST 2.5e8
// From how many of them on it runs.  It is five or six launches, three of them over the operands, against two to five; the fp32
// kernels it replaces make a pass of their own for the max/average terms beside one or three weight channels, two for four in rows
// above 128, and take longer where rows are no multiple of 4 and then most for a small second image (they have few workgroups).
// Time over theirs in 37 000 shapes of 2.5e8 to 4e9, C 32 to 256, just below and just above the line (median / largest but 5 %):
//   with the max/average terms, one or three channels: 0.75 / 1.00 at 2.5e8, others than multiples of 4 0.53 / 0.66; with fewer than
//     8 tiles of d_f2, hundreds of pieces each, 0.85 / 1.20, and at 4e8 0.74 / 0.98
//   two or four: rows of a multiple of 4, 2e9: 0.96 / 1.19 and 0.85 / 1.01; others, 4.5e8: 0.77 / 1.04 and 0.72 / 0.95, small second
//     images 0.61 / 0.93 at 2.5e8
//   alone: rows of a multiple of 4, 2e9: 0.96 / 1.13 and 0.90 / 1.03; others, 7e8: 0.85 / 1.02 and 0.79 / 0.99, small second images
//     0.59 / 0.86 at 5e8
//   up to 64 channels the same ratios are reached at six tenths of that; rows above 128: 0.45 / 0.60 at all sizes.
inline double split_grad_line(bool both, int K, int B, int N1, int H2, int W2, int C) {
    const bool few = (long)B * ((H2 + 7) / 8) * ((W2 + 31) / 32) < 8, small = 12L * H2 * W2 <= N1;
    double line;
    if (W2 > 128) line = both ? SPLIT_GRAD_LEAST : 5e8;
    else if (both && (K == 1 || K == 3)) line = W2 % 4 == 0 && few ? 4e8 : SPLIT_GRAD_LEAST;
    else if (W2 % 4 == 0) line = 2e9;
    else if (small) line = both ? SPLIT_GRAD_LEAST : 5e8;
    else line = both ? 4.5e8 : 7e8;
    return C > 64 ? line : 0.6 * line;
}
// Scratch split_grad() wants for these sizes, whatever the number of channels, 0 where it does not take them.
size_t split_grad_bytes(int B, int N1, int H2, int W2, int C);
// Whether split_grad() takes a call with these arguments and this much scratch.
bool split_grad_fits(int both, int kc, const GradArgs &a, size_t ws_bytes);
// Runs both contractions, with the max/average terms if `both`; a negative SEPCORR_ code on error.  kc: 1 to 4 weight channels.
int split_grad(int both, int kc, GradArgs a, void *ws, size_t ws_bytes, hipStream_t s);
#endif
