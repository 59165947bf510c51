// Forward-type sweeps with every fp32 operand split into two 16-bit halves (split_sweep.hip): what the launchers of
// sepcorr.hip hand over.  Internal to libsepcorr.
#ifndef SEPCORR_SPLIT_SWEEP_H
#define SEPCORR_SPLIT_SWEEP_H
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

enum { SPLIT_MAXAVG = 0, SPLIT_ARGMAX = 1, SPLIT_WEIGHTED = 2 };

struct SplitLevel {
    const float *f2, *wv, *wu;
    float *out_u, *out_v;
    int *am_u, *am_v;
    const float *st_wv, *st_wu, *z_ou, *st_ou, *dot_ou, *z_ov, *st_ov, *dot_ov;   // softmax inside
    int H2, W2;
    // filled by split_sweep()
    int nvc;            // column chunks of 32
    int block0;         // row blocks (image, chunk, row) of the levels before
    int tile0;          // tiles of the levels before
    int step0;          // steps of the levels before
    int fin0;           // output blocks of the levels before (split_finish_kernel)
    char *planes;       // row blocks of this level
    float *part;        // [B][nvc][H2][quantity][npt * 128]
};
struct SplitArgs {
    const float *f1;
    int B, N1, C;
    int KT, k0;         // weight channels in all, first one of this launch
    int logits, dlog;
    int nlev;
    SplitLevel lev[4];
    // filled by split_sweep()
    int pt0, npt;       // pixel tiles of 128 of this launch: [pt0, pt0 + npt)
    char *f1_planes;    // [B][ceil(N1 / 32)] blocks of image 1
    int tiles, steps, blocks, fin_blocks;
    int G;              // workgroups of the sweep
    float *slots;
};

// Scratch split_sweep() wants, 0 where it does not take the sizes.  kc: channels of one launch (0: max/average).  (C
// linkage: a host test holds the library's workspace queries against it.)
extern "C" size_t sepcorr_split_sweep_bytes(int B, int N1, const int *h2, const int *w2, int nlev, int C, int mode, int kc);
// Runs the sweep when the sizes suit it and ws_bytes suffice; returns 1 without launching anything otherwise, 0 when
// it was launched, a negative SEPCORR_ code on error.
int split_sweep(int mode, int kc, SplitArgs a, void *ws, size_t ws_bytes, hipStream_t s);
#endif
