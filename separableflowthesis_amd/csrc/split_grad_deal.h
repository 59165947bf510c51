// How split_grad.hip deals the steps of all tiles out to workgroups, and where a workgroup leaves what it has of a tile.
// Index functions only, without the GPU: a host program can walk them.
#ifndef SEPCORR_SPLIT_GRAD_DEAL_H
#define SEPCORR_SPLIT_GRAD_DEAL_H
#ifdef __HIPCC__
#define DEAL_FN __host__ __device__ __forceinline__
#else
#define DEAL_FN inline
#endif

// Steps whose sums the registers take before they are added to the piece's slot.  d_f1 / d_f2 at B=2, 55x128: 24 steps 1.69e-7
// / 2.5e-7, 813 us a backward call; 48 1.86e-7 / 3.2e-7, 740 us; 96 2.14e-7 / 4.3e-7 (before the signs of block_sign()).
constexpr int FLUSH = 48;

// First of the T steps that workgroup wg of G has.
DEAL_FN long first_step(long wg, int G, long T) { return wg * T / G; }

// What the workgroup with the steps [g0, g1) has of a tile, whose steps are [0, spt).
struct Piece {
    int begin, end;
    DEAL_FN bool whole(int spt) const { return begin == 0 && end == spt; }
};
DEAL_FN Piece piece_of(int tile, int g0, int g1, int spt) {
    Piece p = {g0 - tile * spt, g1 - tile * spt};
    if (p.begin < 0) p.begin = 0;
    if (p.end > spt) p.end = spt;
    return p;
}

// The workgroups [w0, w1] that hold the steps [t0, t1).
DEAL_FN void pieces_of(long t0, long t1, int G, long T, int &w0, int &w1) {
    w0 = (int)((t0 * G) / T);
    while (w0 > 0 && first_step(w0, G, T) > t0) --w0;
    while (first_step(w0 + 1, G, T) <= t0) ++w0;
    w1 = w0;
    while (first_step(w1 + 1, G, T) < t1) ++w1;
}

// Slot of the piece that workgroup wg has of a tile (it is not its first step there if `inside`).  With fewer tiles than
// workgroups every piece has its own.  Otherwise a workgroup has two: one for a tile that it joins, one for a tile that it
// begins.  A tile that it has whole it writes out itself, before it begins the next: that one only passes through the slot.
DEAL_FN int slot_of(int wg, int tile, bool inside, int tiles, int G) {
    return tiles < G ? wg + tile : 2 * wg + (inside ? 0 : 1);
}
DEAL_FN long slots_of(long tiles, int G) { return tiles < G ? G + tiles : 2L * G; }
#endif
