"""How the split feature gradients deal steps out to workgroups (csrc/split_grad_deal.h), walked on the host.

The program below goes through the pieces of every workgroup in the order in which the contractions do and notes what
each leaves in its slot; then it goes through the tiles as the finishing kernel does.  Every step of every tile has to be
in the result exactly once, and no slot may hold two pieces.
"""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "separableflowthesis_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "split_grad_deal.h"

struct Held { int tile = -1, begin = 0, end = 0; };

static int walk(int tiles, int spt, int places) {
    const long T = (long)tiles * spt;
    const int G = (int)(T < places ? T : places);
    std::vector<Held> slots(slots_of(tiles, G));
    std::vector<char> out(tiles, 0);
    for (int wg = 0; wg < G; ++wg) {
        const int g0 = (int)first_step(wg, G, T), g1 = (int)first_step(wg + 1, G, T);
        for (int g = g0; g < g1;) {
            const int tile = g / spt;
            const Piece p = piece_of(tile, g0, g1, spt);
            if (p.begin != g - tile * spt || p.end <= p.begin) return printf("piece of %d %d in %d\n", tiles, spt, wg), 1;
            const int s = slot_of(wg, tile, p.begin > 0, tiles, G);
            if (s < 0 || s >= (int)slots.size()) return printf("slot %d of %d tiles of %d steps\n", s, tiles, spt), 1;
            if (slots[s].tile >= 0) return printf("%d tiles of %d steps: two pieces in slot %d\n", tiles, spt, s), 1;
            if (p.whole(spt)) out[tile]++;          // (passes through the slot)
            else slots[s] = Held{tile, p.begin, p.end};
            g = tile * spt + p.end;
        }
    }
    for (int tile = 0; tile < tiles; ++tile) {
        const long t0 = (long)tile * spt;
        int w0, w1, at = 0;
        pieces_of(t0, t0 + spt, G, T, w0, w1);
        if (w0 == w1) at = out[tile] == 1 ? spt : -1;
        else
            for (int w = w0; w <= w1 && at >= 0; ++w) {
                const Held &h = slots[slot_of(w, tile, first_step(w, G, T) > t0, tiles, G)];
                at = h.tile == tile && h.begin == at ? h.end : -1;
            }
        if (at != spt || out[tile] != (w0 == w1)) return printf("%d tiles of %d steps: tile %d is not whole\n", tiles, spt, tile), 1;
    }
    return 0;
}

int main() {
    const int steps[] = {1, 2, 7, FLUSH - 1, FLUSH, FLUSH + 1, 2 * FLUSH, 2 * FLUSH + 1, 220, 440, 1020};
    for (int spt : steps) {
        for (int tiles = 1; tiles <= 700; ++tiles)
            if (walk(tiles, spt, 256)) return 1;
        for (int tiles : {767, 768, 769, 1023, 1024, 1025, 5000})
            if (walk(tiles, spt, 256)) return 1;
    }
    // (a few workgroups: every way in which a share begins and ends in tiles)
    for (int places = 1; places <= 9; ++places)
        for (int tiles = 1; tiles <= 30; ++tiles)
            for (int spt = 1; spt <= 12; ++spt)
                if (walk(tiles, spt, places)) return 1;
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++ to compile the walk with")
def test_every_step_of_every_tile_is_in_the_result_once(tmp_path):
    (tmp_path / "walk.cpp").write_text(PROGRAM)
    exe = tmp_path / "walk"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", CSRC, str(tmp_path / "walk.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
