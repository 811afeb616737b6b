// Host check of how the narrowphase launch shares out its LDS and its test lists (narrowphase.h).  Prints the
// number of violations.
#include <stdio.h>

#include <vector>

#include "narrowphase.h"

using namespace rp3dg;

// A workgroup's wavefronts may be in tests of different kinds at the same time: a thread's clip buffers lie in its
// wavefront's part, which is what the wavefront's mesh tests write, and no two threads share a word.
static int lds_violations() {
    int bad = 0;
    std::vector<int> owner(kNpWaveFloats * (kNpThreads / 64), -1);
    for (int t = 0; t < kNpThreads; t++)
        for (int b = 0; b < 2; b++)
            for (int i = 0; i < kBoxClip; i++)
                for (int c = 0; c < 3; c++) {
                    const int k = np_clip_lds(t, b, i, c), part = np_wave_lds(t);
                    if (k < part || k >= part + kNpWaveFloats || k >= (int)owner.size()) { bad++; continue; }
                    if (owner[k] >= 0) bad++;
                    owner[k] = t;
                }
    return bad;
}

// Every pair of a list is in one wavefront's share of one tile, and the grid for n pairs has a workgroup for every
// tile of any list up to n.
static void list_violations(int& shares, int& grid) {
    shares = grid = 0;
    for (int bin : {(int)ALGO_POLY_POLY, BIN_POLY_POLY_SEP, BIN_BOX, (int)ALGO_CONCAVE, (int)ALGO_SPHERE_SPHERE}) {
        std::vector<unsigned char> taken;
        for (int n = 0, most = 0; n < 300000; n += n < 20000 ? 1 : 611) {
            const int tiles = np_tiles(bin, n), p = np_wave_pairs(bin, n);
            most = tiles > most ? tiles : most;
            if (np_grid(bin, n) < most) grid++;
            if (p < 1 || p > 64) shares++;
            if (n > 1200 && n % 97) continue;
            taken.assign(n, 0);
            for (int t = 0; t < tiles; t++)
                for (int w = 0; w < kNpThreads / 64; w++)
                    for (int l = 0; l < p; l++) {
                        const int k = np_first_pair(bin, n, t, w) + l;
                        if (k < n) taken[k]++;
                    }
            for (int k = 0; k < n; k++) shares += taken[k] != 1;
        }
    }
}

int main() {
    int shares, grid;
    list_violations(shares, grid);
    printf("lds %d\nshares %d\ngrid %d\n", lds_violations(), shares, grid);
    return 0;
}
