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

int main() {
    printf("lds %d\n", lds_violations());
    return 0;
}
