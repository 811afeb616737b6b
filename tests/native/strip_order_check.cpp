// Host check of the broadphase's collider order (strips.h): how many pairs of tiles (64 consecutive colliders) have
// boxes that meet, for n bodies in a container and the same with some far away.  Usage: scene far [extremes], with
// the sample's bounds taken by rank as the kernel does, or its extremes.  Prints the pairs a tile.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "strips.h"

using namespace rp3dg;

static uint64_t st = 88172645463325252ull;
static float rnd() { st ^= st << 13; st ^= st >> 7; st ^= st << 17; return (float)((st >> 40) * (1.0 / 16777216.0)); }

struct P3 {
    float x[3];
};

int main(int argc, char** argv) {
    const char* scene = argv[1];
    const int far = atoi(argv[2]), n = 20000;
    const bool extremes = argc > 3;
    std::vector<P3> c(n);
    for (P3& p : c) {
        if (!strcmp(scene, "heap")) p = {{100.f * rnd(), 100.f * rnd(), 12.f * rnd()}};
        else if (!strcmp(scene, "row")) p = {{4000.f * rnd(), 6.f * rnd(), 8.f * rnd()}};
        else {   // a mound: dense in the middle
            const float r = 60.f * rnd() * rnd(), a = 6.2831853f * rnd();
            p = {{r * cosf(a), r * sinf(a), 20.f * rnd() * (1.f - r / 60.f)}};
        }
    }
    for (int i = 0; i < far; i++) {   // fallen out, for a while to a long time
        P3& p = c[(int)(n * rnd())];
        p.x[2] -= 10.f * expf(12.f * rnd());
    }
    std::vector<int> sample;
    const size_t m = std::min(n, kOrderSamples);
    for (size_t k = 0; k < m; k++) {
        const size_t lo = k * n / m, hi = (k + 1) * n / m;
        sample.push_back((int)(lo + (size_t)((uint32_t)k * 0x9E3779B1u >> 8) % (hi - lo)));
    }
    float lo[3], hi[3];
    for (int k = 0; k < 3; k++) {
        std::vector<float> v;
        for (int i : sample) v.push_back(c[i].x[k]);
        if (extremes) {
            v.clear();
            for (const P3& p : c) v.push_back(p.x[k]);
        }
        std::sort(v.begin(), v.end());
        const size_t cut = extremes ? 0 : v.size() / kOrderCut;
        lo[k] = v[cut];
        hi[k] = v[v.size() - 1 - cut];
    }
    const StripOrder o = strip_order(lo, hi, (float)n);
    std::vector<std::pair<uint32_t, int>> keys;
    for (int i = 0; i < n; i++) keys.push_back({strip_key(o, c[i].x[o.axis[0]], c[i].x[o.axis[1]]), i});
    std::stable_sort(keys.begin(), keys.end());
    for (const auto& k : keys)
        if (k.first >> 24) { printf("-1\n"); return 0; }   // more than 24 bits
    struct Box {
        float mn[3], mx[3];
    };
    std::vector<Box> tiles;
    for (int i = 0; i < n; i++) {
        if (i % 64 == 0) tiles.push_back({{INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}});
        for (int k = 0; k < 3; k++) {
            Box& b = tiles.back();
            b.mn[k] = fminf(b.mn[k], c[keys[i].second].x[k] - 0.7f);
            b.mx[k] = fmaxf(b.mx[k], c[keys[i].second].x[k] + 0.7f);
        }
    }
    long meet = 0, most = 0;
    for (const Box& a : tiles) {
        long w = 0;
        for (const Box& b : tiles) {
            bool hit = true;
            for (int k = 0; k < 3; k++) hit = hit && a.mn[k] <= b.mx[k] && b.mn[k] <= a.mx[k];
            w += hit;
        }
        meet += w;
        most = std::max(most, w);
    }
    printf("%.2f %ld strips %d\n", (double)meet / tiles.size(), most, o.strips);
    return 0;
}
