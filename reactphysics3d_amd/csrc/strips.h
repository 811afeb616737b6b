// Order of the colliders in the tile broadphase: strips across the second largest extent of the moving colliders'
// centres, run along the largest, every other strip backwards; 8 bits of strip, 16 of position, the world id above
// them.  A strip is as wide as 64 colliders of a world of mean density are long, so a run of 64 is about square,
// and as consecutive keys are neighbours throughout, no run has a box larger than its neighbours'.  (On a curve
// in three dimensions, Morton or Hilbert, the runs across its larger turns meet a good part of the scene,
// and the longest workgroup sets the time: bp_pairs took 1238 and 650 us for 65,536 bodies there, 70 on strips.)
//
// The extents are those of a sample without its outer sixteenths, so that a few bodies far from the others (fallen
// out of the scene) do not stretch them.  With the extremes' extents one body 1 km down left two strips for the
// others and far ones left one, and every tile met every other: bp_pairs of 65,536 bodies took 275 us, and 3220 with
// 50 of them 1 to 1000 km down; 68 and 67 with these.
#pragma once

#include "rp3d_internal.h"

namespace rp3dg {

constexpr int kOrderSamples = 256;   // moving colliders whose centres give the extents
constexpr int kOrderCut = 16;        // a 16th of the sample beyond each bound
constexpr int kOuterStrips = 32;     // strips beyond each end of the extent, of doubling width
constexpr int kInnerStrips = (1 << kStripBits) - 2 * kOuterStrips;
constexpr float kOuterPositions = 8192.f;   // positions beyond each end, closer together the farther out

struct StripOrder {
    int axis[2];      // across the strips, along them
    float lo[2], scale[2];
    int strips;
};

// lo, hi: a 16th of the sample's centres lies below / above; world_colliders: of a mean world
__host__ __device__ inline StripOrder strip_order(const float lo[3], const float hi[3], float world_colliders) {
    float l[3], e[3];
    for (int k = 0; k < 3; k++) {   // the whole extent, if the centres are spread evenly
        const float d = hi[k] - lo[k];
        e[k] = d > 0.f && d < 1e30f ? d * ((float)kOrderCut / (kOrderCut - 2)) : 0.f;   // (no moving collider: 0)
        l[k] = lo[k] - e[k] / kOrderCut;
    }
    int a = 0;
    for (int k = 1; k < 3; k++) a = e[k] > e[a] ? k : a;
    int b = a == 0 ? 1 : 0;
    for (int k = 0; k < 3; k++) b = k != a && e[k] > e[b] ? k : b;
    const float width = 8.0f * sqrtf(e[a] * (e[b] / world_colliders));
    StripOrder o;
    o.strips = width > 0.f ? (int)fminf(fmaxf(ceilf(e[b] / width), 1.f), (float)kInnerStrips) : 1;
    o.axis[0] = b;
    o.axis[1] = a;
    o.lo[0] = l[b];
    o.lo[1] = l[a];
    o.scale[0] = e[b] > 0.f ? (float)o.strips / e[b] : 0.f;
    o.scale[1] = e[a] > 0.f ? 1.0f / e[a] : 0.f;
    return o;
}

// Strip and position of a centre with the coordinates b across the strips and a along them.
__host__ __device__ inline uint32_t strip_key(const StripOrder& o, float b, float a) {
    const float x = (b - o.lo[0]) * o.scale[0], last = (float)o.strips;
    // within two strips of an end, its outermost strip (the sample's bounds are not the scene's to a strip, and a
    // sliver of a strip would make long tiles); then strips of doubling width
    const float far = 0.5f * (x < 0.f ? -x : x - last);
    const int out = far >= 1.0f ? 1 + (int)(fbits_of(far) >> 23) - 127 : 0;
    const int in = (int)fminf(fmaxf(x, 0.f), last - 1.f), w = out < kOuterStrips ? out : kOuterStrips;
    const int u = kOuterStrips + (x < 0.f ? -w : in + w);
    const float v = (a - o.lo[1]) * o.scale[1];
    float p = kOuterPositions + v * (65535.f - 2.f * kOuterPositions);
    if (v < 0.f) p = kOuterPositions / (1.0f - v);
    if (v > 1.f) p = 65535.f - kOuterPositions / v;
    const uint32_t strip = (uint32_t)u, pos = (uint32_t)fminf(fmaxf(p, 0.f), 65535.f);
    return strip << 16 | (strip & 1u ? 65535u - pos : pos);
}

}  // namespace rp3dg
