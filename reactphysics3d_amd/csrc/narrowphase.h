// Kernel argument block of the narrowphase kernels.
#pragma once

#include "rp3d_internal.h"

namespace rp3dg {

// The triangle tests of one step's convex vs concave pairs, pair by pair in middle-phase order.
struct ConcaveTests {
    int* pair;                 // pair slot
    int* tri;                  // triangle id (mesh: triangle index; height field: HeightField::computeTriangleShapeId)
    uint32_t* lf;              // the triangle's LastFrameCollisionInfo after the test
    float4* lfaxis;
    int* hit;                  // NarrowPhaseInfo::isColliding
    int2* pts;                 // its contact points in the point pool (first, count)
    int cap;
    int* count;
};

// The triangles tested this step as hulls: test t's TriangleShape has vertices [3t, 3t+3) and faces
// [2t, 2t+2) (normal, opposite normal), over the six half-edges and face vertex lists that every triangle
// shares (PhysicsCommon.cpp initTriangleShapeHalfEdgeStructure; face_edge0 = each face's first half-edge).
struct TriArena {
    float4* verts;       // 3 per test slot
    float4* normals;     // 2 per test slot
    int* face_edge;      // 2 per test slot
    int* face_verts;     // 2 x 2 per test slot: (offset into vidx, 3)
    const int4* edges;   // 6 shared half-edges
    const int* vidx;     // 6 shared face vertex indices
    int face_edge0[2];
};

struct NpArgs {
    DevBodies B;
    DevColliders C;
    DevPairs P;                // pair table of this step
    DevPairs O;                // previous table: contact caches of surviving pairs (P.prev)
    const int* nb_pairs;
    const HullHeader* hulls;
    const float4* hull_verts;
    const float4* hull_normals;
    const int4* hull_edges;
    const int* hull_face_edge;
    const int* hull_face_verts;
    const int* hull_face_vidx;
    float persistent_threshold;
    float cos_similar;
    int* status;               // device status word (STATUS_*)
    // world queries (PhysicsWorld::testOverlap / testCollision, CD.cpp:1775-1896) run the same kernels:
    int query;                 // NP_STEP, NP_QUERY_ALL (both colliders world-query colliders) or NP_QUERY_BODIES
    int qbody1, qbody2;        // NP_QUERY_BODIES: pairs with body qbody1 (and qbody2 when >= 0)
    int report;                // NP_REPORT_NO_TRIGGER, NP_REPORT_ALL or NP_REPORT_NONE (reportContacts)
    int clip_prev;             // SATAlgorithm's clipWithPreviousAxisIfStillColliding (1 in steps, 0 in queries)
    int lf_update;             // processPotentialContacts updates wasColliding / isValid (0: overlap queries)
    // convex vs concave pairs (concave.cpp arenas; null pointers when the batch has no concave collider)
    const ConcaveInst* cinst;
    const float4* cverts;      // mesh vertices (unscaled)
    const int4* ctris;         // mesh triangles: vertex indices
    const float4* cnorm;       // scaled vertex normals of each concave collider
    const float4* cnodes;      // mesh AABB tree: (min, child0) (max, child1); a leaf has child0 = -1, child1 = triangle
    const float* cheights;     // height field samples
    const float4* hull_bounds; // local bounds of convex meshes (the convex shape's AABB in the concave space)
    ConcaveTests CT, CTo;      // this step's triangle tests, the previous step's (the pairs' last-frame infos)
    float4 *cp_nd, *cp_l1, *cp_l2;   // contact points of the tests: normal + depth, local points
    int cp_cap;
    int* cp_count;
    TriArena tri;
    int tail_base, tail_cap;   // tail entries of P: [tail_base, tail_base + tail_cap)
    int* tail_count;
};
constexpr int NP_STEP = 0, NP_QUERY_ALL = 1, NP_QUERY_BODIES = 2;
constexpr int NP_REPORT_NO_TRIGGER = 0, NP_REPORT_ALL = 1, NP_REPORT_NONE = 2;

// Test lists: one of the pair capacity for each bin but ALGO_NONE, whose slot has BIN_BOX's.
constexpr int kNpListSlots = kNpBins - 1;
__host__ __device__ constexpr int np_list_slot(int bin) { return bin < BIN_BOX ? bin : (bin == BIN_BOX ? 0 : bin - 1); }

__global__ void np_classify(NpArgs A, int* lists, int list_stride, int* counts);
// The lists np_pairs takes and the bins they hold, the longest tests first.
constexpr int kNpLists = kNpBins - 1;
constexpr int kNpOrder[kNpLists] = {ALGO_POLY_POLY, ALGO_CAPSULE_POLY, ALGO_SPHERE_POLY, BIN_BOX, BIN_POLY_POLY_SEP,
                                    BIN_CAPSULE_POLY_SEP, BIN_SPHERE_POLY_SEP, ALGO_CONCAVE, BIN_BOX_SEP,
                                    ALGO_CAPSULE_CAPSULE, ALGO_SPHERE_CAPSULE, ALGO_SPHERE_SPHERE};
// Pairs a wavefront takes of a list of n: a power of two, as few as keep kNpWaves wavefronts for the list.
// With few pairs the chip has SIMDs to spare, and a wavefront is faster with fewer: it runs the shared searches
// of polyhedra one pair after another, and pairs that part at a branch one side after the other.  Pairs of 1000
// boxes (3,952): 81 us with 64 a wavefront, 60 with 8; triangle tests of 600 bodies on a mesh 315 and 248.
constexpr int kNpWaves = 2048;
__host__ __device__ constexpr int np_least_pairs(int bin) { return bin == ALGO_POLY_POLY || bin == BIN_POLY_POLY_SEP ? 2 : 8; }
__host__ __device__ inline int np_wave_pairs(int bin, int n) {
    int p = np_least_pairs(bin);
    while (p < 64 && p * kNpWaves < n) p *= 2;
    return p;
}
struct NpLists {
    const int* list[kNpLists];
    const int* count[kNpLists];
};
// np_pairs runs in workgroups of exactly this many threads.
constexpr int kNpThreads = 128;
// LDS of a narrowphase wavefront: the clip buffers of its box pairs (two a lane), or the search tables of its mesh
// pairs.  A wavefront goes on to its workgroup's next tile, of whatever list, without waiting for the other, so
// each keeps to a part of its own, the same for both uses.
constexpr int kBoxClip = 8;   // vertices of a box face clipped by the four side planes at most
constexpr int kNpWaveFloats = 2 * 3 * kBoxClip * 64;
__host__ __device__ constexpr int np_wave_lds(int thread) { return thread / 64 * kNpWaveFloats; }
// component c of vertex i in clip buffer b of a thread (consecutive lanes, consecutive words)
__host__ __device__ constexpr int np_clip_lds(int thread, int b, int i, int c) {
    return np_wave_lds(thread) + (3 * (kBoxClip * b + i) + c) * 64 + thread % 64;
}
__host__ __device__ inline int np_tiles(int bin, int n) {   // workgroups' worth of a list
    const int p = np_wave_pairs(bin, n) * (kNpThreads / 64);
    return (n + p - 1) / p;
}
// first pair of a wavefront's share in a tile of a list of n
__host__ __device__ inline int np_first_pair(int bin, int n, int tile, int wave) {
    return (tile * (kNpThreads / 64) + wave) * np_wave_pairs(bin, n);
}
// Workgroups for a list of any length up to n: a list takes fewer tiles than a shorter one where the share of a
// wavefront doubles (4,096 mesh pairs are 1,024 tiles, 4,097 are 513), kNpWaves wavefronts' worth before each.
__host__ __device__ inline int np_grid(int bin, int n) {
    const int most = kNpWaves / (kNpThreads / 64), t = np_tiles(bin, n);
    return n > np_least_pairs(bin) * kNpWaves && t < most ? most : t;
}
__global__ void np_pairs(NpArgs A, NpLists L);   // convex vs concave pairs: the middle phase (lists the triangle tests)
void upload_box_topology(const int* edges4, const int* face_edge, const int* face_verts);
// convex vs concave pairs: the tests, then per pair the potential manifolds, their reduction and the warm-start
// transfer
__global__ void np_concave_tri(NpArgs A);
__global__ void np_concave_reduce(NpArgs A, const int* list, const int* count);

}  // namespace rp3dg
