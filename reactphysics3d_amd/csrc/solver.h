// Kernel argument block and launch declarations of the solver / integration kernels.
#pragma once

#include "rp3d_internal.h"

namespace rp3dg {

constexpr int kMaxColors = 64;

struct SvArgs {
    DevBodies B;
    DevColliders C;
    DevPairs P;
    DevSolver S;
    const int* nm;        // number of manifolds
    const int* mlist;     // manifold -> pair slot (pair order)
    const int* order;     // colour-sorted position -> manifold
    const int* cstart;    // colour ranges [cstart[c], cstart[c+1]) (colour-major layout)
    const int* ncolors;
    float restitution_threshold;
    int learned;          // learned warm start for points without a cached impulse
    const int* adj_offs;  // body -> manifold adjacency offsets (manifold count of a dynamic body)
};

__global__ void dyn_integrate_positions(DevBodies B, float dt, float split_factor);
__global__ void dyn_update_state(DevBodies B);
__global__ void sv_flag_manifolds(const int* ncp, const int* xm, const int* nb_pairs, int* flag);
__global__ void sv_compact_manifolds(const int* flag, const int* offs, const int* nb_pairs, const int* ncp, const int* xm,
                                     const int* xs, int* list, int* counters_manifolds, int* counters_points,
                                     unsigned long long* total_points);
__global__ void sv_adj_count(DevBodies B, DevColliders C, DevPairs P, const int* list, const int* nm_ptr, int* cnt);
__global__ void sv_adj_fill(DevBodies B, DevColliders C, DevPairs P, const int* list, const int* nm_ptr, const int* offs,
                            int* cursor, int* adj, int2* mb);
__global__ void sv_color_round(const int2* mb, const int* nm_ptr, const int* offs, const int* adj, int* color,
                               const int* left_prev, int* left, int* status);
__global__ void sv_color_finish(const int2* mb, const int* nm_ptr, const int* offs, const int* adj, int* color,
                                const int* left_prev, int* rounds, int* status);
__global__ void sv_world_ranges(DevBodies B, DevColliders C, DevPairs P, const int* list, const int* nm_ptr, int nw,
                                int2* mb, int* wmstart);
// Arguments of the group colouring (solver.hip).
struct ColorArgs {
    const int2* mb;        // dynamic bodies of every manifold (-1: none)
    const int* wmstart;    // [nw + 1] first manifold of every world
    const int* gworld;
    const int* wbody;
    int ngroups;
    int lds_bytes;         // dynamic LDS of the launch
    int *color, *order;
    uint64_t* keys;
    int* seg_start;
    int *ncolors, *status;
    int *list, *pend;      // HBM scratch: [2 * manifolds] and [manifolds]
};

// LDS of a group besides its manifolds: colour mask, list head and end, two work lists, per body
__host__ __device__ constexpr int color_body_bytes(int bodies) { return bodies * (8 + 4 + 4 + 2 * 4); }
// per manifold: bodies (16 bits each), its two list entries, and two bits
__host__ __device__ constexpr int color_manifold_bytes(int m) { return m * 8 + (m + 15) / 16 * 4; }

__global__ void sv_group_color(ColorArgs A);
__global__ void sv_color_keys(const int* color, const int* nm_ptr, uint64_t* keys, int* vals, int* seg_cnt, int* ncolors);
__global__ void sv_warmstart(SvArgs A, int color);
constexpr int kTailRows = 256;   // rows at most of a colour that one workgroup takes in a pass
template <bool SPLIT>
__global__ void sv_solve_tail(SvArgs A, int c0, float beta_dt);
__global__ void sv_warmstart_tail(SvArgs A, int c0);
__global__ void sv_note_iterations(int* world_iters, float* world_res, int n, int iters);
template <bool SPLIT>
__global__ void sv_solve_color(SvArgs A, int color, float beta_dt);   // one quad of lanes per manifold
__global__ void sv_store(SvArgs A);

}  // namespace rp3dg
