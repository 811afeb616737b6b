// Argument block of the fused per-world kernels (fused.hip).
#pragma once

#include "joints.h"
#include "rp3d_internal.h"
#include "solver.h"

namespace rp3dg {

struct FusedArgs {
    SvArgs A;                  // rows in (world group, colour)-major order; A.cstart unused
    DevJoints J;               // rows sorted by (world group, strand, kind, colour, creation index)
    Settings settings;
    const int* seg_start;      // [g * kMaxColors + c]: first row of colour c of group g; [ng * kMaxColors] = total
    const int4* jt_segs;       // joints [x, y) of kind z and one colour; w: the whole group takes them (below)
    const int* jt_strands;     // [g * kJointStrands + s]: first segment of strand s of group g; [ng * kJointStrands] = total
    const int* wbody;          // [nw + 1] body ranges of the worlds
    const int* wcoll;          // [nw + 1] collider ranges of the worlds
    const int* gworld;         // [ng + 1] world ranges of the groups (consecutive worlds)
    const int* block_world;    // workgroup -> group (largest groups first)
    const float4* hull_bounds;
    float dt, beta_dt;
    int max_iters;             // velocity iterations (fixed), or the cap in residual mode
    float res_thr;             // > 0: iterate to this velocity residual
    float4 *pv, *pw;           // velocities after the previous sweep (residual mode, bodies beyond a thread's first)
    int* world_iters;          // iterations each world ran in the last step
    float* world_res;          // its last residual (residual mode)
    // learned warm start / sample logging
    float* feats;              // [feat_cap][24] features of the points without a cached impulse
    int* row_slot;             // solver point slot (4 * row + point) of each feature row
    int* nrows;                // feature rows written this step
    int feat_cap;
    int lds_bodies;            // bodies the workgroup's LDS holds (stride of the staged arrays)
    int lds_rows;              // manifolds whose impulses and headers it holds
};

// LDS bytes of a fused solver workgroup: `bodies` bodies in the given layout (solver_quad.h) and `rows`
// manifolds
__host__ __device__ constexpr size_t fused_lds_bytes(int state, int bodies, int rows) {
    return (state == 0 ? (size_t)bodies * 6 * sizeof(float4) + ((size_t)bodies + 3) / 4 * sizeof(float4)
                       : state == 1 ? (size_t)bodies * 3 * sizeof(float4) : 0) +
           (size_t)rows * 3 * sizeof(float4);
}

constexpr int kFeatures = 24;

constexpr int kFusedMaxBlock = 1024;   // threads per group of the solver kernel at most (128 registers a lane)
constexpr int kPositionMaxBlock = 256; // threads per group of the position kernel at most
constexpr int kPositionLds = 64;       // LDS bytes of a body in the position kernel
// Joints that no chain of joints and bodies connects can be solved at the same time, whatever their kind and
// colour.  The connected components of a group's joints are packed into strands; a wavefront takes a strand
// through its segments (kind and colour, in solve order) without waiting for the others, so a sweep is as
// long as its longest strand and not as the number of kinds and colours in the group.  Where that would be
// longer (one large component, that many wavefronts share better), strand 0 has every segment of the group
// and the workgroup takes them together, with a barrier after each (w = 1).  64 joints of 3 kinds in 24
// components: a joint sweep is 2 phases long instead of 6, and sv_world_solve takes 65 us instead of 123 (80 on two
// wavefronts, which take two strands each one after the other).
constexpr int kJointStrands = 4;
constexpr int kMaxJointSegs = 256;     // of a group with several strands
constexpr int kGroupMaxWorlds = 64;   // worlds per group at most (one bit each in the convergence mask)
constexpr int kGroupShift = 16;       // staged body flags carry the body's world index in its group here

__global__ void sv_setup(SvArgs A, DevJoints J, Settings settings, float dt);
__global__ void sv_features(FusedArgs F);
// one instance per contact position-correction technique (SPLIT = split impulses, else Baumgarte contacts)
// and place of the body state (STATE_*, solver_quad.h)
template <bool SPLIT, int STATE>
__global__ void sv_world_solve(FusedArgs F);
// positions of worlds with joints; STAGED: kPositionLds bytes of LDS for each of the group's lds_bodies bodies
template <bool STAGED>
__global__ void world_position(FusedArgs F);
__global__ void body_position(DevBodies B, float dt, float split_factor);
// Appends (features, converged impulses) of this step's feature rows to the sample log at *logged.
__global__ void sv_log_samples(FusedArgs F, float* log_feats, float* log_targets, const unsigned long long* logged,
                               long long log_cap);
__global__ void sv_log_advance(const int* nrows, int feat_cap, unsigned long long* logged, long long log_cap);

}  // namespace rp3dg
