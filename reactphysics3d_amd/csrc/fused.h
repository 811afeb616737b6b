// Argument block of the fused per-world kernels (fused.hip).
#pragma once

#include "joints.h"
#include "rp3d_internal.h"
#include "solver.h"

namespace rp3dg {

struct FusedArgs {
    SvArgs A;                  // rows in (world group, colour)-major order; A.cstart unused
    DevJoints J;               // rows sorted by (world group, kind, colour, creation index)
    Settings settings;
    const int* seg_start;      // [g * kMaxColors + c]: first row of colour c of group g; [ng * kMaxColors] = total
    const int2* jt_wr;         // [g * jt_slots + s]: joint rows of slot s (kind, colour) of group g
    const int* jt_kind;        // [s]: joint kind of slot s
    int jt_slots;
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
constexpr int kGroupMaxWorlds = 64;   // worlds per group at most (one bit each in the convergence mask)
constexpr int kGroupShift = 16;       // staged body flags carry the body's world index in its group here

__global__ void sv_setup(SvArgs A, DevJoints J, Settings settings, float dt);
__global__ void sv_features(FusedArgs F);
// one instance per contact position-correction technique (SPLIT = split impulses, else Baumgarte contacts)
// and place of the body state (STATE_*, solver_quad.h)
template <bool SPLIT, int STATE>
__global__ void sv_world_solve(FusedArgs F);
__global__ void world_position(FusedArgs F);
// Appends (features, converged impulses) of this step's feature rows to the sample log at *logged.
__global__ void sv_log_samples(FusedArgs F, float* log_feats, float* log_targets, const unsigned long long* logged,
                               long long log_cap);
__global__ void sv_log_advance(const int* nrows, int feat_cap, unsigned long long* logged, long long log_cap);

}  // namespace rp3dg
