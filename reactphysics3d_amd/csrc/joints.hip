// Per-colour joint kernels (one launch per colour of one joint type).  The rows
// themselves are in joints_dev.h; the fused per-world solver calls the same rows.
#include <hip/hip_runtime.h>

#include "joints.h"
#include "joints_dev.h"
#include "kcommon.h"

namespace rp3dg {

__global__ void jt_warmstart(DevBodies B, DevJoints J, const int* range, int slot) {
    const int lo = range[2 * slot], hi = range[2 * slot + 1];
    RP3DG_GRID_STRIDE(t, hi - lo) jt_warmstart_one(B, J, lo + t);
}

// two lanes per joint
__global__ void jt_solve_velocity(DevBodies B, DevJoints J, const int* range, int slot, int kind, float dt) {
    const int lo = range[2 * slot], hi = range[2 * slot + 1];
    RP3DG_GRID_STRIDE(t, 2 * (hi - lo)) jt_solve_velocity_pair(B, J, kind, lo + (t >> 1), t & 1, dt);
}

__global__ void jt_solve_position(DevBodies B, DevJoints J, const int* range, int slot, int kind) {
    const int lo = range[2 * slot], hi = range[2 * slot + 1];
    const PosBodies<false> P{B.cx, B.cq, B.ii, B.com, B.flags, 0};
    RP3DG_GRID_STRIDE(t, 2 * (hi - lo)) {
        const int j = lo + (t >> 1);
        jt_solve_position_pair(B, P, J, kind, j, t & 1, jt_position_load(J, j, t & 1));
    }
}

}  // namespace rp3dg
