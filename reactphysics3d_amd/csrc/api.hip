// RigidBody state changes between steps, on the device copy of a batch (RigidBody.cpp:151-239, 298-311,
// 794-866, 938-987, 1006-1057).  The host queues the calls in the order the application makes them and
// one thread applies them in that order before the next step or read-back, so a sequence of calls on one
// body composes exactly as the reference's calls do (each reads the state the previous one left).
#include <hip/hip_runtime.h>

#include "api.h"
#include "kcommon.h"
#include "refit_dev.h"

namespace rp3dg {

// RigidBody::setIsSleeping (RigidBody.cpp:1006-1057) for a non-static, active body.
__device__ void api_set_sleeping(const ApiArgs& A, int b, bool sleep) {
    const DevBodies& B = A.B;
    const int f = B.flags[b];
    const bool asleep = !(f & BF_ENABLED);
    if (asleep == sleep) return;
    if (!(f & (BF_DYNAMIC | BF_KINEMATIC))) return;   // a static body is always awake
    if (A.sleep_time) A.sleep_time[b] = 0.0f;
    if (sleep) {
        B.flags[b] = f & ~BF_ENABLED;
        B.v[b] = make_float4(0.f, 0.f, 0.f, 0.f);
        B.w[b] = make_float4(0.f, 0.f, 0.f, 0.f);
        B.force[b] = make_float4(0.f, 0.f, 0.f, 0.f);
        B.torque[b] = make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
        B.flags[b] = f | BF_ENABLED;
        // askForBroadPhaseCollisionCheck: the body's colliders enter the moved set
        for (int k = A.coll_offs[b]; k < A.coll_offs[b + 1]; k++) A.C.moved[A.coll_list[k]] = 1;
    }
}

__global__ void api_apply_ops(ApiArgs A, const ApiOp* ops, int n) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const DevBodies& B = A.B;
    for (int k = 0; k < n; k++) {
        const ApiOp o = ops[k];
        const int b = o.body;
        const int f = B.flags[b];
        const bool dynamic = (f & BF_DYNAMIC) != 0;
        const bool is_static = !(f & (BF_DYNAMIC | BF_KINEMATIC));
        const Q4 q = ldq(B.q, b);
        V3 a = xyz(o.a);
        switch (o.op) {
            case API_SET_TRANSFORM: {   // RigidBody::setTransform (RigidBody.cpp:837-866)
                const Tf t = tf(a, q4(o.b.x, o.b.y, o.b.z, o.b.w));
                const V3 old = ld3(B.x, b);
                const V3 com = tapply(t, ld3(B.com, b));
                B.x[b] = f4(com, 0.f);
                V3 v = ld3(B.v, b);
                v += cross(ld3(B.w, b), com - old);
                st3(B.v, b, v);
                api_set_sleeping(A, b, false);
                B.p[b] = f4(t.p, 0.f);
                B.q[b] = f4q(t.q);
                // Body::setTransform -> updateBroadPhaseState (Body.cpp:226-241, 397-407): new collider
                // transforms, a new fat AABB and a place in the moved set for a shape that left its fat AABB
                for (int j = A.coll_offs[b]; j < A.coll_offs[b + 1]; j++) refit_one(B, A.C, A.hull_bounds, 2, A.coll_list[j]);
                break;
            }
            case API_SET_LINEAR_VELOCITY:   // RigidBody::setLinearVelocity (RigidBody.cpp:794-808)
            case API_SET_ANGULAR_VELOCITY:  // RigidBody::setAngularVelocity (RigidBody.cpp:814-828)
                if (is_static) break;
                if (o.op == API_SET_LINEAR_VELOCITY) st3(B.v, b, a);
                else st3(B.w, b, a);
                if (len2(a) > 0.0f) api_set_sleeping(A, b, false);
                break;
            case API_APPLY_FORCE: {   // RigidBody::apply{Local,World}ForceAt{CenterOfMass,LocalPosition,WorldPosition}
                if (o.flags & API_FORCE_LOCAL) a = qrot(q, a);   // the body orientation times the local force
                if (!dynamic) break;
                api_set_sleeping(A, b, false);
                st3(B.force, b, ld3(B.force, b) + a);
                if (o.flags & API_AT_POINT) {
                    V3 p = xyz(o.b);
                    if (o.flags & API_POINT_LOCAL) p = tapply(tf(ld3(B.p, b), q), p);
                    st3(B.torque, b, ld3(B.torque, b) + cross(p - ld3(B.x, b), a));
                }
                break;
            }
            case API_APPLY_TORQUE:   // RigidBody::applyWorldTorque / applyLocalTorque (RigidBody.cpp:938-967)
                if (o.flags & API_FORCE_LOCAL) a = qrot(q, a);
                if (!dynamic) break;
                api_set_sleeping(A, b, false);
                st3(B.torque, b, ld3(B.torque, b) + a);
                break;
            case API_RESET_FORCE:    // RigidBody::resetForce / resetTorque (RigidBody.cpp:970-987)
                if (dynamic) B.force[b] = make_float4(0.f, 0.f, 0.f, 0.f);
                break;
            case API_RESET_TORQUE:
                if (dynamic) B.torque[b] = make_float4(0.f, 0.f, 0.f, 0.f);
                break;
            case API_SET_SLEEPING:
                api_set_sleeping(A, b, o.flags != 0);
                break;
            default:
                break;
        }
    }
}

// The host's arrays have 3 floats a vector and the device's 4.  Packing on the device and writing over the bus
// costs one launch: 21 us a call for 28 bodies and 224 us for 65,541 (most of it the caller's memory), where
// copying the four arrays whole and packing on the host took 53 and 460 us.  Consecutive lanes write
// consecutive words.
__global__ __launch_bounds__(256) void api_pack_bodies(DevBodies B, int first, int n, float* pos, float* ori, float* lin,
                                                       float* ang) {
    const float* src[4] = {reinterpret_cast<const float*>(B.p + first), reinterpret_cast<const float*>(B.q + first),
                           reinterpret_cast<const float*>(B.v + first), reinterpret_cast<const float*>(B.w + first)};
    float* const dst[4] = {pos, ori, lin, ang};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (!dst[k]) continue;
        if (k == 1) {
            RP3DG_GRID_STRIDE(t, 4 * n) dst[k][t] = src[k][t];
        } else {
            RP3DG_GRID_STRIDE(t, 3 * n) {
                const int i = t / 3;
                dst[k][t] = src[k][4 * i + (t - 3 * i)];
            }
        }
    }
}

// RigidBody::applyWorldForceAtCenterOfMass / applyWorldTorque (RigidBody.cpp:298-311) on every body
__global__ __launch_bounds__(256) void api_add_forces(DevBodies B, int first, int n, const float* force, const float* torque,
                                                      float* sleep_time, int* woke) {
    __shared__ float s_in[2][3 * 256];   // (so that the host's memory is read in whole lines, once)
    for (int i0 = blockIdx.x * 256; i0 < n; i0 += gridDim.x * 256) {
        for (int k = threadIdx.x; k < 3 * 256; k += 256) {
            const bool in = k < 3 * (n - i0);
            s_in[0][k] = in && force ? force[3 * (size_t)i0 + k] : 0.f;
            s_in[1][k] = in && torque ? torque[3 * (size_t)i0 + k] : 0.f;
        }
        __syncthreads();
        const int l = threadIdx.x, i = first + i0 + l;
        if (i0 + l < n) {
            const V3 f = v3(s_in[0][3 * l], s_in[0][3 * l + 1], s_in[0][3 * l + 2]);
            const V3 t = v3(s_in[1][3 * l], s_in[1][3 * l + 1], s_in[1][3 * l + 2]);
            const bool nf = f.x != 0.f || f.y != 0.f || f.z != 0.f, nt = t.x != 0.f || t.y != 0.f || t.z != 0.f;
            const int fl = B.flags[i];
            if ((fl & BF_DYNAMIC) && (nf || nt)) {   // only dynamic bodies take forces
                if (!(fl & BF_ENABLED)) {            // asleep: setIsSleeping(false)
                    B.flags[i] = fl | BF_ENABLED | BF_WOKEN;
                    if (sleep_time) sleep_time[i] = 0.0f;
                    *woke = 1;
                }
                if (nf) st3(B.force, i, ld3(B.force, i) + f);
                if (nt) st3(B.torque, i, ld3(B.torque, i) + t);
            }
        }
        __syncthreads();
    }
}

// Every array of a snapshot in one launch: a copy of its own for each of about 150 took 500 us to put a world
// of 88 bodies back.
__global__ __launch_bounds__(256) void api_copy_arrays(const CopyArray* arrays, int n, int pieces, int back, int skip) {
    __shared__ int s_first[kCopyArrays];
    for (int k = threadIdx.x; k < n; k += 256) s_first[k] = arrays[k].first;
    __syncthreads();
    for (int p = blockIdx.x; p < pieces; p += gridDim.x) {
        int lo = 0, hi = n;   // the last array that starts at or before the piece
        while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            if (s_first[mid] <= p) lo = mid;
            else hi = mid;
        }
        if (lo == skip) continue;
        const CopyArray A = arrays[lo];
        const size_t off = (size_t)(p - s_first[lo]) * kCopyPiece;
        const size_t bytes = min((size_t)kCopyPiece, A.bytes - off);
        const char* src = (back ? A.b : A.a) + off;
        char* dst = (back ? A.a : A.b) + off;
        const int vecs = (int)(bytes / 16);   // (arrays start at multiples of 256 bytes)
        const float4* s4 = reinterpret_cast<const float4*>(src);
        float4* d4 = reinterpret_cast<float4*>(dst);
        for (int k = threadIdx.x; k < vecs; k += 4 * 256) {
            float4 v[4];
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = s4[min(k + 256 * j, vecs - 1)];
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (k + 256 * j < vecs) d4[k + 256 * j] = v[j];
        }
        for (int k = 16 * vecs + threadIdx.x; k < (int)bytes; k += 256) dst[k] = src[k];
    }
}

}  // namespace rp3dg
