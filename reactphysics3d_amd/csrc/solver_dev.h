// Contact solver rows and body integration of the MI355X step path, one item per call.
//
// The reference solves contact manifolds sequentially in island order
// (ContactSolverSystem.cpp:479-759).  Here manifolds are graph-coloured so
// that no two manifolds of a colour share a dynamic body; all manifolds of a
// colour are then solved in parallel, which is exactly the sequential
// Gauss-Seidel sweep in colour order (static and kinematic bodies have zero
// inverse mass and are never written, so they do not constrain the colouring).
// Used by the per-colour kernels (solver.hip) and the fused per-world solver
// (fused.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "kcommon.h"
#include "rp3d_internal.h"
#include "solver.h"

namespace rp3dg {

__device__ __forceinline__ int body_flags(const DevBodies& B, int b) { return B.flags[b - B.vbase]; }
__device__ __forceinline__ bool dyn_body(const DevBodies& B, int b) { return (body_flags(B, b) & BF_DYNAMIC) != 0; }
// lock factors of body b (absolute index; multiplying by 1 is exact, so unit factors are not loaded)
__device__ __forceinline__ void body_locks(const DevBodies& B, int b, V3& ll, V3& al) {
    if (body_flags(B, b) & BF_UNIT_LOCKS) {
        ll = v3(1.0f, 1.0f, 1.0f);
        al = v3(1.0f, 1.0f, 1.0f);
    } else {
        ll = ld3(B.llock, b);
        al = ld3(B.alock, b);
    }
}

// x * f, or x when the lock factor is known to be 1
template <bool LK>
__device__ __forceinline__ float lk(float x, float f) {
    if constexpr (LK) return x * f;
    else return x;
}
template <bool LK>
__device__ __forceinline__ V3 lkv(V3 f, V3 x) {
    if constexpr (LK) return cmul(f, x);
    else return x;
}

// ------------------------------------------------------------------------------------------------
// Integration (DynamicsSystem.cpp, PhysicsWorld.cpp:310-318)
// ------------------------------------------------------------------------------------------------

// updateBodiesInverseWorldInertiaTensors + integrateRigidBodiesVelocities (DynamicsSystem.cpp:117-183)
__device__ __forceinline__ void dyn_integrate_velocities_one(const DevBodies& B, const Settings& S, float dt, int i) {
    {
        const int f = B.flags[i];
        if (!(f & BF_ENABLED)) return;
        const Q4 q = ldq(B.q, i);
        const float4 ii = B.ii[i];
        const M3 Iw = world_inv_inertia(qmat(q), v3(ii.x, ii.y, ii.z));
        B.iw0[i] = f4(Iw.r[0], 0.f);
        B.iw1[i] = f4(Iw.r[1], 0.f);
        B.iw2[i] = f4(Iw.r[2], 0.f);
        B.sv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        B.sw[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        const float4 ll4 = B.llock[i], al4 = B.alock[i];
        const V3 ll = xyz(ll4), al = xyz(al4);
        const float im = ii.w;
        const V3 v = ld3(B.v, i), w = ld3(B.w, i);
        V3 cv = v + cmul((dt * im) * ll, ld3(B.force, i));
        V3 cw = w + cmul(dt * al, mvmul(Iw, ld3(B.torque, i)));
        if (S.gravity_enabled && (f & BF_GRAVITY)) {
            const float mass = B.com[i].w;
            cv = cv + cmul(((dt * im) * ll) * mass, S.gravity);
        }
        const float ld = 1.0f / (1.0f + ll4.w * dt);
        const float ad = 1.0f / (1.0f + al4.w * dt);
        cv = cv * ld;
        cw = cw * ad;
        B.cv[i] = f4(cv, 0.f);
        B.cw[i] = f4(cw, 0.f);
    }
}

// integrateRigidBodiesPositions (DynamicsSystem.cpp:44-71): the split velocities enter with the factor
// 1 (split impulses) or 0 (Baumgarte contacts), multiplied as the reference does
__device__ __forceinline__ void dyn_integrate_positions_one(const DevBodies& B, float dt, int i, float split_factor) {
    {
        if (!(B.flags[i] & BF_ENABLED)) return;
        const V3 nv = ld3(B.cv, i) + split_factor * ld3(B.sv, i);
        const V3 nw = ld3(B.cw, i) + split_factor * ld3(B.sw, i);
        const V3 x = ld3(B.x, i);
        const Q4 q = ldq(B.q, i);
        const V3 cx = x + nv * dt;
        const Q4 dq = qscale(qscale(qmul(q4(nw.x, nw.y, nw.z, 0.0f), q), 0.5f), dt);
        B.cx[i] = f4(cx, 0.f);
        B.cq[i] = f4q(qadd(q, dq));
    }
}

// updateBodiesState (DynamicsSystem.cpp:74-101) and resetBodiesForceAndTorque (:186-195)
__device__ __forceinline__ void dyn_update_state_one(const DevBodies& B, int i) {
    {
        if (B.flags[i] & BF_ENABLED) {
            B.v[i] = B.cv[i];
            B.w[i] = B.cw[i];
            const V3 x = ld3(B.cx, i);
            const Q4 q = qunit(ldq(B.cq, i));
            B.x[i] = f4(x, 0.f);
            B.q[i] = f4q(q);
            B.p[i] = f4(x - qrot(q, ld3(B.com, i)), 0.f);
        }
        B.force[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        B.torque[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
}


// ------------------------------------------------------------------------------------------------
// Solver rows (ContactSolverSystem::initializeForIsland, CS.cpp:115-320) in colour order
// ------------------------------------------------------------------------------------------------

// world inverse inertia rows, indexed [body - vbase] like the velocities (staged in LDS per world)
// World inverse inertia of body b.  Staged in LDS (iw2 == nullptr), its third row lives in the w lanes of
// cw, sv and sw.  The w lanes of the staged velocities are in use in every staged layout (solver_quad.h),
// so the solver rows store velocities with st3 (x, y, z only).
__device__ __forceinline__ M3 body_iw(const DevBodies& B, int b) {
    const int u = b - B.vbase;
    M3 m;
    m.r[0] = ld3(B.iw0, u); m.r[1] = ld3(B.iw1, u);
    m.r[2] = B.iw2 ? ld3(B.iw2, u) : v3(B.cw[u].w, B.sv[u].w, B.sw[u].w);
    return m;
}

// World inverse inertia of body b at the start of a step, in a launch that also runs its velocity
// integration (sv_setup): computed here from the orientation by the integration's own operations for an
// enabled body, whose stored rows that launch rewrites; a disabled body keeps the stored rows.
__device__ __forceinline__ M3 body_iw_setup(const DevBodies& B, int b) {
    M3 m;
    if (B.flags[b] & BF_ENABLED) {
        const float4 ii = B.ii[b];
        m = world_inv_inertia(qmat(ldq(B.q, b)), v3(ii.x, ii.y, ii.z));
    } else {
        m.r[0] = ld3(B.iw0, b); m.r[1] = ld3(B.iw1, b); m.r[2] = ld3(B.iw2, b);
    }
    return m;
}

// computeFrictionVectors (CS.cpp:789-818)
__device__ inline void friction_vectors(V3 dv, V3 n, V3& t1, V3& t2) {
    const float dvn = dot(dv, n);
    const V3 nv = dvn * n;
    const V3 tv = v3(dv.x - nv.x, dv.y - nv.y, dv.z - nv.z);
    const float lt = len(tv);
    if (lt > kMachineEps) t1 = tv / lt;
    else t1 = one_unit_orthogonal(n);
    t2 = cross(n, t1);
}

__device__ __forceinline__ V3 rel_vel(V3 v1, V3 w1, V3 v2, V3 w2, V3 r1, V3 r2) {
    return v3(v2.x + w2.y * r2.z - w2.z * r2.y - v1.x - w1.y * r1.z + w1.z * r1.y,
              v2.y + w2.z * r2.x - w2.x * r2.z - v1.y - w1.z * r1.x + w1.x * r1.z,
              v2.z + w2.x * r2.y - w2.y * r2.x - v1.z - w1.x * r1.y + w1.y * r1.x);
}

__device__ __forceinline__ void sv_prepare_one(const SvArgs& A, int i) {
    {
        const int m = A.order[i];
        const int k = A.mlist[m];
        const DevBodies& B = A.B;
        const DevColliders& C = A.C;
        const DevPairs& P = A.P;
        const DevSolver& S = A.S;
        const int2 c = P.col[k];
        const int b1 = C.body[c.x], b2 = C.body[c.y];
        const V3 x1 = ld3(B.x, b1), x2 = ld3(B.x, b2);
        const M3 I1 = body_iw_setup(B, b1), I2 = body_iw_setup(B, b2);
        const float im1 = B.ii[b1].w, im2 = B.ii[b2].w;
        const float2 m1 = C.mat[c.x], m2 = C.mat[c.y];
        const float mu = m1.x * m2.x;
        const float rest = (m1.y > m2.y) ? m1.y : m2.y;
        const V3 v1 = ld3(B.v, b1), w1 = ld3(B.w, b1), v2 = ld3(B.v, b2), w2 = ld3(B.w, b2);
        const Tf T1 = tf(ld3(C.wpos, c.x), ldq(C.wq, c.x));
        const Tf T2 = tf(ld3(C.wpos, c.y), ldq(C.wq, c.y));
        const int np = P.ncp[k];
        V3 nsum = v3zero(), fp1 = v3zero(), fp2 = v3zero();
        for (int p = 0; p < np; p++) {
            const float4 pn = P.pn[4 * k + p];
            const float4 l1 = P.pl1[4 * k + p];
            const float4 l2 = P.pl2[4 * k + p];
            const V3 n = xyz(pn);
            const V3 p1 = tapply(T1, xyz(l1));
            const V3 p2 = tapply(T2, xyz(l2));
            const V3 r1 = v3(p1.x - x1.x, p1.y - x1.y, p1.z - x1.z);
            const V3 r2 = v3(p2.x - x2.x, p2.y - x2.y, p2.z - x2.z);
            fp1.x += p1.x; fp1.y += p1.y; fp1.z += p1.z;
            fp2.x += p2.x; fp2.y += p2.y; fp2.z += p2.z;
            const V3 dv = rel_vel(v1, w1, v2, w2, r1, r2);
            const V3 i1n = mvmul(I1, cross(r1, n));
            const V3 i2n = mvmul(I2, cross(r2, n));
            const float mp = im1 + im2 + dot(cross(i1n, r1), n) + dot(cross(i2n, r2), n);
            const float imp = mp > 0.0f ? 1.0f / mp : 0.0f;
            float rb = 0.0f;
            const float dvn = dv.x * n.x + dv.y * n.y + dv.z * n.z;
            if (dvn < -A.restitution_threshold) rb = rest * dvn;
            nsum.x += n.x; nsum.y += n.y; nsum.z += n.z;
            S.pn[4 * i + p] = pn;
            S.r1[4 * i + p] = f4(r1, imp);
            S.r2[4 * i + p] = f4(r2, rb);
            S.i1[4 * i + p] = f4(i1n, 0.f);
            S.i2[4 * i + p] = f4(i2n, 0.f);
            // lam: cached normal impulse and resting flag from the warm-start transfer
            S.lam[4 * i + p] = make_float4(l1.w, 0.0f, l2.w, 0.f);
        }
        const float fn = (float)np;
        fp1 = v3(fp1.x / fn, fp1.y / fn, fp1.z / fn);
        fp2 = v3(fp2.x / fn, fp2.y / fn, fp2.z / fn);
        const V3 r1f = v3(fp1.x - x1.x, fp1.y - x1.y, fp1.z - x1.z);
        const V3 r2f = v3(fp2.x - x2.x, fp2.y - x2.y, fp2.z - x2.z);
        const V3 n = normalized(nsum);
        const V3 dvf = rel_vel(v1, w1, v2, w2, r1f, r2f);
        V3 t1, t2;
        friction_vectors(dvf, n, t1, t2);
        const V3 r1ct1 = cross(r1f, t1), r1ct2 = cross(r1f, t2);
        const V3 r2ct1 = cross(r2f, t1), r2ct2 = cross(r2f, t2);
        const float f1m = im1 + im2 + dot(cross(mvmul(I1, r1ct1), r1f), t1) + dot(cross(mvmul(I2, r2ct1), r2f), t1);
        const float f2m = im1 + im2 + dot(cross(mvmul(I1, r1ct2), r1f), t2) + dot(cross(mvmul(I2, r2ct2), r2f), t2);
        const float twm = dot(n, mvmul(I1, n)) + dot(n, mvmul(I2, n));
        S.pair[i] = k;
        S.bodies[i] = make_int2(b1, b2);
        S.npts[i] = np;
        S.n[i] = f4(n, mu);
        S.r1f[i] = f4(r1f, im1);
        S.r2f[i] = f4(r2f, im2);
        S.t1[i] = f4(t1, f1m > 0.0f ? 1.0f / f1m : 0.0f);
        S.t2[i] = f4(t2, f2m > 0.0f ? 1.0f / f2m : 0.0f);
        const float4 fi = P.fimp[k];
        S.imp[i] = make_float4(fi.x, fi.y, fi.z, twm > 0.0f ? 1.0f / twm : 0.0f);   // w: inverse twist mass
        S.oldt1[i] = P.fv1[k];
        S.oldt2[i] = P.fv2[k];
    }
}

// Learned warm start: the 24 features of contact point p of solver row i (after sv_prepare_one and
// the velocity integration): normal, r1, r2, relative velocity in the (t1, t2, n) frame, inverse
// masses, world inverse inertia (xx of each body), the manifold's cached normal impulses (sum over
// its resting points, their count), the manifold counts of both bodies, depth, friction
// coefficient, inverse normal mass, 1 / points in the manifold.
__device__ __forceinline__ void sv_point_features(const SvArgs& A, int i, int p, float* f) {
    const DevBodies& B = A.B;
    const DevSolver& S = A.S;
    const int q = 4 * i + p;
    const int2 bb = S.bodies[i];
    const float4 pn = S.pn[q], r14 = S.r1[q], r24 = S.r2[q];
    const V3 n = xyz(pn), r1 = xyz(r14), r2 = xyz(r24);
    const int u1 = bb.x - B.vbase, u2 = bb.y - B.vbase;
    const V3 dv = rel_vel(ld3(B.cv, u1), ld3(B.cw, u1), ld3(B.cv, u2), ld3(B.cw, u2), r1, r2);
    const V3 t1 = ld3(S.t1, i), t2 = ld3(S.t2, i);
    f[0] = n.x; f[1] = n.y; f[2] = n.z;
    f[3] = r1.x; f[4] = r1.y; f[5] = r1.z;
    f[6] = r2.x; f[7] = r2.y; f[8] = r2.z;
    f[9] = dot(dv, t1); f[10] = dot(dv, t2); f[11] = dot(dv, n);
    f[12] = S.r1f[i].w; f[13] = S.r2f[i].w;
    float cached = 0.0f, resting = 0.0f;
    for (int k = 0; k < S.npts[i]; k++) {
        const float4 l = S.lam[4 * i + k];
        if (l.z != 0.0f) {
            cached += l.x;
            resting += 1.0f;
        }
    }
    const int* ao = A.adj_offs;
    f[14] = B.iw0[bb.x].x; f[15] = cached; f[16] = resting;
    f[17] = B.iw0[bb.y].x;
    f[18] = dyn_body(B, bb.x) ? (float)(ao[bb.x + 1] - ao[bb.x]) : 0.0f;
    f[19] = dyn_body(B, bb.y) ? (float)(ao[bb.y + 1] - ao[bb.y]) : 0.0f;
    f[20] = pn.w;
    f[21] = S.n[i].w;
    f[22] = r14.w;
    f[23] = 1.0f / (float)S.npts[i];
}

// ContactSolverSystem::storeImpulses (CS.cpp:763-785); initializeForIsland marks every point resting (:161)
__device__ __forceinline__ void sv_store_one(const SvArgs& A, int i) {
    {
        const int k = A.S.pair[i];
        const int np = A.S.npts[i];
        const float* lq = reinterpret_cast<const float*>(A.S.lq + 2 * (size_t)i);
        for (int p = 0; p < np; p++) {
            float4 l1 = A.P.pl1[4 * k + p];
            l1.w = lq[p];
            A.P.pl1[4 * k + p] = l1;
            float4 l2 = A.P.pl2[4 * k + p];
            l2.w = 1.0f;
            A.P.pl2[4 * k + p] = l2;
        }
        const float4 imp = A.S.imp[i];
        A.P.fimp[k] = make_float4(imp.x, imp.y, imp.z, 0.f);
        A.P.fv1[k] = f4(ld3(A.S.t1, i), 0.f);
        A.P.fv2[k] = f4(ld3(A.S.t2, i), 0.f);
    }
}

}  // namespace rp3dg
