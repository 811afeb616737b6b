// Joint rows of the MI355X step path, one joint per call: ball-and-socket (with its cone limit), fixed,
// hinge and slider joints (src/systems/Solve{BallAndSocket,Fixed,Hinge,Slider}JointSystem.cpp) with the
// default non-linear Gauss-Seidel position correction.
//
// Joints never change during a run, so the host colours every joint type once
// (no two joints of a colour share a body, static bodies included: the position
// solver rewrites and renormalises the constrained orientation of both bodies,
// static ones too).  Joints of one colour of one type are solved in parallel;
// types follow the reference's order BallAndSocket -> Fixed -> Hinge -> Slider
// (ConstraintSolverSystem.cpp:94-113).  Used by the per-colour kernels (joints.hip)
// and by the fused per-world solver (fused.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "joints.h"
#include "kcommon.h"
#include "solver_dev.h"
#include "solver_quad.h"

namespace rp3dg {

// ---- small matrix helpers (Matrix3x3.h / Matrix2x2.h) ----
__device__ inline M3 m3(float a, float b, float c, float d, float e, float f, float g, float h, float i) {
    M3 m;
    m.r[0] = v3(a, b, c); m.r[1] = v3(d, e, f); m.r[2] = v3(g, h, i);
    return m;
}
__device__ inline M3 madd(const M3& a, const M3& b) {
    M3 r;
    for (int i = 0; i < 3; i++) r.r[i] = a.r[i] + b.r[i];
    return r;
}
__device__ inline M3 skew(V3 v) { return m3(0, -v.z, v.y, v.z, 0, -v.x, -v.y, v.x, 0); }   // Matrix3x3.h:251-253
__device__ inline float mdet(const M3& m) {   // Matrix3x3.h:211-217
    return (m.r[0].x * (m.r[1].y * m.r[2].z - m.r[2].y * m.r[1].z) -
            m.r[0].y * (m.r[1].x * m.r[2].z - m.r[2].x * m.r[1].z) +
            m.r[0].z * (m.r[1].x * m.r[2].y - m.r[2].x * m.r[1].y));
}
__device__ inline M3 minv(const M3& m, float det) {   // Matrix3x3.cpp:33-52
    const float id = 1.0f / det;
    M3 t = m3((m.r[1].y * m.r[2].z - m.r[2].y * m.r[1].z), -(m.r[0].y * m.r[2].z - m.r[2].y * m.r[0].z),
              (m.r[0].y * m.r[1].z - m.r[0].z * m.r[1].y), -(m.r[1].x * m.r[2].z - m.r[2].x * m.r[1].z),
              (m.r[0].x * m.r[2].z - m.r[2].x * m.r[0].z), -(m.r[0].x * m.r[1].z - m.r[1].x * m.r[0].z),
              (m.r[1].x * m.r[2].y - m.r[2].x * m.r[1].y), -(m.r[0].x * m.r[2].y - m.r[2].x * m.r[0].y),
              (m.r[0].x * m.r[1].y - m.r[0].y * m.r[1].x));
    for (int i = 0; i < 3; i++) t.r[i] = v3(t.r[i].x * id, t.r[i].y * id, t.r[i].z * id);
    return t;
}
__device__ inline M3 mzero() { return m3(0, 0, 0, 0, 0, 0, 0, 0, 0); }

__device__ inline M3 ldm(const float4* r0, const float4* r1, const float4* r2, int i) {
    M3 m;
    m.r[0] = ld3(r0, i); m.r[1] = ld3(r1, i); m.r[2] = ld3(r2, i);
    return m;
}
__device__ inline void stm(float4* r0, float4* r1, float4* r2, int i, const M3& m) {
    r0[i] = f4(m.r[0], 0.f); r1[i] = f4(m.r[1], 0.f); r2[i] = f4(m.r[2], 0.f);
}

// K = (m1+m2) I + U1 I1 U1^T + U2 I2 U2^T, inverted when invertible and a body is dynamic
__device__ inline M3 translation_inverse_mass(float imsum, V3 r1, V3 r2, const M3& I1, const M3& I2, bool anyDyn, bool& ok) {
    const M3 U1 = skew(r1), U2 = skew(r2);
    const M3 K = madd(madd(m3(imsum, 0, 0, 0, imsum, 0, 0, 0, imsum), mmul(mmul(U1, I1), mtranspose(U1))),
                      mmul(mmul(U2, I2), mtranspose(U2)));
    const float det = mdet(K);
    ok = fabsf(det) > kMachineEps;
    if (ok && anyDyn) return minv(K, det);
    return mzero();
}

__device__ inline V3 lock_mul(V3 lock, V3 v) { return cmul(lock, v); }

// q += (0, w) q * 0.5 ; q.normalize()
__device__ inline Q4 nudge(Q4 q, V3 w) {
    const Q4 d = qscale(qmul(q4(w.x, w.y, w.z, 0.0f), q), 0.5f);
    Q4 r = qadd(q, d);
    const float l = qlen(r);
    return q4(r.x / l, r.y / l, r.z / l, r.w / l);
}

// ---- hinge angle (SolveHingeJointSystem.cpp:733-799) ----
__device__ inline float normalized_angle(float a) {
    const float twopi = 2.0f * kPi;
    if (!(fabsf(a) < twopi)) a = fmodf(a, twopi);   // (fmodf returns a itself below 2 pi)
    if (a < -kPi) return a + twopi;
    if (a > kPi) return a - twopi;
    return a;
}
__device__ inline float angle_near_limits(float a, float lo, float hi) {
    const float twopi = 2.0f * kPi;
    if (hi <= lo) return a;
    if (a > hi) {
        const float du = fabsf(normalized_angle(a - hi));
        const float dl = fabsf(normalized_angle(a - lo));
        return (du > dl) ? (a - twopi) : a;
    }
    if (a < lo) {
        const float du = fabsf(normalized_angle(hi - a));
        const float dl = fabsf(normalized_angle(lo - a));
        return (du > dl) ? a : (a + twopi);
    }
    return a;
}
__device__ inline float hinge_angle(Q4 q1, Q4 q2, Q4 qinit, V3 a1, float lo, float hi) {
    Q4 diff = qmul(q2, qconj(q1));
    float l = qlen(diff);
    diff = q4(diff.x / l, diff.y / l, diff.z / l, diff.w / l);
    Q4 rel = qmul(diff, qinit);
    l = qlen(rel);
    rel = q4(rel.x / l, rel.y / l, rel.z / l, rel.w / l);
    const float c = rel.w;
    const V3 vv = v3(rel.x, rel.y, rel.z);
    const float s = len(vv);
    const float d = dot(vv, a1);
    float ang = d >= 0.0f ? 2.0f * ref_atan2f(s, c) : 2.0f * ref_atan2f(s, -c);
    ang = normalized_angle(ang);
    return angle_near_limits(ang, lo, hi);
}

// PhysicsWorld::enableDisableJoints (PhysicsWorld.cpp:363-393): a joint whose bodies are both disabled
// (static or sleeping) is not solved and keeps its impulses
__device__ __forceinline__ bool joint_enabled(const DevBodies& B, int b1, int b2) {
    return ((body_flags(B, b1) | body_flags(B, b2)) & BF_ENABLED) != 0;
}

// ------------------------------------------------------------------------------------------------
// initBeforeSolve (all joints, one launch; no body state is written)
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ void jt_init_one(const DevBodies& B, const DevJoints& J, int j, float dt) {
    {
        const int2 bb = J.bodies[j];
        const int b1 = bb.x, b2 = bb.y;
        if (!joint_enabled(B, b1, b2)) return;
        const int t = J.type[j];
        const M3 I1 = body_iw_setup(B, b1), I2 = body_iw_setup(B, b2);
        const Q4 q1 = ldq(B.q, b1), q2 = ldq(B.q, b2);
        const V3 r1 = qrot(q1, ld3(J.la1, j) - ld3(B.com, b1));
        const V3 r2 = qrot(q2, ld3(J.la2, j) - ld3(B.com, b2));
        const float im1 = B.ii[b1].w, im2 = B.ii[b2].w;
        J.r1[j] = f4(r1, im1);
        J.r2[j] = f4(r2, im2);
        const bool anyDyn = ((body_flags(B, b1) | body_flags(B, b2)) & BF_DYNAMIC) != 0;
        bool ok;
        const M3 Kt = translation_inverse_mass(im1 + im2, r1, r2, I1, I2, anyDyn, ok);
        stm(J.kt0, J.kt1, J.kt2, j, Kt);
        // Baumgarte biases (BETA = 0.2, biasFactor = BETA / mTimeStep in every Solve*JointSystem::initBeforeSolve)
        const bool bg = (J.flags[j] & JF_BAUMGARTE) != 0;
        const float bf = 0.2f / dt;
        if (t == JT_BALLSOCKET) {
            // cone-limit axis a x b with a = unit(r1), b = -unit(r2) (SolveBallAndSocketJointSystem.cpp:113-115)
            const V3 r1u = unit(r1), r2u = -unit(r2);
            const V3 acb = cross(r1u, r2u);
            J.a1[j] = f4(acb, 0.f);
            int fl = J.flags[j];
            float cone_bias = 0.0f;
            if (fl & JF_LIMIT) {
                // SolveBallAndSocketJointSystem.cpp:117-146.  A disabled limit keeps the half angle pi
                // (PhysicsWorld.cpp:500), which acos never exceeds: never violated, impulse stays 0.
                const float err = J.lim[j].x - ref_acosf(dot(r1u, r2u));
                const bool old = (fl & JF_LOWER_VIOLATED) != 0;
                const bool vio = err < 0.0f;
                fl = vio ? (fl | JF_LOWER_VIOLATED) : (fl & ~JF_LOWER_VIOLATED);
                if (!vio || vio != old) {
                    float4 il = J.impL[j];
                    il.x = 0.0f;
                    J.impL[j] = il;
                }
                float m = dot(acb, mvmul(I1, acb)) + dot(acb, mvmul(I2, acb));
                J.imlm[j] = m > 0.0f ? 1.0f / m : 0.0f;
                J.flags[j] = fl;
                cone_bias = bf * err;   // SolveBallAndSocketJointSystem.cpp:146-149
            }
            // SolveBallAndSocketJointSystem.cpp:113-117
            if (bg) J.bias0[j] = f4(bf * (ld3(B.x, b2) + r2 - ld3(B.x, b1) - r1), cone_bias);
        } else if (t == JT_FIXED) {
            // SolveFixedJointSystem.cpp:120-129: keeps I1 + I2 when it cannot be inverted
            M3 Kr = madd(I1, I2);
            const float det = mdet(Kr);
            if (fabsf(det) > kMachineEps && anyDyn) Kr = minv(Kr, det);
            stm(J.kr0, J.kr1, J.kr2, j, Kr);
            if (bg) {   // SolveFixedJointSystem.cpp:110-132
                J.bias0[j] = f4(bf * (ld3(B.x, b2) + r2 - ld3(B.x, b1) - r1), 0.f);
                const Q4 qe = qmul(qmul(q2, ldq(J.qinit, j)), qconj(q1));
                J.bias1[j] = f4((bf * 2.0f) * v3(qe.x, qe.y, qe.z), 0.f);
            }
        } else if (t == JT_HINGE) {
            const V3 a1 = normalized(qrot(q1, ld3(J.ax1, j)));
            const V3 a2 = normalized(qrot(q2, ld3(J.ax2, j)));
            const V3 b2v = one_unit_orthogonal(a2);
            const V3 c2v = cross(a2, b2v);
            const V3 b2xa1 = cross(b2v, a1), c2xa1 = cross(c2v, a1);
            J.a1[j] = f4(a1, 0.f);
            J.b2xa1[j] = f4(b2xa1, 0.f);
            J.c2xa1[j] = f4(c2xa1, 0.f);
            const V3 i1b = mvmul(I1, b2xa1), i1c = mvmul(I1, c2xa1), i2b = mvmul(I2, b2xa1), i2c = mvmul(I2, c2xa1);
            const float e11 = dot(b2xa1, i1b) + dot(b2xa1, i2b);
            const float e12 = dot(b2xa1, i1c) + dot(b2xa1, i2c);
            const float e21 = dot(c2xa1, i1b) + dot(c2xa1, i2b);
            const float e22 = dot(c2xa1, i1c) + dot(c2xa1, i2c);
            float4 kr = make_float4(0.f, 0.f, 0.f, 0.f);
            const float det = e11 * e22 - e21 * e12;
            if (fabsf(det) > kMachineEps && anyDyn) {
                const float id = 1.0f / det;
                kr = make_float4(e22 * id, -e12 * id, -e21 * id, e11 * id);
            }
            J.kr0[j] = kr;
            // limits / motor (SolveHingeJointSystem.cpp:159-212)
            int fl = J.flags[j];
            const float4 lim = J.lim[j];
            float4 il = J.impL[j];
            // SolveHingeJointSystem.cpp:91-95, 124-128, 198-209 (the limit biases are read only while a
            // limit is violated, a step in which they are computed)
            float4 brot = make_float4(bf * dot(a1, b2v), bf * dot(a1, c2v), 0.f, 0.f);
            if ((fl & JF_LIMIT) || (fl & JF_MOTOR)) {
                const float ang = hinge_angle(q1, q2, ldq(J.qinit, j), a1, lim.x, lim.y);
                const float le = ang - lim.x, ue = lim.y - ang;
                brot.z = bf * le;
                brot.w = bf * ue;
                const bool oldL = (fl & JF_LOWER_VIOLATED) != 0, oldU = (fl & JF_UPPER_VIOLATED) != 0;
                const bool vl = le <= 0, vu = ue <= 0;
                fl = vl ? (fl | JF_LOWER_VIOLATED) : (fl & ~JF_LOWER_VIOLATED);
                fl = vu ? (fl | JF_UPPER_VIOLATED) : (fl & ~JF_UPPER_VIOLATED);
                if (!vl || vl != oldL) il.x = 0.0f;
                if (!vu || vu != oldU) il.y = 0.0f;
                if ((fl & JF_MOTOR) || ((fl & JF_LIMIT) && (vl || vu))) {
                    float m = dot(a1, mvmul(I1, a1)) + dot(a1, mvmul(I2, a1));
                    m = m > 0.0f ? 1.0f / m : 0.0f;
                    J.imlm[j] = m;
                }
                J.flags[j] = fl;
                J.impL[j] = il;
            }
            if (bg) {
                J.bias0[j] = f4(bf * (ld3(B.x, b2) + r2 - ld3(B.x, b1) - r1), 0.f);
                J.bias1[j] = brot;
            }
        } else {   // slider, SolveSliderJointSystem.cpp:52-237
            const V3 ax = normalized(qrot(q1, ld3(J.ax1, j)));
            const V3 n1 = one_unit_orthogonal(ax);
            const V3 n2 = cross(ax, n1);
            const V3 u = ld3(B.x, b2) + r2 - ld3(B.x, b1) - r1;
            const V3 rpu = r1 + u;
            const V3 un1 = cross(rpu, n1), un2 = cross(rpu, n2), ua = cross(rpu, ax);
            J.a1[j] = f4(ax, 0.f);
            J.b2xa1[j] = f4(n1, 0.f);
            J.c2xa1[j] = f4(n2, 0.f);
            J.un1[j] = f4(un1, 0.f);
            J.un2[j] = f4(un2, 0.f);
            J.ua[j] = f4(ua, 0.f);
            // limit state is tracked whether or not the limit is enabled
            const float ud = dot(u, ax);
            const float4 lim = J.lim[j];
            const float le = ud - lim.x, ue = lim.y - ud;
            int fl = J.flags[j];
            float4 il = J.impL[j];
            const bool oldL = (fl & JF_LOWER_VIOLATED) != 0, oldU = (fl & JF_UPPER_VIOLATED) != 0;
            const bool vl = le <= 0, vu = ue <= 0;
            fl = vl ? (fl | JF_LOWER_VIOLATED) : (fl & ~JF_LOWER_VIOLATED);
            fl = vu ? (fl | JF_UPPER_VIOLATED) : (fl & ~JF_UPPER_VIOLATED);
            if (!vl || vl != oldL) il.x = 0.0f;
            if (!vu || vu != oldU) il.y = 0.0f;
            J.flags[j] = fl;
            J.impL[j] = il;
            if (bg) {   // SolveSliderJointSystem.cpp:116-122, 142-152, 208-213
                J.bias0[j] = make_float4(dot(u, n1) * bf, dot(u, n2) * bf, bf * le, bf * ue);
                const Q4 qe = qmul(qmul(q2, ldq(J.qinit, j)), qconj(q1));
                J.bias1[j] = f4((bf * 2.0f) * v3(qe.x, qe.y, qe.z), 0.f);
                if (J.bfirst) atomicMin(J.bfirst + B.world[b1], J.srank[j]);
            }
            const float ims = im1 + im2;
            if ((fl & JF_LIMIT) && (vl || vu)) {
                // reads r2 x axis of the previous step (recomputed only below)
                const V3 ra_old = ld3(J.ra, j);
                const float m = ims + dot(ua, mvmul(I1, ua)) + dot(ra_old, mvmul(I2, ra_old));
                J.imlm[j] = m > 0.0f ? 1.0f / m : 0.0f;
            }
            const V3 rn1 = cross(r2, n1), rn2 = cross(r2, n2);
            J.rn1[j] = f4(rn1, 0.f);
            J.rn2[j] = f4(rn2, 0.f);
            J.ra[j] = f4(cross(r2, ax), 0.f);
            const V3 i1n1 = mvmul(I1, un1), i1n2 = mvmul(I1, un2), i2n1 = mvmul(I2, rn1), i2n2 = mvmul(I2, rn2);
            const float e11 = ims + dot(un1, i1n1) + dot(rn1, i2n1);
            const float e12 = dot(un1, i1n2) + dot(rn1, i2n2);
            const float e21 = dot(un2, i1n1) + dot(rn2, i2n1);
            const float e22 = ims + dot(un2, i1n2) + dot(rn2, i2n2);
            float4 kt = make_float4(0.f, 0.f, 0.f, 0.f);
            const float det = e11 * e22 - e21 * e12;
            if (fabsf(det) > kMachineEps && anyDyn) {
                const float id = 1.0f / det;
                kt = make_float4(e22 * id, -e12 * id, -e21 * id, e11 * id);
            }
            J.kt0[j] = kt;
            M3 Kr = madd(I1, I2);
            const float detr = mdet(Kr);
            if (fabsf(detr) > kMachineEps && anyDyn) Kr = minv(Kr, detr);
            stm(J.kr0, J.kr1, J.kr2, j, Kr);
            if (fl & JF_MOTOR) J.imm[j] = ims > 0.0f ? 1.0f / ims : 0.0f;
        }
    }
}

// ------------------------------------------------------------------------------------------------
// warm start (per colour)
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ void jt_warmstart_one(const DevBodies& B, const DevJoints& J, int j) {
    {
        const int2 bb = J.bodies[j];
        const int b1 = bb.x, b2 = bb.y;
        if (!joint_enabled(B, b1, b2)) return;
        const int type = J.type[j];
        const int u1 = b1 - B.vbase, u2 = b2 - B.vbase;
        V3 v1 = ld3(B.cv, u1), w1 = ld3(B.cw, u1), v2 = ld3(B.cv, u2), w2 = ld3(B.cw, u2);
        const float im1 = B.ii[b1].w, im2 = B.ii[b2].w;
        V3 ll1, al1, ll2, al2;
        body_locks(B, b1, ll1, al1);
        body_locks(B, b2, ll2, al2);
        const M3 I1 = body_iw(B, b1), I2 = body_iw(B, b2);   // as jt_init_one's: the state's rows do not change in a step
        const V3 r1 = ld3(J.r1, j), r2 = ld3(J.r2, j);
        const V3 it = ld3(J.impT, j);
        if (type == JT_BALLSOCKET) {   // SolveBallAndSocketJointSystem.cpp:196-241
            // the cone impulse stays 0 while the limit is disabled; 0 * (a x b) is still added (keeps the
            // sign of zero components identical to the reference)
            const V3 cone = J.impL[j].x * ld3(J.a1, j);
            const V3 li1 = -it;
            V3 ai1 = cross(it, r1);
            ai1 += cone;
            v1 += lock_mul((im1 * ll1), li1);
            w1 += cmul(al1, mvmul(I1, ai1));
            V3 ai2 = -cross(it, r2);
            ai2 += -cone;
            v2 += lock_mul((im2 * ll2), it);
            w2 += cmul(al2, mvmul(I2, ai2));
        } else if (type == JT_FIXED) {   // SolveFixedJointSystem.cpp:142-186
            const V3 ir = ld3(J.impR, j);
            const V3 li1 = -it;
            V3 ai1 = cross(it, r1);
            ai1 += -ir;
            v1 += lock_mul((im1 * ll1), li1);
            w1 += cmul(al1, mvmul(I1, ai1));
            V3 ai2 = -cross(it, r2);
            ai2 += ir;
            v2 += lock_mul((im2 * ll2), it);
            w2 += cmul(al2, mvmul(I2, ai2));
        } else if (type == JT_HINGE) {   // SolveHingeJointSystem.cpp:216-270
            const float4 ir = J.impR[j];
            const float4 il = J.impL[j];
            const V3 a1 = ld3(J.a1, j), bxa = ld3(J.b2xa1, j), cxa = ld3(J.c2xa1, j);
            const V3 rot = (-bxa) * ir.x - cxa * ir.y;
            const V3 limI = (il.y - il.x) * a1;
            const V3 motI = (-il.z) * a1;
            const V3 li1 = -it;
            V3 ai1 = cross(it, r1);
            ai1 += rot;
            ai1 += limI;
            ai1 += motI;
            v1 += lock_mul((im1 * ll1), li1);
            w1 += cmul(al1, mvmul(I1, ai1));
            V3 ai2 = -cross(it, r2);
            ai2 += -rot;
            ai2 += -limI;
            ai2 += -motI;
            v2 += lock_mul((im2 * ll2), it);
            w2 += cmul(al2, mvmul(I2, ai2));
        } else {   // slider, SolveSliderJointSystem.cpp:240-314
            const float4 ir = J.impR[j];
            const float4 il = J.impL[j];
            const V3 ax = ld3(J.a1, j), n1 = ld3(J.b2xa1, j), n2 = ld3(J.c2xa1, j);
            const V3 un1 = ld3(J.un1, j), un2 = ld3(J.un2, j);
            const float lims = il.y - il.x;
            const V3 linLim = lims * ax;
            const V3 motI = il.z * ax;
            V3 li1 = (-n1) * it.x - n2 * it.y;
            V3 ai1 = (-un1) * it.x - un2 * it.y;
            ai1 += -v3(ir.x, ir.y, ir.z);
            li1 += linLim;
            ai1 += lims * ld3(J.ua, j);
            li1 += motI;
            v1 += lock_mul((im1 * ll1), li1);
            w1 += cmul(al1, mvmul(I1, ai1));
            V3 li2 = n1 * it.x + n2 * it.y;
            V3 ai2 = ld3(J.rn1, j) * it.x + ld3(J.rn2, j) * it.y;
            ai2 += v3(ir.x, ir.y, ir.z);
            li2 += -linLim;
            ai2 += (-lims) * ld3(J.ra, j);
            li2 += -motI;
            v2 += lock_mul((im2 * ll2), li2);
            w2 += cmul(al2, mvmul(I2, ai2));
        }
        st3(B.cv, u1, v1); st3(B.cw, u1, w1);
        st3(B.cv, u2, v2); st3(B.cw, u2, w2);
    }
}

// ------------------------------------------------------------------------------------------------
// velocity constraints (per colour), two lanes per joint: the even lane holds body 1, the odd lane body 2
// ------------------------------------------------------------------------------------------------
// A joint row is a dependent chain like a contact's (solver_quad.h) and a colour has few joints, so the two
// bodies' halves run side by side: each lane keeps its body's velocities, inertia and lever arm and does
// half of the arithmetic, in the reference's operations and order; the row's impulse is computed in body 2's
// lane and passed by DPP, and body 1's sign is applied by flipping sign bits (exact).
struct JointBody {
    V3 v, w, iml, al;   // velocities; inverse mass x linear lock factors, angular lock factors
    M3 I;
    unsigned int s1, s2;   // sign bits: s1 flips in body 1's lane, s2 in body 2's
};
__device__ __forceinline__ V3 flip3(V3 a, unsigned int m) { return v3(flip(a.x, m), flip(a.y, m), flip(a.z, m)); }
__device__ __forceinline__ V3 pair_from1(V3 a) { return v3(dpp<kQuadFrom1>(a.x), dpp<kQuadFrom1>(a.y), dpp<kQuadFrom1>(a.z)); }
__device__ __forceinline__ V3 pair_from2(V3 a) { return v3(dpp<kQuadFrom2>(a.x), dpp<kQuadFrom2>(a.y), dpp<kQuadFrom2>(a.z)); }
__device__ __forceinline__ void joint_spin(JointBody& b, V3 angular) { b.w += cmul(b.al, mvmul(b.I, angular)); }

// v2 + w2 x r2 - v1 - w1 x r1 (valid in body 2's lane)
__device__ __forceinline__ V3 joint_rel_vel(const JointBody& b, V3 r) {
    const V3 c = cross(b.w, r);
    return b.v + c - pair_from1(b.v) - pair_from1(c);
}
// translation impulse dl (of body 2's lane) of the three point-to-point rows
__device__ __forceinline__ void joint_push(JointBody& b, V3 r, V3 dl2) {
    const V3 dl = pair_from2(dl2);
    b.v += lock_mul(b.iml, flip3(dl, b.s1));
    joint_spin(b, flip3(cross(dl, r), b.s2));
}

// kind: the joint kind of the slot (uniform)
__device__ __forceinline__ void jt_solve_velocity_pair(const DevBodies& B, const DevJoints& J, int kind, int j, int side,
                                                       float dt) {
    const int2 bb = J.bodies[j];
    const int bi = side ? bb.y : bb.x, u = bi - B.vbase;
    const int fl = J.flags[j];
    const float4 r4 = side ? J.r2[j] : J.r1[j];   // w: inverse mass
    float4 it = J.impT[j];
    if (!joint_enabled(B, bb.x, bb.y)) return;
    const V3 r = xyz(r4);
    JointBody b;
    b.v = ld3(B.cv, u);
    b.w = ld3(B.cw, u);
    b.I = body_iw(B, bi);
    V3 ll;
    body_locks(B, bi, ll, b.al);
    b.iml = r4.w * ll;
    b.s1 = side ? 0u : 0x80000000u;
    b.s2 = side ? 0x80000000u : 0u;
    // Baumgarte biases; zero under non-linear Gauss-Seidel position correction
    float4 bias0 = make_float4(0.f, 0.f, 0.f, 0.f), bias1 = bias0;
    if (fl & JF_BAUMGARTE) {
        bias0 = J.bias0[j];
        bias1 = J.bias1[j];
    }
    const V3 bt = v3(bias0.x, bias0.y, bias0.z);
    if (kind == JT_BALLSOCKET) {   // SolveBallAndSocketJointSystem.cpp:245-308
        const M3 Kt = ldm(J.kt0, J.kt1, J.kt2, j);
        if ((fl & (JF_LIMIT | JF_LOWER_VIOLATED)) == (JF_LIMIT | JF_LOWER_VIOLATED)) {
            const V3 acb = ld3(J.a1, j);
            const float JvC = dot(acb, pair_from1(b.w) - b.w);
            float d = J.imlm[j] * (-JvC - bias0.w);
            float4 il = J.impL[j];
            const float lt = il.x;
            il.x = fmax_s(il.x + d, 0.0f);
            d = dpp<kQuadFrom2>(il.x - lt);
            if (side) J.impL[j] = il;
            joint_spin(b, flip(d, b.s2) * acb);
        }
        const V3 dl = mvmul(Kt, -joint_rel_vel(b, r) - bt);
        if (side) J.impT[j] = f4(xyz(it) + dl, 0.f);
        joint_push(b, r, dl);
    } else if (kind == JT_FIXED) {   // SolveFixedJointSystem.cpp:189-262
        const M3 Kt = ldm(J.kt0, J.kt1, J.kt2, j), Kr = ldm(J.kr0, J.kr1, J.kr2, j);
        const V3 ir = ld3(J.impR, j);
        const V3 dl = mvmul(Kt, -joint_rel_vel(b, r) - bt);
        if (side) J.impT[j] = f4(xyz(it) + dl, 0.f);
        joint_push(b, r, dl);
        const V3 Jvr = b.w - pair_from1(b.w);
        const V3 dl2 = mvmul(Kr, -Jvr - v3(bias1.x, bias1.y, bias1.z));
        if (side) J.impR[j] = f4(ir + dl2, 0.f);
        joint_spin(b, flip3(pair_from2(dl2), b.s1));
    } else if (kind == JT_HINGE) {   // SolveHingeJointSystem.cpp:273-440
        const M3 Kt = ldm(J.kt0, J.kt1, J.kt2, j);
        const V3 a1 = ld3(J.a1, j), bxa = ld3(J.b2xa1, j), cxa = ld3(J.c2xa1, j);
        const float4 kr = J.kr0[j];
        float4 ir = J.impR[j];
        if (fl & (JF_LIMIT | JF_MOTOR)) {
            float4 il = J.impL[j];
            const float imlm = J.imlm[j];
            if (fl & JF_LIMIT) {
                if (fl & JF_LOWER_VIOLATED) {
                    const float JvL = dot(b.w - pair_from1(b.w), a1);
                    float d = imlm * (-JvL - bias1.z);
                    const float lt = il.x;
                    il.x = fmax_s(il.x + d, 0.0f);
                    d = dpp<kQuadFrom2>(il.x - lt);
                    joint_spin(b, flip(d, b.s1) * a1);
                }
                if (fl & JF_UPPER_VIOLATED) {
                    const float JvU = -dot(b.w - pair_from1(b.w), a1);
                    float d = imlm * (-JvU - bias1.w);
                    const float lt = il.y;
                    il.y = fmax_s(il.y + d, 0.0f);
                    d = dpp<kQuadFrom2>(il.y - lt);
                    joint_spin(b, flip(d, b.s2) * a1);
                }
            }
            if (fl & JF_MOTOR) {
                const float4 lim = J.lim[j];
                const float JvM = dot(a1, pair_from1(b.w) - b.w);
                const float maxI = lim.w * dt;
                float d = imlm * (-JvM - lim.z);
                const float lt = il.z;
                il.z = clampf(il.z + d, -maxI, maxI);
                d = dpp<kQuadFrom2>(il.z - lt);
                joint_spin(b, flip(d, b.s1) * a1);
            }
            if (side) J.impL[j] = il;
        }
        const float db = dot(bxa, b.w), dc = dot(cxa, b.w);
        const float jr0 = -dpp<kQuadFrom1>(db) + db;
        const float jr1 = -dpp<kQuadFrom1>(dc) + dc;
        const float x0 = -jr0 - bias1.x, x1 = -jr1 - bias1.y;
        float d0 = kr.x * x0 + kr.y * x1;
        float d1 = kr.z * x0 + kr.w * x1;
        ir.x += d0;
        ir.y += d1;
        if (side) J.impR[j] = ir;
        d0 = dpp<kQuadFrom2>(d0);
        d1 = dpp<kQuadFrom2>(d1);
        joint_spin(b, flip3(bxa, b.s1) * d0 + flip3(cxa, b.s1) * d1);
        const V3 dl = mvmul(Kt, -joint_rel_vel(b, r) - bt);
        if (side) J.impT[j] = f4(xyz(it) + dl, 0.f);
        joint_push(b, r, dl);
    } else {   // slider, SolveSliderJointSystem.cpp:317-510
        const V3 ax = ld3(J.a1, j), arm = side ? ld3(J.ra, j) : ld3(J.ua, j);
        const M3 Kr = ldm(J.kr0, J.kr1, J.kr2, j);
        const V3 ir = ld3(J.impR, j);
        if (fl & (JF_LIMIT | JF_MOTOR)) {
            float4 il = J.impL[j];
            if (fl & JF_LIMIT) {
                const float imlm = J.imlm[j];
                if (fl & JF_LOWER_VIOLATED) {
                    const float dv = dot(ax, b.v), dw = dot(arm, b.w);
                    const float JvL = dv + dw - dpp<kQuadFrom1>(dv) - dpp<kQuadFrom1>(dw);
                    float d = imlm * (-JvL - bias0.z);
                    const float lt = il.x;
                    il.x = fmax_s(il.x + d, 0.0f);
                    d = flip(dpp<kQuadFrom2>(il.x - lt), b.s1);
                    b.v += lock_mul(b.iml, d * ax);
                    joint_spin(b, d * arm);
                }
                if (fl & JF_UPPER_VIOLATED) {
                    const float dv = dot(ax, b.v), dw = dot(arm, b.w);
                    const float JvU = dpp<kQuadFrom1>(dv + dw) - dv - dw;
                    float d = imlm * (-JvU - bias0.w);
                    const float lt = il.y;
                    il.y = fmax_s(il.y + d, 0.0f);
                    d = flip(dpp<kQuadFrom2>(il.y - lt), b.s2);
                    b.v += lock_mul(b.iml, d * ax);
                    joint_spin(b, d * arm);
                }
            }
            if (fl & JF_MOTOR) {
                const float4 lim = J.lim[j];
                const float dv = dot(ax, b.v);
                const float JvM = dpp<kQuadFrom1>(dv) - dv;
                const float maxI = lim.w * dt;
                float d = J.imm[j] * (-JvM - lim.z);
                const float lt = il.z;
                il.z = clampf(il.z + d, -maxI, maxI);
                d = flip(dpp<kQuadFrom2>(il.z - lt), b.s2);
                b.v += lock_mul(b.iml, d * ax);
            }
            if (side) J.impL[j] = il;
        }
        // 3 rotation rows
        const V3 Jvr = b.w - pair_from1(b.w);
        const V3 dr = mvmul(Kr, -Jvr - v3(bias1.x, bias1.y, bias1.z));
        if (side) J.impR[j] = f4(ir + dr, 0.f);
        joint_spin(b, flip3(pair_from2(dr), b.s1));
        // 2 translation rows
        const V3 n1 = ld3(J.b2xa1, j), n2 = ld3(J.c2xa1, j);
        const V3 arm1 = side ? ld3(J.rn1, j) : ld3(J.un1, j), arm2 = side ? ld3(J.rn2, j) : ld3(J.un2, j);
        const float p1 = dot(n1, b.v), q1 = dot(b.w, arm1), p2 = dot(n2, b.v), q2 = dot(b.w, arm2);
        const float el1 = -dpp<kQuadFrom1>(p1) - dpp<kQuadFrom1>(q1) + p1 + q1;
        const float el2 = -dpp<kQuadFrom1>(p2) - dpp<kQuadFrom1>(q2) + p2 + q2;
        const float x0 = -el1 - bias0.x, x1 = -el2 - bias0.y;
        const float4 kt = J.kt0[j];
        float d0 = kt.x * x0 + kt.y * x1;
        float d1 = kt.z * x0 + kt.w * x1;
        it.x += d0;
        it.y += d1;
        if (side) J.impT[j] = it;
        d0 = dpp<kQuadFrom2>(d0);
        d1 = dpp<kQuadFrom2>(d1);
        const V3 li1 = (-n1) * d0 - n2 * d1;
        b.v += lock_mul(b.iml, flip3(li1, b.s2));
        joint_spin(b, flip3(arm1, b.s1) * d0 + flip3(arm2, b.s1) * d1);
    }
    st3(B.cv, u, b.v);
    st3(B.cw, u, b.w);
}

// ------------------------------------------------------------------------------------------------
// non-linear Gauss-Seidel position correction (per colour), two lanes per joint as above
// ------------------------------------------------------------------------------------------------
// Constrained positions and what the correction reads of a body, indexed [body - base]: arrays of the whole
// batch, or staged in LDS with the body's flags in the w lanes of x (STAGED).
template <bool STAGED>
struct PosBodies {
    float4 *x, *q;
    const float4 *ii, *com;
    const int* flags;   // unless STAGED
    int base;
    __device__ __forceinline__ int body_flags(int u) const {
        if constexpr (STAGED) return __float_as_int(x[u].w);
        else return flags[u];
    }
};

// What the correction reads of a joint and does not change, loaded ahead of its turn.
struct JointPos {
    int2 bodies;
    int fl;              // the violation bits may be old: they are found anew
    V3 la, ax;           // this side's anchor and axis
    Q4 qinit;
    float4 lim;
};
__device__ __forceinline__ JointPos jt_position_load(const DevJoints& J, int j, int side) {
    JointPos p;
    p.bodies = J.bodies[j];
    p.fl = J.flags[j];
    p.la = side ? ld3(J.la2, j) : ld3(J.la1, j);
    p.ax = side ? ld3(J.ax2, j) : ld3(J.ax1, j);
    p.qinit = ldq(J.qinit, j);
    p.lim = J.lim[j];
    return p;
}

__device__ __forceinline__ float pair_other(float a) { return dpp<kQuadOther>(a); }
__device__ __forceinline__ float pair_from1(float a) { return dpp<kQuadFrom1>(a); }
__device__ __forceinline__ float pair_from2(float a) { return dpp<kQuadFrom2>(a); }
__device__ __forceinline__ Q4 pair_from1(Q4 a) { return q4(dpp<kQuadFrom1>(a.x), dpp<kQuadFrom1>(a.y), dpp<kQuadFrom1>(a.z), dpp<kQuadFrom1>(a.w)); }
__device__ __forceinline__ Q4 pair_from2(Q4 a) { return q4(dpp<kQuadFrom2>(a.x), dpp<kQuadFrom2>(a.y), dpp<kQuadFrom2>(a.z), dpp<kQuadFrom2>(a.w)); }
__device__ __forceinline__ M3 pair_from1(const M3& a) { M3 m; for (int i = 0; i < 3; i++) m.r[i] = pair_from1(a.r[i]); return m; }
__device__ __forceinline__ M3 pair_from2(const M3& a) { M3 m; for (int i = 0; i < 3; i++) m.r[i] = pair_from2(a.r[i]); return m; }

struct JointSide {
    V3 x, r, iml, al;   // position, lever arm; inverse mass x linear lock factors, angular lock factors
    Q4 q;
    M3 I;
    unsigned int s1, s2;
};
__device__ __forceinline__ void side_turn(JointSide& b, V3 angular) { b.q = nudge(b.q, cmul(b.al, mvmul(b.I, angular))); }

// x2 + r2 - x1 - r1
__device__ __forceinline__ V3 side_gap(const JointSide& b) {
    return pair_from2(b.x + b.r) - pair_from1(b.x) - pair_from1(b.r);
}

// the three point-to-point rows
__device__ __forceinline__ void side_translation(JointSide& b, float imsum, bool anyDyn) {
    const M3 U = skew(b.r);
    const M3 A = mmul(mmul(U, b.I), mtranspose(U));
    const M3 K = madd(madd(m3(imsum, 0, 0, 0, imsum, 0, 0, 0, imsum), pair_from1(A)), pair_from2(A));
    const float det = mdet(K);
    if (fabsf(det) > kMachineEps) {
        const M3 Kt = anyDyn ? minv(K, det) : mzero();
        const V3 lam = mvmul(Kt, -side_gap(b));
        const V3 turn = flip3(cross(lam, b.r), b.s2);
        b.x += lock_mul(b.iml, flip3(lam, b.s1));
        side_turn(b, turn);
    }
}

// the three rotation rows of a fixed or slider joint
__device__ __forceinline__ void side_rotation(JointSide& b, Q4 qinit, bool anyDyn) {
    M3 Kr = madd(pair_from1(b.I), pair_from2(b.I));
    const float det = mdet(Kr);
    if (fabsf(det) > kMachineEps) {
        if (anyDyn) Kr = minv(Kr, det);
        const Q4 qe = qmul(qmul(pair_from2(b.q), qinit), qconj(pair_from1(b.q)));
        const V3 er = 2.0f * v3(qe.x, qe.y, qe.z);
        side_turn(b, flip3(mvmul(Kr, -er), b.s1));
    }
}

// B: the batch's bodies (absolute indices); P: their positions; kind: the joint kind of the slot (uniform)
template <bool STAGED>
__device__ __forceinline__ void jt_solve_position_pair(const DevBodies& B, const PosBodies<STAGED>& P, const DevJoints& J,
                                                       int kind, int j, int side, const JointPos& p) {
    const int b1 = p.bodies.x, bi = side ? p.bodies.y : b1, u = bi - P.base;
    const int fo = P.body_flags(u), fa = fo | P.body_flags((side ? b1 : p.bodies.y) - P.base);
    if (!(fa & BF_ENABLED)) return;
    // only non-linear Gauss-Seidel joints (SolveBallAndSocketJointSystem.cpp:309,
    // SolveFixedJointSystem.cpp:299, SolveHingeJointSystem.cpp:479); the slider system stops at its
    // first Baumgarte joint (SolveSliderJointSystem.cpp:527)
    int fl = p.fl;
    if (fl & JF_BAUMGARTE) return;
    if (kind == JT_SLIDER && J.bfirst && J.srank[j] >= J.bfirst[B.world[b1]]) return;
    const bool anyDyn = (fa & BF_DYNAMIC) != 0;
    const float4 ii = P.ii[u];
    JointSide b;
    b.x = ld3(P.x, u);
    b.q = ldq(P.q, u);
    V3 ll = v3(1.0f, 1.0f, 1.0f);
    b.al = ll;
    if (!(fo & BF_UNIT_LOCKS)) {
        ll = ld3(B.llock, bi);
        b.al = ld3(B.alock, bi);
    }
    b.iml = ii.w * ll;
    b.s1 = side ? 0u : 0x80000000u;
    b.s2 = side ? 0x80000000u : 0u;
    b.I = world_inv_inertia(qmat(b.q), v3(ii.x, ii.y, ii.z));
    b.r = qrot(b.q, p.la - ld3(P.com, u));
    const float ims = ii.w + pair_other(ii.w);
    if (kind == JT_BALLSOCKET) {   // SolveBallAndSocketJointSystem.cpp:312-445
        if (fl & JF_LIMIT) {
            const V3 ru = flip3(unit(b.r), b.s2);
            const V3 r1u = pair_from1(ru), r2u = pair_from2(ru);
            const V3 acb = cross(r1u, r2u);
            const float err = p.lim.x - ref_acosf(dot(r1u, r2u));
            fl = err < 0.0f ? (fl | JF_LOWER_VIOLATED) : (fl & ~JF_LOWER_VIOLATED);
            if (side) J.flags[j] = fl;
            if (fl & JF_LOWER_VIOLATED) {
                const float d = dot(acb, mvmul(b.I, acb));
                const float m = d + pair_other(d);
                const float l = (m > 0.0f ? 1.0f / m : 0.0f) * (-err);
                side_turn(b, flip(l, b.s2) * acb);
            }
        }
        side_translation(b, ims, anyDyn);
    } else if (kind == JT_FIXED) {   // SolveFixedJointSystem.cpp:266-448
        side_translation(b, ims, anyDyn);
        side_rotation(b, p.qinit, anyDyn);
    } else if (kind == JT_HINGE) {   // SolveHingeJointSystem.cpp:444-730
        const V3 a = normalized(qrot(b.q, p.ax));
        const V3 a1 = pair_from1(a), a2 = pair_from2(a);
        const V3 b2v = one_unit_orthogonal(a2);
        const V3 c2v = cross(a2, b2v);
        const V3 bxa = cross(b2v, a1), cxa = cross(c2v, a1);
        if (side) {
            J.a1[j] = f4(a1, 0.f);
            J.b2xa1[j] = f4(bxa, 0.f);
            J.c2xa1[j] = f4(cxa, 0.f);
        }
        if (fl & (JF_LIMIT | JF_MOTOR)) {
            const float ang = hinge_angle(pair_from1(b.q), pair_from2(b.q), p.qinit, a1, p.lim.x, p.lim.y);
            const float le = ang - p.lim.x, ue = p.lim.y - ang;
            fl = le <= 0 ? (fl | JF_LOWER_VIOLATED) : (fl & ~JF_LOWER_VIOLATED);
            fl = ue <= 0 ? (fl | JF_UPPER_VIOLATED) : (fl & ~JF_UPPER_VIOLATED);
            if (side) J.flags[j] = fl;
            if ((fl & JF_LIMIT) && (fl & (JF_LOWER_VIOLATED | JF_UPPER_VIOLATED))) {
                const float imlm_old = J.imlm[j];
                const float d = dot(a1, mvmul(b.I, a1));
                const float m = pair_from1(d) + pair_from2(d);
                if (side) J.imlm[j] = imlm_old > 0.0f ? 1.0f / m : 0.0f;   // reference tests the old value
                if (fl & JF_LOWER_VIOLATED) side_turn(b, flip(imlm_old * (-le), b.s1) * a1);
                if (fl & JF_UPPER_VIOLATED) side_turn(b, flip(imlm_old * (-ue), b.s2) * a1);
            }
        }
        const V3 ib = mvmul(b.I, bxa), ic = mvmul(b.I, cxa);
        const float d11 = dot(bxa, ib), d12 = dot(bxa, ic), d21 = dot(cxa, ib), d22 = dot(cxa, ic);
        const float e11 = d11 + pair_other(d11);
        const float e12 = d12 + pair_other(d12);
        const float e21 = d21 + pair_other(d21);
        const float e22 = d22 + pair_other(d22);
        const float det = e11 * e22 - e21 * e12;
        if (fabsf(det) > kMachineEps) {
            float k00 = 0, k01 = 0, k10 = 0, k11 = 0;
            if (anyDyn) {
                const float id = 1.0f / det;
                k00 = e22 * id; k01 = -e12 * id; k10 = -e21 * id; k11 = e11 * id;
            }
            const float x0 = -dot(a1, b2v), x1 = -dot(a1, c2v);
            const float l0 = k00 * x0 + k01 * x1;
            const float l1 = k10 * x0 + k11 * x1;
            side_turn(b, flip3(bxa, b.s1) * l0 + flip3(cxa, b.s1) * l1);
        }
        side_translation(b, ims, anyDyn);
    } else {   // slider, SolveSliderJointSystem.cpp:514-826
        const V3 u21 = side_gap(b);
        const V3 ax = pair_from1(normalized(qrot(b.q, p.ax)));
        const V3 n1 = one_unit_orthogonal(ax);
        const V3 n2 = cross(ax, n1);
        const float ud = dot(u21, ax);
        fl = (ud - p.lim.x) <= 0 ? (fl | JF_LOWER_VIOLATED) : (fl & ~JF_LOWER_VIOLATED);
        fl = (p.lim.y - ud) <= 0 ? (fl | JF_UPPER_VIOLATED) : (fl & ~JF_UPPER_VIOLATED);
        const V3 arm = side ? b.r : b.r + u21;   // r2, r1 + u
        const V3 m1 = cross(arm, n1), m2 = cross(arm, n2), ma = cross(arm, ax);
        if (side) {
            J.flags[j] = fl;
            J.ra[j] = f4(ma, 0.f);   // read by the next step's limit inverse mass
        }
        if ((fl & JF_LIMIT) && (fl & (JF_LOWER_VIOLATED | JF_UPPER_VIOLATED))) {
            const float d = dot(ma, mvmul(b.I, ma));
            const float m = ims + pair_from1(d) + pair_from2(d);
            const float imlm = m > 0.0f ? 1.0f / m : 0.0f;
            if (side) J.imlm[j] = imlm;
            if (fl & JF_LOWER_VIOLATED) {
                const float l = flip(imlm * (-(dot(side_gap(b), ax) - p.lim.x)), b.s1);
                b.x += lock_mul(b.iml, l * ax);
                side_turn(b, l * ma);
            }
            if (fl & JF_UPPER_VIOLATED) {
                const float l = flip(imlm * (-(p.lim.y - dot(side_gap(b), ax))), b.s2);
                b.x += lock_mul(b.iml, l * ax);
                side_turn(b, l * ma);
            }
        }
        side_rotation(b, p.qinit, anyDyn);
        // 2 translation rows (with u and the cross products from before the corrections above)
        const V3 i1 = mvmul(b.I, m1), i2 = mvmul(b.I, m2);
        const float d11 = dot(m1, i1), d12 = dot(m1, i2), d21 = dot(m2, i1), d22 = dot(m2, i2);
        const float e11 = ims + pair_from1(d11) + pair_from2(d11);
        const float e12 = d12 + pair_other(d12);
        const float e21 = d21 + pair_other(d21);
        const float e22 = ims + pair_from1(d22) + pair_from2(d22);
        const float det = e11 * e22 - e21 * e12;
        if (fabsf(det) > kMachineEps) {
            float k00 = 0, k01 = 0, k10 = 0, k11 = 0;
            if (anyDyn) {
                const float id = 1.0f / det;
                k00 = e22 * id; k01 = -e12 * id; k10 = -e21 * id; k11 = e11 * id;
            }
            const float t0 = -dot(u21, n1), t1 = -dot(u21, n2);
            const float l0 = k00 * t0 + k01 * t1;
            const float l1 = k10 * t0 + k11 * t1;
            b.x += lock_mul(b.iml, flip3(n1, b.s1) * l0 + flip3(n2, b.s1) * l1);
            side_turn(b, flip3(m1, b.s1) * l0 + flip3(m2, b.s1) * l1);
        }
    }
    P.x[u] = f4(b.x, STAGED ? __int_as_float(fo) : 0.f);
    P.q[u] = f4q(b.q);
}

}  // namespace rp3dg
