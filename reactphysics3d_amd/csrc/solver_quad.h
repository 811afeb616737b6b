// Contact sweeps with four lanes per manifold.
//
// ContactSolverSystem::solve (CS.cpp:479-759) is one long dependent chain per manifold: the points one
// after another, each a velocity row and a split-impulse row, then two friction rows and the twist, all
// over the velocities of two bodies.  A colour of one world seldom fills a wavefront, so the length of
// that chain in instructions, not the number of lanes, sets the time of a colour.  The four lanes of a
// quad share it:
//
//   lane 0: body 1, velocities         lane 2: body 1, split velocities
//   lane 1: body 2, velocities         lane 3: body 2, split velocities
//
// The velocity row and the split row of a point have the same form (they differ in the bias and in the
// velocities they read), and what a row does to body 1 it does to body 2 with the opposite sign, so the
// quad runs one instruction stream.  Lanes exchange by DPP quad permutations.  Every value is computed by
// the same FP32 operations in the same order as the reference's; the sign of body 1 is applied to the
// impulse by flipping its sign bit (x + (-y) is x - y, and (-a) * b is -(a * b), exactly).
//
// The rows are loaded once per quad: lane k loads point k's normal and depth, lanes of one side load the
// lever arms of its points, and lane k one of (t1, t2, normal, impulses); the broadcasts are DPP moves.
//
// Issue per manifold of four points: about 520 vector instructions instead of 1,300 on one lane.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "kcommon.h"
#include "rp3d_internal.h"
#include "solver_dev.h"

namespace rp3dg {

// Where the body state of a sweep lives.
//   STATE_LDS: velocities, inertia rows and flags in LDS, 100 B a body; the third inertia row rides in the
//              w lanes of cw, sv and sw
//   STATE_VEL: velocities in LDS, 48 B a body, the split angular velocity in the w lanes of cv, cw and sv;
//              inertia rows and flags in HBM
//   STATE_HBM: everything in HBM
constexpr int STATE_LDS = 0, STATE_VEL = 1, STATE_HBM = 2;

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, true));
}
constexpr int kQuadFrom1 = 0 | 0 << 2 | 2 << 4 | 2 << 6;   // body 1's lane of the same half
constexpr int kQuadFrom2 = 1 | 1 << 2 | 3 << 4 | 3 << 6;   // body 2's lane of the same half
constexpr int kQuadOther = 1 | 0 << 2 | 3 << 4 | 2 << 6;   // the other body's lane of the same half
constexpr int kQuadLow = 0 | 1 << 2 | 0 << 4 | 1 << 6;     // the velocity lane of the same body
constexpr int kQuadHigh = 2 | 3 << 2 | 2 << 4 | 3 << 6;    // the split lane of the same body
template <int K>
__device__ __forceinline__ float quad_lane(float x) { return dpp<K | K << 2 | K << 4 | K << 6>(x); }
template <int K>
__device__ __forceinline__ V3 quad_lane3(float4 x) { return v3(quad_lane<K>(x.x), quad_lane<K>(x.y), quad_lane<K>(x.z)); }

// What one lane loads of a manifold's row.
struct QuadRow {
    float4 pn;       // point k's normal and depth (lane k)
    float4 ra, rb;   // lever arms of this side's body: points 0 and 2 (velocity lanes), 1 and 3 (split lanes)
    float4 ia, ib;   // inverse inertia x (lever arm x normal) of the same points
    float4 rf;       // friction lever arm, w: inverse mass
    float4 tn;       // t1 | t2 | normal, friction coefficient | impulses, inverse twist mass (lane k)
};

// Row pointers of a lane (they depend only on its place in the quad).
struct QuadSrc {
    const float4 *pn, *r, *in, *rf, *tn;
    int sub, side, part;
    unsigned int smask;   // sign bit for body 1
    __device__ __forceinline__ QuadSrc(const DevSolver& S, int lane) {
        sub = lane & 3;
        side = lane & 1;
        part = sub >> 1;
        pn = S.pn;
        r = side ? S.r2 : S.r1;
        in = side ? S.i2 : S.i1;
        rf = side ? S.r2f : S.r1f;
        tn = sub == 0 ? S.t1 : (sub == 1 ? S.t2 : (sub == 2 ? S.n : S.imp));
        smask = side ? 0u : 0x80000000u;
    }
    // points beyond the manifold's np repeat its last one (and are not used): no lane is masked off
    __device__ __forceinline__ void load(int i, int np, QuadRow& R) const {
        const int last = np - 1;
        const size_t o = 4 * (size_t)i, a = o + min(part, last), b = o + min(part + 2, last);
        R.pn = pn[o + min(sub, last)];
        R.ra = r[a];
        R.rb = r[b];
        R.ia = in[a];
        R.ib = in[b];
        R.rf = rf[i];
        R.tn = tn[i];
    }
};

// Velocities and inertia of the lane's body.
struct QuadBody {
    V3 V, W;
    M3 I;
    float im;
    V3 ll, al;   // lock factors (LK only)
};

__device__ __forceinline__ float flip(float x, unsigned int mask) { return __uint_as_float(__float_as_uint(x) ^ mask); }

// rel_vel (v2 + w2 x r2 - v1 - w1 x r1 in the reference's order), valid in body 2's lanes
__device__ __forceinline__ V3 quad_rel_vel(V3 V, V3 W, V3 r) {
    const float ax = W.y * r.z, bx = W.z * r.y, ay = W.z * r.x, by = W.x * r.z, az = W.x * r.y, bz = W.y * r.x;
    const float tx = V.x + ax - bx, ty = V.y + ay - by, tz = V.z + az - bz;
    return v3(tx - dpp<kQuadFrom1>(V.x) - dpp<kQuadFrom1>(ax) + dpp<kQuadFrom1>(bx),
              ty - dpp<kQuadFrom1>(V.y) - dpp<kQuadFrom1>(ay) + dpp<kQuadFrom1>(by),
              tz - dpp<kQuadFrom1>(V.z) - dpp<kQuadFrom1>(az) + dpp<kQuadFrom1>(bz));
}

template <int P, bool LK, bool SPLIT>
__device__ __forceinline__ void quad_point(const QuadSrc& Q, const QuadRow& R, QuadBody& b, float& lam, float& sum_pen,
                                           float beta_dt) {
    const V3 n = quad_lane3<P>(R.pn);
    const float depth = quad_lane<P>(R.pn.w);
    constexpr int kFrom = (P & 1) ? kQuadHigh : kQuadLow;
    const float4 rr = P < 2 ? R.ra : R.rb;
    const V3 r = v3(dpp<kFrom>(rr.x), dpp<kFrom>(rr.y), dpp<kFrom>(rr.z));
    const float rw = dpp<kFrom>(rr.w);   // body 1: inverse penetration mass, body 2: restitution bias
    const float4 ii = P < 2 ? R.ia : R.ib;
    const V3 in = v3(dpp<kFrom>(ii.x), dpp<kFrom>(ii.y), dpp<kFrom>(ii.z));
    const V3 dv = quad_rel_vel(b.V, b.W, r);
    const float Jv = dv.x * n.x + dv.y * n.y + dv.z * n.z;
    float bias_pen = 0.0f;
    if (depth > 0.01f) bias_pen = -(beta_dt) * fmax_s(0.0f, depth - 0.01f);
    const float ipm = dpp<kQuadFrom1>(rw);
    const float bias = SPLIT ? (Q.part ? bias_pen : rw) : bias_pen + rw;
    float dl = -(Jv + bias) * ipm;
    const float lt = lam;
    lam = fmax_s(lt + dl, 0.0f);
    dl = lam - lt;
    const float dls = flip(dpp<kQuadFrom2>(dl), Q.smask);
    b.V.x += lk<LK>(b.im * (n.x * dls), b.ll.x);
    b.V.y += lk<LK>(b.im * (n.y * dls), b.ll.y);
    b.V.z += lk<LK>(b.im * (n.z * dls), b.ll.z);
    b.W.x += lk<LK>(in.x, b.al.x) * dls;
    b.W.y += lk<LK>(in.y, b.al.y) * dls;
    b.W.z += lk<LK>(in.z, b.al.z) * dls;
    sum_pen += lam;
}

// One friction row: direction t, inverse mass m, accumulated impulse imp, limit lim.
template <bool LK>
__device__ __forceinline__ void quad_friction(const QuadSrc& Q, QuadBody& b, V3 t, float m, V3 rf, float lim, float& imp) {
    const V3 dv = quad_rel_vel(b.V, b.W, rf);
    const float Jv = dv.x * t.x + dv.y * t.y + dv.z * t.z;
    float dl = -Jv * m;
    const float lt = imp;
    imp = fmax_s(-lim, fmin_s(lt + dl, lim));
    dl = imp - lt;
    const float dls = flip(dpp<kQuadFrom2>(dl), Q.smask);
    const V3 rct = cross(rf, t);
    const V3 a = v3(rct.x * dls, rct.y * dls, rct.z * dls);
    b.V.x += lk<LK>(b.im * (t.x * dls), b.ll.x);
    b.V.y += lk<LK>(b.im * (t.y * dls), b.ll.y);
    b.V.z += lk<LK>(b.im * (t.z * dls), b.ll.z);
    const V3 aw = lkv<LK>(b.al, mvmul(b.I, a));
    b.W.x += aw.x; b.W.y += aw.y; b.W.z += aw.z;
}

// The sweep of one manifold by its quad.  lam: this half's impulses of the four points; imp: friction 1,
// friction 2, twist (both valid in body 2's lanes).  store_split() is called after the points, when the
// split lanes hold their final velocities; the caller stores the velocity lanes' afterwards.
template <bool LK, bool SPLIT, class StoreSplit>
__device__ __forceinline__ void quad_solve(const QuadSrc& Q, const QuadRow& R, int np, QuadBody& b, float4& lam, V3& imp,
                                           float beta_dt, StoreSplit store_split) {
    float sum_pen = 0.0f;
    if (np > 0) quad_point<0, LK, SPLIT>(Q, R, b, lam.x, sum_pen, beta_dt);
    if (np > 1) quad_point<1, LK, SPLIT>(Q, R, b, lam.y, sum_pen, beta_dt);
    if (np > 2) quad_point<2, LK, SPLIT>(Q, R, b, lam.z, sum_pen, beta_dt);
    if (np > 3) quad_point<3, LK, SPLIT>(Q, R, b, lam.w, sum_pen, beta_dt);
    store_split();
    const V3 rf = xyz(R.rf);
    const float mu = quad_lane<2>(R.tn.w);
    const float lim = mu * sum_pen;
    quad_friction<LK>(Q, b, quad_lane3<0>(R.tn), quad_lane<0>(R.tn.w), rf, lim, imp.x);
    quad_friction<LK>(Q, b, quad_lane3<1>(R.tn), quad_lane<1>(R.tn.w), rf, lim, imp.y);
    // twist
    const V3 n = quad_lane3<2>(R.tn);
    const V3 dw = v3(b.W.x - dpp<kQuadFrom1>(b.W.x), b.W.y - dpp<kQuadFrom1>(b.W.y), b.W.z - dpp<kQuadFrom1>(b.W.z));
    const float Jv = dw.x * n.x + dw.y * n.y + dw.z * n.z;
    float dl = -Jv * quad_lane<3>(R.tn.w);
    const float lt = imp.z;
    imp.z = fmax_s(-lim, fmin_s(lt + dl, lim));
    dl = dpp<kQuadFrom2>(imp.z - lt);
    const V3 aw = lkv<LK>(b.al, mvmul(b.I, v3(n.x * dl, n.y * dl, n.z * dl)));
    b.W.x += flip(aw.x, Q.smask); b.W.y += flip(aw.y, Q.smask); b.W.z += flip(aw.z, Q.smask);
}

// Loads the lane's body (index u into the state arrays, absolute index b), solves, and stores it back when
// it is dynamic.  A: the sweep's arrays (A.B's velocity arrays as STATE says).
template <int STATE, bool LK, bool SPLIT>
__device__ __forceinline__ void quad_sweep(const SvArgs& A, const QuadSrc& Q, const QuadRow& R, int u, int b, int np,
                                           float4& lam, V3& imp, float beta_dt) {
    const DevBodies& B = A.B;
    QuadBody q;
    const int flags = B.flags[u];
    if constexpr (STATE == STATE_LDS) {
        q.V = Q.part ? ld3(B.sv, u) : ld3(B.cv, u);
        q.W = Q.part ? ld3(B.sw, u) : ld3(B.cw, u);
        q.I.r[0] = ld3(B.iw0, u);
        q.I.r[1] = ld3(B.iw1, u);
        q.I.r[2] = v3(B.cw[u].w, B.sv[u].w, B.sw[u].w);
    } else if constexpr (STATE == STATE_VEL) {
        const float4 cv = B.cv[u], cw = B.cw[u], sv = B.sv[u];
        q.V = Q.part ? xyz(sv) : xyz(cv);
        q.W = Q.part ? v3(cv.w, cw.w, sv.w) : xyz(cw);
        q.I.r[0] = ld3(B.iw0, u);
        q.I.r[1] = ld3(B.iw1, u);
        q.I.r[2] = ld3(B.iw2, u);
    } else {
        q.V = Q.part ? ld3(B.sv, u) : ld3(B.cv, u);
        q.W = Q.part ? ld3(B.sw, u) : ld3(B.cw, u);
        q.I.r[0] = ld3(B.iw0, u);
        q.I.r[1] = ld3(B.iw1, u);
        q.I.r[2] = ld3(B.iw2, u);
    }
    q.im = R.rf.w;
    q.ll = q.al = v3(1.0f, 1.0f, 1.0f);
    if constexpr (LK) {
        if (!(flags & BF_UNIT_LOCKS)) {
            q.ll = ld3(B.llock, b);
            q.al = ld3(B.alock, b);
        }
    }
    const bool dyn = (flags & BF_DYNAMIC) != 0;
    quad_solve<LK, SPLIT>(Q, R, np, q, lam, imp, beta_dt, [&]() {
        if (SPLIT && Q.part && dyn) {
            st3(B.sv, u, q.V);
            if constexpr (STATE == STATE_VEL) {
                B.cv[u].w = q.W.x;
                B.cw[u].w = q.W.y;
                B.sv[u].w = q.W.z;
            } else {
                st3(B.sw, u, q.W);
            }
        }
    });
    if (!Q.part && dyn) {
        st3(B.cv, u, q.V);
        st3(B.cw, u, q.W);
    }
}

// A manifold whose row state (impulses, bodies, points) lives in HBM: the per-colour kernels, and rows of
// the fused solver beyond its LDS.
template <int STATE, bool SPLIT>
__device__ __forceinline__ void quad_sweep_row(const SvArgs& A, const QuadSrc& Q, int i, float beta_dt) {
    const DevSolver& S = A.S;
    const int2 bb = S.bodies[i];
    const int np = S.npts[i];
    QuadRow R;
    Q.load(i, 4, R);   // (all four slots, so that these loads do not wait for np; a row's slots share a line)
    const int b = Q.side ? bb.y : bb.x, u = b - A.B.vbase;
    float4 lam = S.lq[2 * (size_t)i + Q.part];
    V3 imp = ld3(S.imp, i);
    if (body_flags(A.B, bb.x) & body_flags(A.B, bb.y) & BF_UNIT_LOCKS)
        quad_sweep<STATE, false, SPLIT>(A, Q, R, u, b, np, lam, imp, beta_dt);
    else
        quad_sweep<STATE, true, SPLIT>(A, Q, R, u, b, np, lam, imp, beta_dt);
    if (Q.side) {
        if (SPLIT || !Q.part) S.lq[2 * (size_t)i + Q.part] = lam;
        if (!Q.part) st3(S.imp, i, imp);
    }
}

// ContactSolverSystem::warmStart (CS.cpp:326-476) of row i by its quad: lane k loads point k and one of
// (t1, t2, normal, impulses), the lanes of one side add up their body's velocities (both halves alike, the
// velocity lanes store).  On one lane a manifold's points were loaded one after another behind its number of
// points: 16 us a colour (65,536-body heap) and 13 us (6,000 hulls).
__device__ __forceinline__ void quad_warmstart(const SvArgs& A, const QuadSrc& Q, int i) {
    const DevBodies& B = A.B;
    const DevSolver& S = A.S;
    const int2 bb = S.bodies[i];
    const int np = S.npts[i];
    const size_t o = 4 * (size_t)i;
    const float4 pn = Q.pn[o + Q.sub], lam4 = S.lam[o + Q.sub];
    const float4 ra = Q.in[o + Q.part], rb = Q.in[o + Q.part + 2];
    const float4 tn = Q.tn[i], rf4 = Q.rf[i];
    const float4 ot1 = S.oldt1[i], ot2 = S.oldt2[i];
    const int b = Q.side ? bb.y : bb.x, u = b - B.vbase;
    const int flags = B.flags[u];
    V3 v = ld3(B.cv, u), w = ld3(B.cw, u);
    const M3 I = body_iw(B, b);
    V3 ll, al;
    body_locks(B, b, ll, al);
    const float im = rf4.w;
    // this lane's point: resting (its cached impulse), new (a learned one, or none) or absent
    const bool resting = Q.sub < np && lam4.z != 0.0f, fresh = Q.sub < np && !resting && A.learned;
    float lam = resting ? lam4.x : 0.0f;
    float4 pr = make_float4(0.f, 0.f, 0.f, 0.f);
    if (fresh) {
        pr = S.pred[o + Q.sub];
        lam = fmax_s(pr.x, 0.0f);
    }
    const float kind = resting ? 1.0f : (fresh ? 2.0f : 0.0f);
    bool any = false;
    float plx = 0.0f, ply = 0.0f;   // learned friction impulses summed over the new points
    float4 lq;
    auto point = [&](auto P, float4 in4) {
        constexpr int K = decltype(P)::value, kFrom = (K & 1) ? kQuadHigh : kQuadLow;
        const float l = quad_lane<K>(lam), k = quad_lane<K>(kind);
        const V3 n = quad_lane3<K>(pn);
        const V3 in = v3(dpp<kFrom>(in4.x), dpp<kFrom>(in4.y), dpp<kFrom>(in4.z));
        const float py = quad_lane<K>(pr.y), pz = quad_lane<K>(pr.z);
        if (k != 0.0f) {
            if (k == 1.0f) any = true;
            else {
                plx += py;
                ply += pz;
            }
            const float ls = flip(l, Q.smask);
            v.x += im * (n.x * ls) * ll.x; v.y += im * (n.y * ls) * ll.y; v.z += im * (n.z * ls) * ll.z;
            w.x += in.x * al.x * ls; w.y += in.y * al.y * ls; w.z += in.z * al.z * ls;
        }
        return l;
    };
    lq.x = point(std::integral_constant<int, 0>{}, ra);
    lq.y = point(std::integral_constant<int, 1>{}, ra);
    lq.z = point(std::integral_constant<int, 2>{}, rb);
    lq.w = point(std::integral_constant<int, 3>{}, rb);
    float4 imp = make_float4(quad_lane<3>(tn.x), quad_lane<3>(tn.y), quad_lane<3>(tn.z), quad_lane<3>(tn.w));
    const V3 t1 = quad_lane3<0>(tn), t2 = quad_lane3<1>(tn), n = quad_lane3<2>(tn);
    // learned friction only for a manifold with no resting point (the reference then starts from zero)
    if (any || (A.learned && np > 0)) {
        if (any) {
            const V3 oi = v3(imp.x * ot1.x + imp.y * ot2.x, imp.x * ot1.y + imp.y * ot2.y, imp.x * ot1.z + imp.y * ot2.z);
            imp.x = dot(oi, t1);
            imp.y = dot(oi, t2);
        } else {
            imp.x = plx;
            imp.y = ply;
            imp.z = 0.0f;
        }
        const V3 rf = xyz(rf4);
        const V3 rct1 = cross(rf, t1), rct2 = cross(rf, t2);
        const float s1 = flip(imp.x, Q.smask), s2 = flip(imp.y, Q.smask), s3 = flip(imp.z, Q.smask);
        v += cmul(im * v3(t1.x * s1, t1.y * s1, t1.z * s1), ll);
        w += cmul(al, mvmul(I, v3(rct1.x * s1, rct1.y * s1, rct1.z * s1)));
        v += cmul(im * v3(t2.x * s2, t2.y * s2, t2.z * s2), ll);
        w += cmul(al, mvmul(I, v3(rct2.x * s2, rct2.y * s2, rct2.z * s2)));
        w += cmul(al, mvmul(I, v3(n.x * s3, n.y * s3, n.z * s3)));
        // the reference applies the twist impulse a second time (CS.cpp:457-466)
        const V3 tw = cmul(al, mvmul(I, v3(n.x * imp.z, n.y * imp.z, n.z * imp.z)));
        w += v3(flip(tw.x, Q.smask), flip(tw.y, Q.smask), flip(tw.z, Q.smask));
    } else {
        imp.x = imp.y = imp.z = 0.0f;
    }
    if (Q.part) {
        if (Q.side) S.imp[i] = imp;
        else S.lq[2 * (size_t)i + 1] = make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    if (!Q.side) S.lq[2 * (size_t)i] = lq;
    if (flags & BF_DYNAMIC) {
        st3(B.cv, u, v);
        st3(B.cw, u, w);
    }
}

}  // namespace rp3dg
