// Fused per-world solver for batches of many small worlds.
//
// sv_setup integrates the velocities and writes the contact and joint rows of the
// whole batch.  Then one workgroup owns one group of consecutive worlds for the
// sweeps: warm start, every velocity iteration (colours and joint slots separated
// by workgroup barriers), impulse store; a third kernel does position
// integration, the joint position iterations, the state update and the
// fat-AABB refit.  Groups share nothing, so no grid-wide synchronisation and no
// per-colour launches are needed.  Colour c of a group is colour c of each of
// its worlds side by side (worlds share no body), so every world runs its
// sweeps in the same order as the per-colour kernels (joint slots, then contact
// colours) and results are identical; packing worlds fills the wavefronts of
// the colour phases, which a single small world leaves mostly idle.
//
// In residual mode a world iterates until the velocity residual
//   r_k = max over its dynamic bodies of max(|dv|_inf, |dw|_inf) between sweeps
// drops below the threshold (or the iteration cap is reached); a converged
// world of a group skips the remaining sweeps of the others.  This mode has no
// counterpart in the reference, which always runs a fixed iteration count
// (PhysicsWorld.cpp:334).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fused.h"
#include "joints_dev.h"
#include "kcommon.h"
#include "refit_dev.h"
#include "solver_dev.h"
#include "solver_quad.h"

namespace rp3dg {

__device__ __forceinline__ float block_maxf(float v, float* red) {
    v = wave_maxf(v);
    const int wid = threadIdx.x / kWave;
    const int nwv = blockDim.x / kWave;
    if (lane_id() == 0) red[wid] = v;
    __syncthreads();
    float r = red[0];
    for (int k = 1; k < nwv; k++) r = red[k] > r ? red[k] : r;
    __syncthreads();
    return r;
}

// Start of the solver phase, over the whole batch at once: inverse world inertia tensors and velocity
// integration of every body (PhysicsWorld.cpp:266-272), contact rows (ContactSolverSystem::init), joint
// rows (ConstraintSolverSystem::initialize).  The three parts share no data: the rows recompute the inertia
// of their bodies instead of waiting for the integration to store it, which saves a launch or a barrier
// and lets a single large world use the whole chip here.
__global__ __launch_bounds__(256) void sv_setup(SvArgs A, DevJoints J, Settings settings, float dt) {
    const DevBodies& B = A.B;
    const int nm = *A.nm;
    const int jw = (J.n + kWave - 1) & ~(kWave - 1), mw = (nm + kWave - 1) & ~(kWave - 1);   // whole wavefronts each
    const int total = jw + mw + B.n;
    RP3DG_GRID_STRIDE(t, total) {
        if (t < jw) {
            if (t < J.n) jt_init_one(B, J, t, dt);
        } else if (t < jw + mw) {
            if (t - jw < nm) sv_prepare_one(A, t - jw);
        } else {
            dyn_integrate_velocities_one(B, settings, dt, t - jw - mw);
        }
    }
}

// Feature rows of the points without a cached impulse (learned warm start, sample log), after sv_setup.
__global__ __launch_bounds__(256) void sv_features(FusedArgs F) {
    const SvArgs& A = F.A;
    const int nm = *A.nm;
    const int lane = lane_id();
    for (int base = (blockIdx.x * blockDim.x + threadIdx.x) & ~(kWave - 1); base < nm; base += gridDim.x * blockDim.x) {
        const int i = base + lane;
        int k = 0;
        if (i < nm) {
            const int np = A.S.npts[i];
            for (int p = 0; p < np; p++) k += A.S.lam[4 * i + p].z == 0.0f ? 1 : 0;
        }
        const int incl = wave_incl_scan(k);
        int start = 0;
        if (lane == kWave - 1 && incl > 0) start = atomicAdd(F.nrows, incl);
        start = __shfl(start, kWave - 1, kWave) + incl - k;
        if (i < nm) {
            const int np = A.S.npts[i];
            for (int p = 0; p < np; p++) {
                const int q = 4 * i + p;
                if (A.S.lam[q].z != 0.0f) continue;
                A.S.pred[q] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (start < F.feat_cap) {
                    float f[kFeatures];
                    sv_point_features(A, i, p, f);
                    for (int e = 0; e < kFeatures; e++) F.feats[(size_t)start * kFeatures + e] = f[e];
                    F.row_slot[start] = q;
                }
                start++;
            }
        }
    }
}

// Barrier between two phases of a group.  With the body state in LDS only LDS is shared between threads
// (a row is always solved by the same quad, a joint by the same thread), so loads and stores to HBM stay
// in flight across it.
template <int STATE>
__device__ __forceinline__ void phase_barrier() {
    if constexpr (STATE == STATE_HBM) {
        __syncthreads();
    } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
}

// The kernel's arguments, read again from the kernel argument segment.  The sweeps name some sixty arrays;
// kept in registers over the whole iteration they exceed the scalar registers and spill, so each phase
// reads the pointers it needs (scalar loads that hit the constant cache).
__device__ __forceinline__ const FusedArgs& phase_args() {
    auto p = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const FusedArgs*)p;
}

// Thread index of a phase from the wavefront's number, computed anew (two instructions) so that it is not
// kept in a register, or spilled, across the other phases.
__device__ __forceinline__ int phase_thread(int wave) {
    int zero = 0;
    asm volatile("" : "+v"(zero));
    return wave * kWave + (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, (unsigned)zero));
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ unsigned long long uniform(unsigned long long x) {
    return (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(x >> 32)) << 32 |
           (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)x);
}

// Tables that no kernel writes, read through the scalar cache.
template <class T>
using Table = const __attribute__((address_space(4))) T*;
template <class T>
__device__ __forceinline__ Table<T> table(const T* p) { return (Table<T>)(uintptr_t)p; }

// Calls f(arguments, segment, all) for the segments of this wavefront's strands of group g, or of the whole
// group's (all); ends with a barrier if there were any.
template <int STATE, class F>
__device__ __forceinline__ void joint_strands(int g, int wave, int waves, F&& f) {
    const FusedArgs& P = phase_args();
    const Table<int> st = table(P.jt_strands) + (size_t)g * kJointStrands;
    const int first = st[0];
    if (first == st[kJointStrands]) return;
    const bool all = table(&P.jt_segs[first].w)[0] != 0;
    for (int s = all ? 0 : wave; s < (all ? 1 : kJointStrands); s += waves) {
        const int end = st[s + 1];
        for (int k = st[s]; k < end; k++) {
            const FusedArgs& FP = phase_args();
            const Table<int> e = table(&FP.jt_segs[k].x);
            const int4 r = make_int4(e[0], e[1], e[2], 0);
            f(FP, r, all);
            if (all) phase_barrier<STATE>();
            else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
    if (!all) phase_barrier<STATE>();
}

// Header of a row: bodies relative to the group's first (14 bits each), points (3 bits).
__device__ __forceinline__ unsigned int row_header(int u1, int u2, int np) {
    return (unsigned)u1 | (unsigned)u2 << 14 | (unsigned)np << 28;
}
__device__ __forceinline__ int header_points(unsigned int h) { return (int)(h >> 28); }

// Warm start, velocity iterations and impulse store of one group of worlds.  The body state is in LDS or
// HBM as STATE says (solver_quad.h).  When the group has at most F.lds_rows manifolds and only unit lock
// factors (`fast`), the accumulated impulses and the headers of its rows are in LDS too: the sweeps then
// read the constant part of a row (up to 416 B) from HBM and write nothing there, and the next row is
// loaded while the current one is solved.  (The two cases are separate code: a pointer that may be either
// becomes a flat access, which waits for every load in flight.)
template <bool SPLIT, int STATE>
__global__ __launch_bounds__(kFusedMaxBlock) void sv_world_solve(FusedArgs F) {
    __shared__ float red[16];
    __shared__ unsigned int s_wres[kGroupMaxWorlds];   // residual of each world of the group (float bits)
    __shared__ unsigned long long s_done;               // converged worlds of the group
    __shared__ int s_seg[kMaxColors + 1];               // first row of each colour
    extern __shared__ float4 s_dyn[];   // STATE_LDS: [lds_bodies] cv, cw, sv, sw, iw0, iw1, flags; STATE_VEL: cv,
                                        // cw, sv; then [lds_rows] impulses (velocity half, split half: two each)
                                        // and (friction impulses, header)
    const DevBodies& B = F.A.B;
    const int g = F.block_world[blockIdx.x];
    const int tid = threadIdx.x, nt = blockDim.x;
    const int w0 = F.gworld[g], ngw = F.gworld[g + 1] - w0;
    const int b0 = F.wbody[w0], b1 = F.wbody[w0 + ngw], nbw = b1 - b0;
    const int* seg = F.seg_start + (size_t)g * kMaxColors;
    const int m0 = seg[0], m1 = seg[kMaxColors];
    const int mcap = F.lds_rows;

    // ---------------- staging
    const int L = F.lds_bodies;
    constexpr int kArrays = STATE == STATE_LDS ? 6 : (STATE == STATE_VEL ? 3 : 0);
    float4* s_rows = s_dyn + (size_t)kArrays * L + (STATE == STATE_LDS ? (L + 3) / 4 : 0);
    float4* s_lq = s_rows;              // [2 * row + half]
    float4* s_ih = s_rows + 2 * mcap;   // friction 1, friction 2, twist, header
    for (int k = tid; k <= kMaxColors; k += nt) s_seg[k] = seg[k];
    SvArgs A = F.A;
    DevBodies& BS = A.B;
    if constexpr (STATE == STATE_LDS) {
        float4 *lcv = s_dyn, *lcw = s_dyn + L, *lsv = s_dyn + 2 * L, *lsw = s_dyn + 3 * L;
        float4 *li0 = s_dyn + 4 * L, *li1 = s_dyn + 5 * L;
        int* lfl = reinterpret_cast<int*>(s_dyn + 6 * L);
        for (int i = tid; i < nbw; i += nt) {
            lfl[i] = B.flags[b0 + i] | ((B.world[b0 + i] - w0) << kGroupShift);
            const float4 r2 = B.iw2[b0 + i];
            lcv[i] = B.cv[b0 + i];
            lcw[i] = f4(ld3(B.cw, b0 + i), r2.x);
            lsv[i] = f4(ld3(B.sv, b0 + i), r2.y);
            lsw[i] = f4(ld3(B.sw, b0 + i), r2.z);
            li0[i] = B.iw0[b0 + i];
            li1[i] = B.iw1[b0 + i];
        }
        BS.cv = lcv; BS.cw = lcw; BS.sv = lsv; BS.sw = lsw;
        BS.iw0 = li0; BS.iw1 = li1; BS.iw2 = nullptr;
        BS.flags = lfl;
        BS.vbase = b0;
    } else if constexpr (STATE == STATE_VEL) {
        float4 *lcv = s_dyn, *lcw = s_dyn + L, *lsv = s_dyn + 2 * L;
        for (int i = tid; i < nbw; i += nt) {
            const V3 sw = ld3(B.sw, b0 + i);
            lcv[i] = f4(ld3(B.cv, b0 + i), sw.x);
            lcw[i] = f4(ld3(B.cw, b0 + i), sw.y);
            lsv[i] = f4(ld3(B.sv, b0 + i), sw.z);
        }
        BS.cv = lcv; BS.cw = lcw; BS.sv = BS.sw = lsv;   // (sw: in the w lanes)
        BS.iw0 = B.iw0 + b0; BS.iw1 = B.iw1 + b0; BS.iw2 = B.iw2 + b0;
        BS.flags = B.flags + b0;
        BS.vbase = b0;
    }
    const int ub = b0 - BS.vbase;   // first body of the group in the state arrays
    __syncthreads();
    int nc = 0;   // colours of the group (dense from 0)
    while (nc < kMaxColors && uniform(s_seg[nc]) < m1) nc++;

    // ---------------- warm start: contacts colour by colour (CS.cpp:326-476), then joints slot by slot
    {
        const QuadSrc Q(F.A.S, tid);
        for (int c = 0; c < nc; c++) {
            const int lo = s_seg[c], hi = s_seg[c + 1];
            for (int t = tid; t < 4 * (hi - lo); t += nt) quad_warmstart(A, Q, lo + (t >> 2));
            phase_barrier<STATE>();
        }
    }
    bool unit = true;
    for (int i = tid; i < nbw; i += nt) unit = unit && (BS.flags[ub + i] & BF_UNIT_LOCKS);
    const bool fast = __syncthreads_and(unit && m1 - m0 <= mcap);   // (and the impulses written above are visible)
    if (fast)
        for (int r = tid; r < m1 - m0; r += nt) {
            const int i = m0 + r;
            const int2 bb = F.A.S.bodies[i];
            s_lq[2 * r] = F.A.S.lq[2 * (size_t)i];
            s_lq[2 * r + 1] = F.A.S.lq[2 * (size_t)i + 1];
            s_ih[r] = f4(ld3(F.A.S.imp, i), __uint_as_float(row_header(bb.x - b0, bb.y - b0, F.A.S.npts[i])));
        }
    joint_strands<STATE>(g, uniform(tid / kWave), nt / kWave, [&](const FusedArgs& FP, const int4& r, bool all) {
        for (int j = r.x + (all ? tid : tid & (kWave - 1)); j < r.y; j += all ? nt : kWave) jt_warmstart_one(BS, FP.J, j);
    });
    const bool residual = F.res_thr > 0.0f;
    // residual mode with several worlds: each world stops on its own residual (mask of converged worlds)
    const bool masked = residual && ngw > 1;
    const unsigned long long all = ngw >= 64 ? ~0ull : (1ull << ngw) - 1ull;
    unsigned long long done = 0;
    // world (within the group) of the body at index u of the state arrays
    auto world_of = [&](int u) {
        if constexpr (STATE == STATE_LDS) return (BS.flags[u] >> kGroupShift) & 63;
        else return B.world[u - ub + b0] - w0;
    };
    // velocities after the previous sweep: the thread's first body in registers, the others in HBM
    V3 pv0 = v3(0.f, 0.f, 0.f), pw0 = pv0;
    if (residual) {
        if (tid < nbw) {
            pv0 = ld3(BS.cv, ub + tid);
            pw0 = ld3(BS.cw, ub + tid);
        }
        for (int i = tid + nt; i < nbw; i += nt) {
            F.pv[b0 + i] = BS.cv[ub + i];
            F.pw[b0 + i] = BS.cw[ub + i];
        }
        if (masked)
            for (int k = tid; k < ngw; k += nt) {
                s_wres[k] = 0u;
                F.world_iters[w0 + k] = 0;
                F.world_res[w0 + k] = 0.0f;
            }
    }
    __syncthreads();

    // ---------------- velocity iterations: joints, then contacts (ConstraintSolverSystem, CS.cpp:479-759)
    const int nq = nt >> 2, wave = uniform(tid / kWave);
    // one velocity iteration over the contact rows, colour by colour; FAST: every row's impulses and header
    // are in LDS and every body of the group has unit lock factors.  Rows are contiguous over the colours,
    // so a quad's first row of colour c + 1 is at that colour's start; each quad loads its next row before
    // it solves the current one.
    auto contact_sweep = [&](auto fast_tag) {
        constexpr bool FAST = decltype(fast_tag)::value;
        const DevSolver S = phase_args().A.S;
        const int t0 = phase_thread(wave), qd = t0 >> 2;
        const QuadSrc Q(S, t0);
        auto fetch = [&](int i, QuadRow& R, unsigned int& hd) {
            if constexpr (FAST) {
                hd = __float_as_uint(s_ih[i - m0].w);
            } else {
                const int2 bb = S.bodies[i];
                hd = row_header(bb.x - b0, bb.y - b0, S.npts[i]);
            }
            Q.load(i, header_points(hd), R);
        };
        QuadRow R;
        unsigned int hd = 0;
        int lo = m0, hi = nc ? uniform(s_seg[1]) : m0;
        if (lo + qd < hi) fetch(lo + qd, R, hd);
        for (int c = 0; c < nc; c++) {
            const int hi2 = c + 1 < nc ? uniform(s_seg[c + 2]) : hi;
            int i = lo + qd;
            bool more = true;
            while (more) {
                const QuadRow cur = R;
                const unsigned int h = hd;
                const int ic = i;
                i += nq;
                more = i < hi;
                const int nx = more ? i : hi + qd;
                if (nx < (more ? hi : hi2)) fetch(nx, R, hd);
                if (ic >= hi) continue;
                if (masked && ((done >> world_of(ub + (int)(h & 0x3fffu))) & 1ull)) continue;
                const int rel = (int)((Q.side ? h >> 14 : h) & 0x3fffu);
                float4* lq = FAST ? s_lq + 2 * (ic - m0) + Q.part : S.lq + 2 * (size_t)ic + Q.part;
                float4* ih = FAST ? s_ih + (ic - m0) : S.imp + ic;
                float4 lam = *lq;
                V3 imp = xyz(*ih);
                quad_sweep<STATE, !FAST, SPLIT>(A, Q, cur, ub + rel, b0 + rel, header_points(h), lam, imp, F.beta_dt);
                if (Q.side) {
                    if (SPLIT || !Q.part) *lq = lam;
                    if (!Q.part) st3(ih, 0, imp);
                }
            }
            phase_barrier<STATE>();
            lo = hi;
            hi = hi2;
        }
    };
    int it = 0;
    float res = 0.0f;
    while (it < F.max_iters) {
        joint_strands<STATE>(g, wave, nt / kWave, [&](const FusedArgs& FP, const int4& r, bool all) {
            const int t0 = phase_thread(all ? wave : 0), kind = r.z;
            for (int j = r.x + (t0 >> 1); j < r.y; j += (all ? nt : kWave) >> 1) {
                if (masked && ((done >> world_of(FP.J.bodies[j].x - BS.vbase)) & 1ull)) continue;
                jt_solve_velocity_pair(BS, FP.J, kind, j, t0 & 1, FP.dt);
            }
        });
        if (fast) contact_sweep(std::true_type{});
        else contact_sweep(std::false_type{});
        it++;
        if (residual) {
            float r = 0.0f;
            for (int i = tid; i < nbw; i += nt) {
                if (!(BS.flags[ub + i] & BF_DYNAMIC)) continue;
                int k = 0;
                if (masked) {
                    k = world_of(ub + i);
                    if ((done >> k) & 1ull) continue;
                }
                const V3 v = ld3(BS.cv, ub + i), wv = ld3(BS.cw, ub + i);
                V3 pv = pv0, pw = pw0;
                if (i != tid) {
                    pv = ld3(F.pv, b0 + i);
                    pw = ld3(F.pw, b0 + i);
                    F.pv[b0 + i] = f4(v, 0.f);
                    F.pw[b0 + i] = f4(wv, 0.f);
                } else {
                    pv0 = v;
                    pw0 = wv;
                }
                float d = fabsf(v.x - pv.x);
                d = fmaxf(d, fabsf(v.y - pv.y));
                d = fmaxf(d, fabsf(v.z - pv.z));
                d = fmaxf(d, fabsf(wv.x - pw.x));
                d = fmaxf(d, fabsf(wv.y - pw.y));
                d = fmaxf(d, fabsf(wv.z - pw.z));
                if (masked) atomicMax(&s_wres[k], __float_as_uint(d));   // d >= 0: bit order = value order
                else r = fmaxf(r, d);
            }
            if (!masked) {
                res = block_maxf(r, red);
                if (res < F.res_thr) break;
            } else {
                phase_barrier<STATE>();
                if (tid < kWave) {
                    bool fin = false;
                    if (tid < ngw && !((done >> tid) & 1ull)) {
                        const float rk = __uint_as_float(s_wres[tid]);
                        s_wres[tid] = 0u;
                        fin = rk < F.res_thr;
                        F.world_iters[w0 + tid] = it;
                        F.world_res[w0 + tid] = rk;
                    }
                    const unsigned long long bal = __ballot(fin);
                    if (tid == 0) s_done = done | bal;
                }
                phase_barrier<STATE>();
                done = uniform(s_done);
                if (done == all) break;
            }
        }
    }
    // ---------------- storeImpulses (CS.cpp:763-785) and the solved velocities
    __syncthreads();
    if (fast)
        for (int r = tid; r < m1 - m0; r += nt) {
            const int i = m0 + r;
            F.A.S.lq[2 * (size_t)i] = s_lq[2 * r];
            F.A.S.lq[2 * (size_t)i + 1] = s_lq[2 * r + 1];
            st3(F.A.S.imp, i, xyz(s_ih[r]));
        }
    for (int i = m0 + tid; i < m1; i += nt) sv_store_one(F.A, i);   // row i is this thread's in both loops
    if constexpr (STATE != STATE_HBM) {
        for (int i = tid; i < nbw; i += nt) {
            const float4 cv = BS.cv[i], cw = BS.cw[i], sv = BS.sv[i];
            B.cv[b0 + i] = f4(xyz(cv), 0.f);
            B.cw[b0 + i] = f4(xyz(cw), 0.f);
            B.sv[b0 + i] = f4(xyz(sv), 0.f);
            if constexpr (STATE == STATE_VEL) B.sw[b0 + i] = make_float4(cv.w, cw.w, sv.w, 0.f);
            else B.sw[b0 + i] = f4(ld3(BS.sw, i), 0.f);
        }
    }
    if (!masked)
        for (int k = tid; k < ngw; k += nt) {
            F.world_iters[w0 + k] = it;
            F.world_res[w0 + k] = res;
        }
}
template __global__ void sv_world_solve<true, STATE_LDS>(FusedArgs F);
template __global__ void sv_world_solve<true, STATE_VEL>(FusedArgs F);
template __global__ void sv_world_solve<true, STATE_HBM>(FusedArgs F);
template __global__ void sv_world_solve<false, STATE_LDS>(FusedArgs F);
template __global__ void sv_world_solve<false, STATE_VEL>(FusedArgs F);
template __global__ void sv_world_solve<false, STATE_HBM>(FusedArgs F);

// Position integration, joint position correction, body state and refit of a group of worlds with joints
// (PhysicsWorld.cpp:275-288).  A strand of joints is a chain of short phases, each of them one joint's
// dependent chain for its lanes, so the length of that chain sets the time: two lanes share a joint
// (joints_dev.h), the bodies are staged in LDS, and the next segment's joints are loaded while the current
// ones are solved.  64 joints of 3 kinds (88 bodies), 5 iterations: 181 us with one lane a joint, positions
// in HBM and a barrier after each kind and colour, 119 with two lanes and LDS, 61 with strands; 1024 worlds
// of 8 to 128 bodies: 123, 103, 78.
template <bool STAGED>
__global__ __launch_bounds__(kPositionMaxBlock) void world_position(FusedArgs F) {
    extern __shared__ float4 s_pos[];
    const DevBodies& B = F.A.B;
    const int g = F.block_world[blockIdx.x];
    const int tid = threadIdx.x, nt = blockDim.x;
    const int w0 = F.gworld[g], w1 = F.gworld[g + 1];
    const int b0 = F.wbody[w0], b1 = F.wbody[w1];
    const int c0 = F.wcoll[w0], c1 = F.wcoll[w1];
    const float split_factor = F.settings.split_impulse ? 1.0f : 0.0f;
    for (int i = b0 + tid; i < b1; i += nt) dyn_integrate_positions_one(B, F.dt, i, split_factor);
    PosBodies<STAGED> P;
    if constexpr (STAGED) {
        float4* com = s_pos + 3 * F.lds_bodies;
        P = {s_pos, s_pos + F.lds_bodies, s_pos + 2 * F.lds_bodies, com, nullptr, b0};
        for (int i = b0 + tid; i < b1; i += nt) {   // each thread reads what it wrote
            P.x[i - b0] = f4(ld3(B.cx, i), __int_as_float(B.flags[i]));
            P.q[i - b0] = B.cq[i];
            s_pos[2 * F.lds_bodies + i - b0] = B.ii[i];
            com[i - b0] = B.com[i];
        }
    } else {
        P = {B.cx, B.cq, B.ii, B.com, B.flags, 0};
    }
    __syncthreads();
    const Table<int> st = table(F.jt_strands) + (size_t)g * kJointStrands;
    const int first = st[0];
    if (first != st[kJointStrands]) {
        const Table<int> segs = table(&F.jt_segs[0].x);   // 4 ints each
        const bool all = segs[4 * (size_t)first + 3] != 0;
        const int wave = uniform(tid / kWave), side = tid & 1, step = (all ? nt : kWave) >> 1;
        const int turn = (all ? tid : tid & (kWave - 1)) >> 1;
        for (int s = all ? 0 : wave; s < (all ? 1 : kJointStrands); s += nt / kWave) {
            const int k0 = st[s], k1 = st[s + 1], total = (k1 - k0) * F.settings.pos_iters;
            JointPos next;
            if (total > 0) {
                const Table<int> e = segs + 4 * (size_t)k0;
                next = jt_position_load(F.J, min(e[0] + turn, e[1] - 1), side);
            }
            for (int n = 0, k = k0; n < total; n++) {
                const Table<int> e = segs + 4 * (size_t)k;
                const int last = e[1], kind = e[2];
                JointPos p = next;
                int j = e[0] + turn;
                k = k + 1 < k1 ? k + 1 : k0;
                if (n + 1 < total) {
                    const Table<int> e2 = segs + 4 * (size_t)k;
                    next = jt_position_load(F.J, min(e2[0] + turn, e2[1] - 1), side);
                }
                while (j < last) {   // (rarely more than once: one copy of the code)
                    jt_solve_position_pair(B, P, F.J, kind, j, side, p);
                    j += step;
                    if (j < last) p = jt_position_load(F.J, j, side);
                }
                if (all) phase_barrier<STAGED ? STATE_LDS : STATE_HBM>();
                else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        }
        __syncthreads();
    }
    for (int i = b0 + tid; i < b1; i += nt) {
        if constexpr (STAGED) {
            B.cx[i] = f4(xyz(P.x[i - b0]), 0.f);
            B.cq[i] = P.q[i - b0];
        }
        dyn_update_state_one(B, i);
    }
    __syncthreads();
    // collider transforms and fat AABBs for the next broadphase
    for (int i = c0 + tid; i < c1; i += nt) refit_one(B, F.A.C, F.hull_bounds, 0, i);
}
template __global__ void world_position<true>(FusedArgs F);
template __global__ void world_position<false>(FusedArgs F);

// Positions and state of the bodies of worlds without joints, whatever world they are in.  One thread a body
// over the whole batch, and the colliders after it in a launch of their own: a workgroup per group of worlds
// leaves the chip idle with few groups and waits for its slowest load three times over with many.  1001
// bodies: 30 us in one workgroup, 6 and 7 us in the two launches.
__global__ __launch_bounds__(256) void body_position(DevBodies B, float dt, float split_factor) {
    RP3DG_GRID_STRIDE(i, B.n) {
        dyn_integrate_positions_one(B, dt, i, split_factor);
        dyn_update_state_one(B, i);
    }
}

__global__ void sv_log_samples(FusedArgs F, float* log_feats, float* log_targets, const unsigned long long* logged,
                               long long log_cap) {
    const int n = min(*F.nrows, F.feat_cap);
    const long long base = (long long)*logged;
    RP3DG_GRID_STRIDE(r, n) {
        const long long dst = base + r;
        if (dst >= log_cap) continue;
        const int q = F.row_slot[r], i = q >> 2;
        const float4 imp = F.A.S.imp[i];
        const float inv_np = 1.0f / (float)F.A.S.npts[i];
        for (int e = 0; e < kFeatures; e++) log_feats[dst * kFeatures + e] = F.feats[(size_t)r * kFeatures + e];
        log_targets[dst * 3 + 0] = reinterpret_cast<const float*>(F.A.S.lq)[8 * (size_t)i + (q & 3)];
        log_targets[dst * 3 + 1] = imp.x * inv_np;
        log_targets[dst * 3 + 2] = imp.y * inv_np;
    }
}

__global__ void sv_log_advance(const int* nrows, int feat_cap, unsigned long long* logged, long long log_cap) {
    const long long n = min(*nrows, feat_cap);
    const long long v = (long long)*logged + n;
    *logged = (unsigned long long)(v < log_cap ? v : log_cap);
}

}  // namespace rp3dg
