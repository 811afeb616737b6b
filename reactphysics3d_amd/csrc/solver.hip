// Manifold list, graph colouring and the per-colour solver kernels.
//
// Colouring is Jones-Plassmann with hashed priorities: a manifold takes the
// smallest colour unused by its higher-priority neighbours once they are all
// coloured, which equals sequential greedy colouring in priority order and is
// therefore deterministic.  A launch colours as far as bounded waiting goes,
// nearly always everything; another finds nothing left and returns at once, or
// goes on, and a single-workgroup finisher completes whatever remains, so the
// step needs no host round trip.
#include <hip/hip_runtime.h>

#include "kcommon.h"
#include "rp3d_internal.h"
#include "solver.h"
#include "solver_dev.h"
#include "solver_quad.h"

namespace rp3dg {

// ------------------------------------------------------------------------------------------------
// Integration and per-colour rows (bodies in solver_dev.h)
// ------------------------------------------------------------------------------------------------

__global__ void dyn_integrate_positions(DevBodies B, float dt, float split_factor) {
    RP3DG_GRID_STRIDE(i, B.n) dyn_integrate_positions_one(B, dt, i, split_factor);
}

__global__ void dyn_update_state(DevBodies B) {
    RP3DG_GRID_STRIDE(i, B.n) dyn_update_state_one(B, i);
}

__global__ __launch_bounds__(512) void sv_warmstart(SvArgs A, int color) {
    if (color >= *A.ncolors) return;
    const int lo = A.cstart[color], n = 4 * (A.cstart[color + 1] - lo);
    const QuadSrc Q(A.S, threadIdx.x);
    RP3DG_GRID_STRIDE(t, n) quad_warmstart(A, Q, lo + (t >> 2));
}

// four lanes a manifold (solver_quad.h)
template <bool SPLIT>
__global__ __launch_bounds__(512) void sv_solve_color(SvArgs A, int color, float beta_dt) {
    if (color >= *A.ncolors) return;
    const int lo = A.cstart[color], n = 4 * (A.cstart[color + 1] - lo);
    const QuadSrc Q(A.S, threadIdx.x);
    RP3DG_GRID_STRIDE(t, n) quad_sweep_row<STATE_HBM, SPLIT>(A, Q, lo + (t >> 2), beta_dt);
}
template __global__ void sv_solve_color<true>(SvArgs A, int color, float beta_dt);
template __global__ void sv_solve_color<false>(SvArgs A, int color, float beta_dt);

// The colours from c0 on, one after another in one workgroup: the last colours of a batch have a few rows each,
// and a launch of their own costs twice what the rows do.
template <bool SPLIT>
__global__ __launch_bounds__(4 * kTailRows) void sv_solve_tail(SvArgs A, int c0, float beta_dt) {
    const QuadSrc Q(A.S, threadIdx.x);
    const int c1 = *A.ncolors;
    for (int c = c0; c < c1; c++) {
        const int lo = A.cstart[c], n = 4 * (A.cstart[c + 1] - lo);
        for (int t = threadIdx.x; t < n; t += 4 * kTailRows) quad_sweep_row<STATE_HBM, SPLIT>(A, Q, lo + (t >> 2), beta_dt);
        __syncthreads();
    }
}
template __global__ void sv_solve_tail<true>(SvArgs A, int c0, float beta_dt);
template __global__ void sv_solve_tail<false>(SvArgs A, int c0, float beta_dt);
__global__ __launch_bounds__(4 * kTailRows) void sv_warmstart_tail(SvArgs A, int c0) {
    const QuadSrc Q(A.S, threadIdx.x);
    const int c1 = *A.ncolors;
    for (int c = c0; c < c1; c++) {
        const int lo = A.cstart[c], n = 4 * (A.cstart[c + 1] - lo);
        for (int t = threadIdx.x; t < n; t += 4 * kTailRows) quad_warmstart(A, Q, lo + (t >> 2));
        __syncthreads();
    }
}

__global__ void sv_note_iterations(int* world_iters, float* world_res, int n, int iters) {
    RP3DG_GRID_STRIDE(w, n) {
        world_iters[w] = iters;
        world_res[w] = 0.0f;
    }
}

__global__ void sv_store(SvArgs A) {
    const int nm = *A.nm;
    RP3DG_GRID_STRIDE(i, nm) sv_store_one(A, i);
}

// ------------------------------------------------------------------------------------------------
// Manifold list: pairs with at least one contact point, in pair order
// ------------------------------------------------------------------------------------------------

// a pair's manifolds: its entry, then (concave pairs, xm non-null) its xm tail entries from xs
__global__ void sv_flag_manifolds(const int* ncp, const int* xm, const int* nb_pairs, int* flag) {
    const int np = *nb_pairs;
    RP3DG_GRID_STRIDE(k, np) flag[k] = ncp[k] > 0 ? 1 + (xm ? xm[k] : 0) : 0;
}

__global__ void sv_compact_manifolds(const int* flag, const int* offs, const int* nb_pairs, const int* ncp, const int* xm,
                                     const int* xs, int* list, int* counters_manifolds, int* counters_points,
                                     unsigned long long* total_points) {
    const int np = *nb_pairs;
    if (blockIdx.x == 0 && threadIdx.x == 0) *counters_manifolds = offs[np];
    int pts = 0;
    RP3DG_GRID_STRIDE(k, np) {
        if (flag[k]) {
            list[offs[k]] = k;
            pts += ncp[k];
            for (int j = 1; j < flag[k]; j++) {
                const int slot = xs[k] + j - 1;
                list[offs[k] + j] = slot;
                pts += ncp[slot];
            }
        }
    }
    // one atomic per workgroup: same-address atomics from every wave would serialise in the L2
    __shared__ int s_pts;
    if (threadIdx.x == 0) s_pts = 0;
    __syncthreads();
    pts = wave_sum(pts);
    if (lane_id() == 0 && pts) atomicAdd(&s_pts, pts);
    __syncthreads();
    if (threadIdx.x == 0 && s_pts) {
        atomicAdd(counters_points, s_pts);
        atomicAdd(total_points, (unsigned long long)s_pts);
    }
}

// ------------------------------------------------------------------------------------------------
// body -> manifold adjacency (counts, then fill after a scan)
// ------------------------------------------------------------------------------------------------

__global__ void sv_adj_count(DevBodies B, DevColliders C, DevPairs P, const int* list, const int* nm_ptr, int* cnt) {
    const int nm = *nm_ptr;
    RP3DG_GRID_STRIDE(m, nm) {
        const int2 c = P.col[list[m]];
        const int b1 = C.body[c.x], b2 = C.body[c.y];
        if (dyn_body(B, b1)) atomicAdd(&cnt[b1], 1);
        if (dyn_body(B, b2)) atomicAdd(&cnt[b2], 1);
    }
}

__global__ void sv_adj_fill(DevBodies B, DevColliders C, DevPairs P, const int* list, const int* nm_ptr, const int* offs,
                            int* cursor, int* adj, int2* mb) {
    const int nm = *nm_ptr;
    RP3DG_GRID_STRIDE(m, nm) {
        const int2 c = P.col[list[m]];
        const int b1 = C.body[c.x], b2 = C.body[c.y];
        const int d1 = dyn_body(B, b1) ? b1 : -1;
        const int d2 = dyn_body(B, b2) ? b2 : -1;
        mb[m] = make_int2(d1, d2);
        if (d1 >= 0) adj[offs[d1] + atomicAdd(&cursor[d1], 1)] = m;
        if (d2 >= 0) adj[offs[d2] + atomicAdd(&cursor[d2], 1)] = m;
    }
}

// ------------------------------------------------------------------------------------------------
// Jones-Plassmann colouring
// ------------------------------------------------------------------------------------------------

__device__ __forceinline__ uint32_t prio(uint32_t m) {
    uint32_t x = m * 0x9E3779B1u;
    x ^= x >> 16;
    x *= 0x85EBCA6Bu;
    x ^= x >> 13;
    return x;
}
__device__ __forceinline__ bool higher(uint32_t a, uint32_t b) {  // priority of a > priority of b
    const uint32_t pa = prio(a), pb = prio(b);
    return pa > pb || (pa == pb && a > b);
}

// Tries to colour manifold m (color[m] == -1 while uncoloured).  Returns false when a
// higher-priority neighbour is still uncoloured.  A neighbour coloured concurrently is read either
// as -1 or as its final colour, so the result does not depend on timing.
__device__ __forceinline__ void jp_choose(int m, uint64_t used, int* color, int* status) {
    const uint64_t freem = ~used;
    int c = freem ? __ffsll((unsigned long long)freem) - 1 : 64;
    if (c >= kMaxColors) { atomicOr(status, STATUS_COLOR_OVERFLOW); c = kMaxColors - 1; }
    __atomic_store_n(&color[m], c, __ATOMIC_RELAXED);
}
__device__ __forceinline__ bool jp_try(int m, const int2* mb, const int* offs, const int* adj, int* color, int* status) {
    const int2 bb = mb[m];
    uint64_t used = 0;
    for (int s = 0; s < 2; s++) {
        const int b = s == 0 ? bb.x : bb.y;
        if (b < 0) continue;
        const int e = offs[b + 1];
        for (int k = offs[b]; k < e; k++) {
            const int o = adj[k];
            if (o == m) continue;
            if (higher((uint32_t)o, (uint32_t)m)) {
                const int co = __atomic_load_n(&color[o], __ATOMIC_RELAXED);
                if (co < 0) return false;
                if (co < 64) used |= 1ull << co;
            }
        }
    }
    jp_choose(m, used, color, status);
    return true;
}

// One launch colours as far as the waiting goes; left[0] != 0 afterwards if manifolds are left
// (left_prev: the last launch's, nullptr for the first).
//
// A manifold waits for the neighbours of higher priority, and the longest such chain is some 25 manifolds.
// A launch per link of that chain, each looking at every neighbour of every manifold that is left, took 26 us
// a launch (65,536-body heap, 120,000 manifolds, 25 launches) and 13 us (6,000 hulls, 20).  Here a lane walks
// its manifold's neighbours once, eight at a time, and stays at eight while one of them has no colour yet:
// a link costs a store and a load that reaches it, and one launch does nearly all (114 and 77 us, and an
// empty launch to confirm it).  The lanes of a wavefront step together, so none keeps another from going on, and a wavefront gives up after kColorPolls steps in
// which none of its lanes got further: nothing depends on workgroups running side by side.
constexpr int kColorPolls = 48, kColorChunk = 8;
__global__ __launch_bounds__(256) void sv_color_round(const int2* mb, const int* nm_ptr, const int* offs, const int* adj,
                                                      int* color, const int* left_prev, int* left, int* status) {
    if (left_prev && *left_prev == 0) return;
    const int nm = *nm_ptr;
    bool any_left = false;
    for (int m0 = blockIdx.x * blockDim.x; m0 < nm; m0 += gridDim.x * blockDim.x) {
        const int m = m0 + threadIdx.x;
        bool todo = m < nm && color[m] < 0;
        const int2 bb = todo ? mb[m] : make_int2(-1, -1);
        // both bodies' lists as one: [k1, e1), then [k2, e2)
        int k1 = 0, e1 = 0, k2 = 0, e2 = 0;
        if (bb.x >= 0) { k1 = offs[bb.x]; e1 = offs[bb.x + 1]; }
        if (bb.y >= 0) { k2 = offs[bb.y]; e2 = offs[bb.y + 1]; }
        uint64_t used = 0;
        int wait[kColorChunk];   // neighbours of the current chunk that are waited for, -1: none
        bool fresh = true;
        for (int polls = 0; polls < kColorPolls && __any(todo);) {
            bool moved = false;
            if (todo) {
                if (fresh) {
                    const int n1 = min(kColorChunk, e1 - k1), n = n1 + min(kColorChunk - n1, e2 - k2);
                    moved = true;
                    if (n == 0) {
                        jp_choose(m, used, color, status);
                        todo = false;
                    } else {
                        for (int j = 0; j < kColorChunk; j++) wait[j] = adj[j < n1 ? k1 + j : (n > n1 ? k2 + min(j, n - 1) - n1 : k1 + n1 - 1)];
                        for (int j = 0; j < kColorChunk; j++)
                            if (j >= n || !higher((uint32_t)wait[j], (uint32_t)m)) wait[j] = -1;   // (m itself is not higher)
                        k1 += n1;
                        k2 += n - n1;
                        fresh = false;
                    }
                }
                if (todo) {
                    int co[kColorChunk];
                    for (int j = 0; j < kColorChunk; j++)
                        co[j] = wait[j] >= 0 ? __hip_atomic_load(&color[wait[j]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 64;
                    bool all = true;
                    for (int j = 0; j < kColorChunk; j++) {
                        if (co[j] < 0) { all = false; continue; }
                        if (wait[j] >= 0) moved = true;
                        wait[j] = -1;
                        if (co[j] < 64) used |= 1ull << co[j];
                    }
                    if (all) fresh = moved = true;
                }
            }
            if (!__any(moved)) {
                polls++;
                __builtin_amdgcn_s_sleep(2);
            }
        }
        any_left |= __any(todo) != 0;
    }
    if (any_left && lane_id() == 0) *left = 1;   // (a flag: counting on one address would cost more than the round)
}

// Single workgroup: rounds until every manifold is coloured.  Each round colours at least the
// highest-priority uncoloured manifold, so nm + 1 rounds always suffice.
__global__ __launch_bounds__(1024) void sv_color_finish(const int2* mb, const int* nm_ptr, const int* offs,
                                                        const int* adj, int* color, const int* left_prev, int* rounds,
                                                        int* status) {
    if (left_prev && *left_prev == 0) return;
    __shared__ int left;
    const int nm = *nm_ptr;
    for (int r = 0; r <= nm; r++) {
        if (threadIdx.x == 0) left = 0;
        __syncthreads();
        int mine = 0;
        for (int m = threadIdx.x; m < nm; m += blockDim.x) {
            if (color[m] >= 0) continue;
            if (!jp_try(m, mb, offs, adj, color, status)) mine++;
        }
        if (mine) atomicAdd(&left, mine);
        __syncthreads();
        const int l = left;
        __syncthreads();
        if (l == 0) {
            if (threadIdx.x == 0) *rounds = r + 1;
            return;
        }
    }
    if (threadIdx.x == 0) atomicOr(status, STATUS_COLOR_STALL);
}

// ------------------------------------------------------------------------------------------------
// Colouring per world group (fused layout)
// ------------------------------------------------------------------------------------------------

// The manifold list is in pair-table order (sorted by the lower collider index) and colliders are
// numbered world by world, so the manifolds of a world form one contiguous range.  One pass writes the
// dynamic bodies of every manifold (-1 for static or kinematic) and the first manifold of every world
// (wmstart[nw] = number of manifolds).
__global__ void sv_world_ranges(DevBodies B, DevColliders C, DevPairs P, const int* list, const int* nm_ptr, int nw,
                                int2* mb, int* wmstart) {
    const int nm = *nm_ptr;
    if (nm == 0) {
        RP3DG_GRID_STRIDE(w, nw + 1) wmstart[w] = 0;
        return;
    }
    RP3DG_GRID_STRIDE(m, nm) {
        const int2 c = P.col[list[m]];
        const int b1 = C.body[c.x], b2 = C.body[c.y];
        mb[m] = make_int2(dyn_body(B, b1) ? b1 : -1, dyn_body(B, b2) ? b2 : -1);
        const int w = C.world[c.x];
        const int wp = m ? C.world[P.col[list[m - 1]].x] : -1;
        for (int k = wp + 1; k <= w; k++) wmstart[k] = m;
        if (m == nm - 1)
            for (int k = w + 1; k <= nw; k++) wmstart[k] = nm;
    }
}

// Greedy colouring of a group of worlds: manifolds in order, each the smallest colour unused at either of
// its dynamic bodies; then the rows are placed colour by colour, in manifold order within a colour:
// order[row] = manifold, keys[row] = group * kMaxColors + colour, seg_start[group * kMaxColors + c] = first
// row of colour c of the group.
//
// A manifold's colour depends on the earlier manifolds of its two bodies alone, so it can be chosen as soon
// as it heads both bodies' lists of uncoloured manifolds (kept in manifold order); choosing it makes the
// next manifold of each list a candidate.  Every round colours all manifolds that are ready, and the colours
// are the sequential pass's.  The rounds are as many as the longest chain of manifolds in which each shares
// a body with an earlier one: a few dozen where the sequential pass takes one step per manifold.
// One workgroup per group; bodies' masks and lists, and the manifolds' bodies, in LDS, or (LDS == false,
// groups whose manifolds do not fit) the lists and counts in HBM scratch.
template <bool LDS>
__device__ __forceinline__ void color_group(const ColorArgs& A, char* lds, int b0, int nb, int ma, int nm, int* s_n) {
    const int tid = threadIdx.x, nt = blockDim.x;
    unsigned long long* mask = reinterpret_cast<unsigned long long*>(lds);
    int* head = reinterpret_cast<int*>(mask + nb);
    int* end = head + nb;
    int* work = end + nb;   // [2][nb]
    unsigned int* s_mb = reinterpret_cast<unsigned int*>(work + 2 * nb);
    unsigned int* s_pend = s_mb + nm;
    unsigned short* s_list = reinterpret_cast<unsigned short*>(s_pend + (nm + 15) / 16);
    int* g_list = A.list + 2 * (size_t)ma;
    int* g_pend = A.pend + ma;
    constexpr unsigned int kNone = 0xffffu;
    auto bodies_of = [&](int m) -> unsigned int {   // body 1 | body 2 << 16, relative to the group
        if constexpr (LDS) return s_mb[m];
        const int2 bb = A.mb[ma + m];
        return (bb.x >= 0 ? (unsigned)(bb.x - b0) : kNone) | (bb.y >= 0 ? (unsigned)(bb.y - b0) : kNone) << 16;
    };
    auto list_at = [&](int k) -> int { if constexpr (LDS) return s_list[k]; else return g_list[k]; };
    auto put_list = [&](int k, int m) { if constexpr (LDS) s_list[k] = (unsigned short)m; else g_list[k] = m; };
    for (int i = tid; i < nb; i += nt) {
        mask[i] = 0ull;
        head[i] = 0;
    }
    if (tid < 3) s_n[tid] = 0;
    __syncthreads();
    // lists: count, scan, fill, sort
    for (int m = tid; m < nm; m += nt) {
        unsigned int bb;
        if constexpr (LDS) {
            const int2 g = A.mb[ma + m];
            bb = (g.x >= 0 ? (unsigned)(g.x - b0) : kNone) | (g.y >= 0 ? (unsigned)(g.y - b0) : kNone) << 16;
            s_mb[m] = bb;
        } else {
            bb = bodies_of(m);
        }
        if ((bb & kNone) != kNone) atomicAdd(&head[bb & kNone], 1);
        if (bb >> 16 != kNone) atomicAdd(&head[bb >> 16], 1);
        if constexpr (!LDS) g_pend[m] = ((bb & kNone) != kNone ? 1 : 0) | (bb >> 16 != kNone ? 2 : 0);
    }
    if constexpr (LDS)
        for (int k = tid; k < (nm + 15) / 16; k += nt) s_pend[k] = 0u;
    __syncthreads();
    {
        int carry = 0;
        for (int base = 0; base < nb; base += nt) {
            const int i = base + tid;
            const int c = i < nb ? head[i] : 0;
            int total;
            const int e = block_excl_scan(c, s_n + 8, &total) + carry + c;
            if (i < nb) head[i] = end[i] = e;
            carry += total;
        }
    }
    __syncthreads();
    for (int m = tid; m < nm; m += nt) {
        const unsigned int bb = bodies_of(m);
        if ((bb & kNone) != kNone) put_list(atomicSub(&head[bb & kNone], 1) - 1, m);
        if (bb >> 16 != kNone) put_list(atomicSub(&head[bb >> 16], 1) - 1, m);
        if constexpr (LDS) {
            const unsigned int bits = ((bb & kNone) != kNone ? 1u : 0u) | (bb >> 16 != kNone ? 2u : 0u);
            if (bits) atomicOr(&s_pend[m >> 4], bits << (2 * (m & 15)));
        }
        if (bb == 0xffffffffu) A.color[ma + m] = 0;   // no dynamic body
    }
    __syncthreads();
    // the manifold m became the first uncoloured one of body b: true when it is of both its bodies
    auto arrive = [&](int m, unsigned int b) -> bool {
        const unsigned int bb = bodies_of(m), bit = (bb & kNone) == b ? 1u : 2u;
        if constexpr (LDS) {
            const int sh = 2 * (m & 15);
            const unsigned int left = atomicAnd(&s_pend[m >> 4], ~(bit << sh)) & ~(bit << sh);
            return ((left >> sh) & 3u) == 0u;
        } else {
            return (atomicAnd((unsigned int*)&g_pend[m], ~bit) & ~bit) == 0u;
        }
    };
    for (int b = tid; b < nb; b += nt) {
        const int s = head[b], e = end[b];
        for (int i = s + 1; i < e; i++) {   // insertion sort: lists are short
            const int m = list_at(i);
            int j = i;
            for (; j > s && list_at(j - 1) > m; j--) put_list(j, list_at(j - 1));
            put_list(j, m);
        }
        if (s < e) {
            const int m = list_at(s);
            if (arrive(m, (unsigned)b)) work[atomicAdd(&s_n[0], 1)] = m;
        }
    }
    __syncthreads();
    // rounds.  A ready manifold owns its bodies, so their masks and heads need no atomics; at most one ready
    // manifold per body bounds the work lists.
    for (int round = 0;; round++) {
        const int cur = round % 3, nxt = (round + 1) % 3;
        const int n = s_n[cur];
        if (n == 0) break;
        const int* wl = work + (round & 1) * nb;
        int* wn = work + ((round + 1) & 1) * nb;
        if (tid == 0) s_n[(round + 2) % 3] = 0;
        for (int t = tid; t < n; t += nt) {
            const int m = wl[t];
            const unsigned int bb = bodies_of(m), x = bb & kNone, y = bb >> 16;
            unsigned long long used = 0ull;
            if (x != kNone) used |= mask[x];
            if (y != kNone) used |= mask[y];
            int c = ~used ? __ffsll(~used) - 1 : kMaxColors;
            if (c >= kMaxColors) {
                atomicOr(A.status, STATUS_COLOR_OVERFLOW);
                c = kMaxColors - 1;
            }
            A.color[ma + m] = c;
            for (int k = 0; k < 2; k++) {
                const unsigned int b = k ? y : x;
                if (b == kNone) continue;
                mask[b] |= 1ull << c;
                const int h = head[b] + 1;
                head[b] = h;
                if (h < end[b]) {
                    const int q = list_at(h);
                    if (arrive(q, b)) wn[atomicAdd(&s_n[nxt], 1)] = q;
                }
            }
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(1024) void sv_group_color(ColorArgs A) {
    extern __shared__ char s_color[];
    __shared__ int s_n[8 + 17];          // work list lengths; scan scratch
    __shared__ int s_base[kMaxColors];   // next row of each colour
    __shared__ int s_wave[16][kMaxColors];
    const int g = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
    const int w0 = A.gworld[g], w1 = A.gworld[g + 1];
    const int b0 = A.wbody[w0], nb = A.wbody[w1] - b0;
    const int ma = A.wmstart[w0], nm = A.wmstart[w1] - ma;
    if (tid < kMaxColors) s_base[tid] = 0;
    if (color_body_bytes(nb) + color_manifold_bytes(nm) <= A.lds_bytes && nm <= 0x7fff)
        color_group<true>(A, s_color, b0, nb, ma, nm, s_n);
    else
        color_group<false>(A, s_color, b0, nb, ma, nm, s_n);
    // rows: colour counts, their exclusive prefix, then stable ranks tile by tile (a wavefront's lanes of one
    // colour by ballots, the wavefronts of the tile in order)
    for (int m = tid; m < nm; m += nt) atomicAdd(&s_base[A.color[ma + m]], 1);
    __syncthreads();
    if (tid < kWave) {
        const int cnt = s_base[tid];
        const int base = ma + wave_incl_scan(cnt) - cnt;
        A.seg_start[(size_t)g * kMaxColors + tid] = base;
        s_base[tid] = base;
        const unsigned long long present = __ballot(cnt > 0);
        if (tid == 0 && present) atomicMax(A.ncolors, 64 - __clzll((long long)present));
        if (g == A.ngroups - 1 && tid == 0) A.seg_start[(size_t)A.ngroups * kMaxColors] = A.wmstart[A.gworld[A.ngroups]];
    }
    const int wave = tid / kWave, lane = tid & (kWave - 1), nwave = nt / kWave;
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int t0 = 0; t0 < nm; t0 += nt) {
        const int m = t0 + tid;
        const int c = m < nm ? A.color[ma + m] : -1;
        s_wave[wave][lane] = 0;
        __syncthreads();
        unsigned long long same = __ballot(c >= 0);
#pragma unroll
        for (int b = 0; b < 6; b++) {
            const unsigned long long bal = __ballot((c >> b) & 1);
            same &= ((c >> b) & 1) ? bal : ~bal;
        }
        const int rank = __popcll(same & below);
        if (c >= 0 && rank == 0) s_wave[wave][c] = __popcll(same);
        __syncthreads();
        if (tid < kMaxColors) {   // first row of each wavefront's share
            int run = s_base[tid];
            for (int w = 0; w < nwave; w++) {
                const int n = s_wave[w][tid];
                s_wave[w][tid] = run;
                run += n;
            }
            s_base[tid] = run;
        }
        __syncthreads();
        if (c >= 0) {
            const int row = s_wave[wave][c] + rank;
            A.order[row] = ma + m;
            A.keys[row] = (uint64_t)g * kMaxColors + c;
        }
        __syncthreads();
    }
}

// Segment key of every manifold: its colour.  Counts per segment and the number of colours are accumulated for
// the segment table.
__global__ __launch_bounds__(256) void sv_color_keys(const int* color, const int* nm_ptr, uint64_t* keys, int* vals,
                                                     int* seg_cnt, int* ncolors) {
    __shared__ int hist[kMaxColors];
    for (int i = threadIdx.x; i < kMaxColors; i += blockDim.x) hist[i] = 0;
    __syncthreads();
    const int nm = *nm_ptr;
    RP3DG_GRID_STRIDE(m, nm) {
        const int c = color[m];
        atomicAdd(&hist[c], 1);
        keys[m] = (uint64_t)c;
        vals[m] = m;
    }
    __syncthreads();
    // the colours in use, once a workgroup: same-address atomics serialise
    static_assert(kMaxColors == kWave, "one lane a colour");
    if (threadIdx.x < kWave) {
        const int n = hist[threadIdx.x];
        if (n) atomicAdd(&seg_cnt[threadIdx.x], n);
        const unsigned long long in_use = __ballot(n != 0);
        if (threadIdx.x == 0 && in_use) atomicMax(ncolors, 64 - __clzll((long long)in_use));
    }
}

}  // namespace rp3dg
