// Broadphase of the MI355X step path.
//
// The reference keeps an incremental DynamicAABBTree of *fat* AABBs and only
// re-inserts a collider when its tight AABB leaves its fat AABB
// (DynamicAABBTree.cpp:186-214).  Because a fat AABB changes only on such a
// move, the reference pair set after computeBroadPhase() is exactly
//   { collider pairs whose current fat AABBs overlap (closed test, AABB.h:179) }
// filtered by different-body / category masks / no-collision body pairs
// (CollisionDetectionSystem.cpp:270-343).  We therefore keep the persistent
// fat AABB per collider (same FP32 refit as BroadPhaseSystem.cpp:155-185) and
// find the overlaps of the current boxes anew every step, without a tree:
//   bp_tiles  boxes in spatial order (strips, radix sort) or, up to a few
//             thousand colliders, in index order; the union box of every 64
//   bp_pairs  one workgroup per tile of 64 colliders against the tiles it meets
//   scan of the partner counts
//   bp_emit   partners -> each collider's sorted segment of the pair keys
//   bp_merge  carries orientation, temporal-coherence record and contact cache
//             of surviving pairs; orients new pairs like the reference.
// Batches of many small worlds scan each world in LDS instead (bp_world_scan).
#include <hip/hip_runtime.h>

#include "kcommon.h"
#include "rp3d_internal.h"
#include "refit_dev.h"
#include "strips.h"

namespace rp3dg {

__global__ void bp_refit(DevBodies B, DevColliders C, const float4* hull_bounds, int init) {
    RP3DG_GRID_STRIDE(i, C.n) refit_one(B, C, hull_bounds, init, i);
}

__device__ __forceinline__ void box_union(float4& mn, float4& mx, float4 bmn, float4 bmx) {
    mn = make_float4(fminf(mn.x, bmn.x), fminf(mn.y, bmn.y), fminf(mn.z, bmn.z), 0.f);
    mx = make_float4(fmaxf(mx.x, bmx.x), fmaxf(mx.y, bmx.y), fmaxf(mx.z, bmx.z), 0.f);
}

__device__ __forceinline__ void wave_box_union(float4& mn, float4& mx) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        float4 omn, omx;
        omn.x = __shfl_xor(mn.x, off, kWave); omn.y = __shfl_xor(mn.y, off, kWave); omn.z = __shfl_xor(mn.z, off, kWave);
        omx.x = __shfl_xor(mx.x, off, kWave); omx.y = __shfl_xor(mx.y, off, kWave); omx.z = __shfl_xor(mx.z, off, kWave);
        box_union(mn, mx, omn, omx);
    }
}

__device__ __forceinline__ bool aabb_overlap(float4 amn, float4 amx, float4 bmn, float4 bmx) {
    // AABB::testCollision (AABB.h:179-187), closed intervals
    if (amx.x < bmn.x || bmx.x < amn.x) return false;
    if (amx.y < bmn.y || bmx.y < amn.y) return false;
    if (amx.z < bmn.z || bmx.z < amn.z) return false;
    return true;
}

// Body pairs that must not collide (joints with collideConnected = false): per-body partner lists
__device__ __forceinline__ bool no_collision(const NoColLists& L, int ba, int bb) {
    const int e = L.offs[ba + 1];
    for (int k = L.offs[ba]; k < e; k++)
        if (L.list[k] == bb) return true;
    return false;
}

__device__ __forceinline__ bool filters_pass(uint32_t fa, uint32_t fb) {
    const uint32_t cata = fa & 0xffffu, maska = fa >> 16, catb = fb & 0xffffu, maskb = fb >> 16;
    return (maska & catb) != 0 && (cata & maskb) != 0;
}

// Pair filter of CollisionDetectionSystem::updateOverlappingPairs (CD.cpp:284-331): different bodies, no
// joint excluding the pair, collision category / mask, at least one convex shape (:324-331)
__device__ __forceinline__ bool pair_allowed(const DevColliders& C, int a, int b, const NoColLists& L) {
    const int ba = C.body[a], bb = C.body[b];
    if (ba == bb) return false;
    if (no_collision(L, ba, bb)) return false;
    if (shape_is_concave(C.type[a]) && shape_is_concave(C.type[b])) return false;
    return filters_pass(C.filter[a], C.filter[b]);
}

// ---------------------------------------------------------------------------------------------
// Order of the colliders (strips.h).  Every workgroup finds the bounds for itself, by the ranks of the sample's
// centres: 3 us of integer compares, where bounds from all centres took a launch of their own.
// ---------------------------------------------------------------------------------------------

__device__ __forceinline__ V3 box_centre(const DevColliders& C, int i) {
    const V3 a = ld3(C.amin, i), b = ld3(C.amax, i);
    return v3((a.x + b.x) * 0.5f, (a.y + b.y) * 0.5f, (a.z + b.z) * 0.5f);
}

// sample: up to kOrderSamples moving colliders; world_colliders: colliders of a mean world
__global__ __launch_bounds__(kOrderSamples) void bp_cells(DevColliders C, const int* sample, int nsample, float world_colliders,
                                                          uint64_t* keys, int* vals) {
    __shared__ uint4 s_rank[kOrderSamples];
    __shared__ float s_bound[2][3];
    __shared__ StripOrder s_order;
    static_assert(kOrderSamples == 256, "eight bits of thread in a rank key");
    const int t = threadIdx.x;
    V3 c = v3(INFINITY, INFINITY, INFINITY);
    if (t < nsample) c = box_centre(C, sample[t]);
    const bool ok = fabsf(c.x) < INFINITY && fabsf(c.y) < INFINITY && fabsf(c.z) < INFINITY;
    // the float's leading 24 bits in an order of integers, and the thread, so that no two are equal
    auto key = [&](float x) -> uint32_t {
        const uint32_t u = __float_as_uint(x);
        return ok ? ((u ^ (u >> 31 ? 0xffffffffu : 0x80000000u)) & ~255u) | (uint32_t)t : 0xffffffffu;
    };
    const uint4 mine = make_uint4(key(c.x), key(c.y), key(c.z), 0u);
    s_rank[t] = mine;
    if (t < 3) s_bound[0][t] = s_bound[1][t] = 0.f;
    const int m = __syncthreads_count(ok);
    int rank[3] = {0, 0, 0};
#pragma unroll 8
    for (int j = 0; j < kOrderSamples; j++) {
        const uint4 o = s_rank[j];
        rank[0] += o.x < mine.x ? 1 : 0;
        rank[1] += o.y < mine.y ? 1 : 0;
        rank[2] += o.z < mine.z ? 1 : 0;
    }
    for (int k = 0; k < 3; k++) {
        if (ok && rank[k] == m / kOrderCut) s_bound[0][k] = comp(c, k);
        if (ok && rank[k] == m - 1 - m / kOrderCut) s_bound[1][k] = comp(c, k);
    }
    __syncthreads();
    if (t == 0) s_order = strip_order(s_bound[0], s_bound[1], world_colliders);
    __syncthreads();
    RP3DG_GRID_STRIDE(i, C.n) {
        const V3 p = box_centre(C, i);
        keys[i] = ((uint64_t)(uint32_t)C.world[i] << kCellBits) | strip_key(s_order, comp(p, s_order.axis[0]), comp(p, s_order.axis[1]));
        vals[i] = i;
    }
}

// ---------------------------------------------------------------------------------------------
// Stable LSD radix sort, 8-bit digits.  Tiles of 256 x ITEMS keys per block; inside a tile keys are
// ranked by wave-level multisplit (8 ballots give the lanes sharing a digit) and cross-wave
// prefix counts in LDS, so equal digits keep their input order.
// ---------------------------------------------------------------------------------------------

constexpr int kSortThreads = 256;

// n: key count, or its upper bound when nptr (the count in device memory) is given.  ITEMS: keys a thread; 16,
// or 4 for a sort that would otherwise run on a fraction of the CUs.
template <int ITEMS>
__global__ __launch_bounds__(kSortThreads) void rs_hist(const uint64_t* keys, int n, const int* nptr, int shift, int* hist,
                                                        int nblocks) {
    if (nptr) n = min(n, *nptr);
    __shared__ int h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int base = blockIdx.x * kSortThreads * ITEMS;
    for (int k = 0; k < ITEMS; k++) {
        const int i = base + k * kSortThreads + threadIdx.x;
        if (i < n) atomicAdd(&h[(keys[i] >> shift) & 0xff], 1);
    }
    __syncthreads();
    hist[threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

__device__ __forceinline__ uint64_t lanemask_lt() {
    const int lane = lane_id();
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

template <int ITEMS>
__global__ __launch_bounds__(kSortThreads) void rs_scatter(const uint64_t* kin, const int* vin, uint64_t* kout,
                                                           int* vout, int n, const int* nptr, int shift, const int* offs,
                                                           int nblocks) {
    if (nptr) n = min(n, *nptr);
    __shared__ int base[256];
    __shared__ int wcnt[kSortThreads / kWave][256];
    const int t = threadIdx.x;
    base[t] = offs[t * nblocks + blockIdx.x];
    const int wid = t / kWave;
    const int blk = blockIdx.x * kSortThreads * ITEMS;
    for (int k = 0; k < ITEMS; k++) {
        for (int w = 0; w < kSortThreads / kWave; w++) wcnt[w][t] = 0;
        __syncthreads();
        const int i = blk + k * kSortThreads + t;
        const bool valid = i < n;
        uint64_t key = valid ? kin[i] : 0;
        const int d = valid ? (int)((key >> shift) & 0xff) : 0;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (d >> b) & 1;
            const uint64_t bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        const int rank = __popcll(peers & lanemask_lt());
        if (valid && rank == 0) wcnt[wid][d] = __popcll(peers);
        __syncthreads();
        {  // exclusive prefix over waves for digit t, advance base
            int run = 0;
            for (int w = 0; w < kSortThreads / kWave; w++) {
                const int c = wcnt[w][t];
                wcnt[w][t] = run;
                run += c;
            }
            __syncthreads();
            if (valid) {
                const int pos = base[d] + wcnt[wid][d] + rank;
                kout[pos] = key;
                vout[pos] = vin[i];
            }
            __syncthreads();
            base[t] += run;
        }
        __syncthreads();
    }
}

#define RS_INSTANCE(I)                                                                                            \
    template __global__ void rs_hist<I>(const uint64_t*, int, const int*, int, int*, int);                        \
    template __global__ void rs_scatter<I>(const uint64_t*, const int*, uint64_t*, int*, int, const int*, int,     \
                                           const int*, int);
RS_INSTANCE(4)
RS_INSTANCE(16)
#undef RS_INSTANCE

// ---------------------------------------------------------------------------------------------
// Overlaps.  Each overlapping pair is emitted by exactly one of its colliders (the pair key's high word):
//   moving vs moving -> the lower collider index; moving vs static -> the moving one;
//   static vs static -> the lower index, from the constant list built at creation.
// Each emitter's partners end sorted ascending in its segment, so the pair table is sorted by key.
// ---------------------------------------------------------------------------------------------

constexpr int kTile = kWave;   // colliders per tile
constexpr int kLargeList = 1024;   // partners that bp_emit_large sorts in LDS
constexpr int kTileWalk = 8192;    // colliders of a world that are walked by tiles for one that has so many
constexpr int kWalkTiles = -1, kWalkWorld = -2;   // first slab entry of a collider whose partners the slab does not hold

// Boxes in the order of `sorted` (null: index order), the union of every tile and its range of worlds.
// smn.w = collider, smx.w = world * 2 + static (int bits); tmn.w / tmx.w = first / last world of the tile.
__global__ __launch_bounds__(256) void bp_tiles(DevColliders C, const int* sorted, int n, float4* smn, float4* smx,
                                                float4* tmn, float4* tmx) {
    const int nt = (n + kTile - 1) / kTile;
    for (int base = (blockIdx.x * blockDim.x + threadIdx.x) & ~(kTile - 1); base < nt * kTile;
         base += gridDim.x * blockDim.x) {
        const int s = base + lane_id();
        float4 mn = make_float4(INFINITY, INFINITY, INFINITY, 0.f), mx = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
        int w = 0;
        if (s < n) {
            const int c = sorted ? sorted[s] : s;
            mn = C.amin[c];
            mx = C.amax[c];
            w = C.world[c];
            smn[s] = make_float4(mn.x, mn.y, mn.z, __int_as_float(c));
            smx[s] = make_float4(mx.x, mx.y, mx.z, __int_as_float(2 * w + (C.is_static[c] ? 1 : 0)));
        }
        wave_box_union(mn, mx);
        const int last = min(n - base, kTile) - 1;   // worlds ascend in either order
        const int w0 = __shfl(w, 0, kWave), w1 = __shfl(w, last, kWave);
        if (lane_id() == 0) {
            tmn[base / kTile] = make_float4(mn.x, mn.y, mn.z, __int_as_float(w0));
            tmx[base / kTile] = make_float4(mx.x, mx.y, mx.z, __int_as_float(w1));
        }
    }
}

// Does collider c emit the pair (c, o)?  (Their boxes overlap; both are of one world.)
__device__ __forceinline__ bool emits(const DevColliders& C, int c, int o, const NoColLists& L) {
    return o != c && (C.is_static[o] || o > c) && pair_allowed(C, c, o, L);
}

__device__ __forceinline__ bool tile_meets(const float4* tmn, const float4* tmx, int T, float4 mn, float4 mx, int w) {
    const float4 a = tmn[T], b = tmx[T];
    return __float_as_int(a.w) <= w && __float_as_int(b.w) >= w && aabb_overlap(mn, mx, a, b);
}
// Does the lane's collider o of tile T, one of world w, overlap the box?
__device__ __forceinline__ bool tile_hit(int n, const float4* smn, const float4* smx, int T, float4 mn, float4 mx, int w, int& o) {
    const int s = T * kTile + lane_id();
    if (s >= n) return false;
    const float4 a = smn[s], b = smx[s];
    o = __float_as_int(a.w);
    return (__float_as_int(b.w) >> 1) == w && aabb_overlap(mn, mx, a, b);
}

// One workgroup per tile of 64 querying colliders, one per lane, the same in every wavefront.  The
// wavefronts share the tiles whose box meets the queries': a wavefront loads a tile's boxes (one per lane),
// drops those outside the queries' union, and every lane tests its box against the others eight at a time from
// scalar registers, collecting a bit for each (one at a time, read from the lanes that hold them, with the
// bookkeeping of a hit after every test: 36 us for 1001 boxes, 74 for 3,006 bodies, 129 for 6,965, in index
// order; now 24, 50 and 89).  A tree walk is a chain of dependent loads per collider with most lanes of a wavefront
// waiting for the deepest; here every load is a full tile, and the arithmetic grows with the overlapping
// tiles only.  Overlaps are collected in LDS, filtered (pair_allowed), sorted by rank and written to the
// collider's slab; count[c] = its partners.  A collider with more overlaps than the slab holds is counted
// over the tiles that it meets by a wavefront (over its world, by the workgroup, where that is a few steps or the
// overlaps are more than kLargeList), and listed for bp_emit_large.  From the fourth hit of a wavefront on, colliders of the query's own body are left out at once, so
// that the parts of a compound do not fill its slab.
__global__ __launch_bounds__(1024) void bp_pairs(DevColliders C, int n, const float4* smn, const float4* smx,
                                                 const float4* tmn, const float4* tmx, const int* wcoll, NoColLists L,
                                                 int* count, int* slab, int* large, int* nb_large) {
    __shared__ int s_cnt[kTile], s_id[kTile];
    __shared__ int s_list[kTile][kSlab];
    __shared__ int2 s_box[1024 / kWave][kTile];   // the collider and kind of a wavefront's current boxes
    __shared__ int s_total;
    typedef float Vec4 __attribute__((ext_vector_type(4)));
    using BoxTable = const __attribute__((address_space(4))) Vec4*;   // read through the scalar cache
    const BoxTable bmin = (BoxTable)(uintptr_t)smn, bmax = (BoxTable)(uintptr_t)smx;
    constexpr int kBoxGroup = 8;   // boxes loaded and tested at a time
    const int tid = threadIdx.x, lane = tid & (kWave - 1), nw = blockDim.x / kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int nt = (n + kTile - 1) / kTile;
    const int s0 = blockIdx.x * kTile + lane;
    float4 qmn = make_float4(INFINITY, INFINITY, INFINITY, 0.f), qmx = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    int c = -1, world = 0;
    bool query = false;
    if (s0 < n) {
        qmn = smn[s0];
        qmx = smx[s0];
        c = __float_as_int(qmn.w);
        const int t = __float_as_int(qmx.w);
        world = t >> 1;
        query = !(t & 1);
        if (!query && wave == 0) count[c] = C.ss_offs[c + 1] - C.ss_offs[c];
    }
    if (!query) {   // overlaps nothing
        qmn = make_float4(INFINITY, INFINITY, INFINITY, 0.f);
        qmx = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    }
    if (wave == 0) {
        s_cnt[lane] = 0;
        s_id[lane] = query ? c : -1;
    }
    if (!__ballot(query)) return;   // (the same in every wavefront)
    float4 umn = qmn, umx = qmx;
    wave_box_union(umn, umx);
    int wlo = query ? world : 0x7fffffff, whi = query ? world : -1;
    whi = wave_max(whi);
    wlo = -wave_max(-wlo);
    __syncthreads();
    int seen = 0;   // tiles that meet the queries so far
    int hit_here = 0;   // of the lane's query in this wavefront
    for (int T0 = 0; T0 < nt; T0 += kWave) {
        const int T = T0 + lane;
        bool meets = false;
        if (T < nt) {
            const float4 a = tmn[T], b = tmx[T];
            meets = __float_as_int(a.w) <= whi && __float_as_int(b.w) >= wlo && aabb_overlap(umn, umx, a, b);
        }
        unsigned long long m = __ballot(meets);
        while (m) {
            const int k = __ffsll(m) - 1;
            m &= m - 1;
            if ((seen++ & (nw - 1)) != wave) continue;   // (a power of two)
            const int s = (T0 + k) * kTile + lane;
            float4 bmn = make_float4(INFINITY, INFINITY, INFINITY, 0.f), bmx = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
            if (s < n) {
                bmn = smn[s];
                bmx = smx[s];
            }
            const unsigned long long cand = __ballot(s < n && aabb_overlap(umn, umx, bmn, bmx));
            if (!cand) continue;
            s_box[wave][lane] = make_int2(__float_as_int(bmn.w), __float_as_int(bmx.w));
            const int base = __builtin_amdgcn_readfirstlane((T0 + k) * kTile);
            unsigned long long hits = 0;
            for (int g = 0; g < kTile; g += kBoxGroup) {
                if (!((cand >> g) & ((1u << kBoxGroup) - 1u))) continue;
                unsigned int bits = 0;
#pragma unroll
                for (int j = 0; j < kBoxGroup; j++) {
                    const int i = min(base + g + j, n - 1);   // (beyond n: no candidate)
                    const Vec4 a = bmin[i], b = bmax[i];
                    const bool apart = (qmx.x < a.x) | (b.x < qmn.x) | (qmx.y < a.y) | (b.y < qmn.y) | (qmx.z < a.z) |
                                       (b.z < qmn.z);   // aabb_overlap
                    bits |= apart ? 0u : 1u << j;
                }
                hits |= (unsigned long long)bits << g;
            }
            hits &= cand;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            while (hits) {
                const int q = __ffsll(hits) - 1;
                hits &= hits - 1;
                const int o = s_box[wave][q].x, t = s_box[wave][q].y;
                if ((t >> 1) == world && o != c && ((t & 1) || o > c)) {
                    if (++hit_here > 3 && C.body[o] == C.body[c]) continue;
                    const int pos = atomicAdd(&s_cnt[lane], 1);
                    if (pos < kSlab) s_list[lane][pos] = o;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
    __syncthreads();
    // filters, one entry a thread
    constexpr int kDrop = 0x7fffffff;
    for (int e = tid; e < kTile * kSlab; e += blockDim.x) {
        const int q = e / kSlab, k = e % kSlab;
        if (k >= s_cnt[q] || s_cnt[q] > kSlab) s_list[q][k] = kDrop;
        else if (!pair_allowed(C, s_id[q], s_list[q][k], L)) s_list[q][k] = kDrop;
    }
    __syncthreads();
    for (int q = wave; q < kTile; q += nw) {   // rank sort; ids are unique
        const int cq = s_id[q], len = s_cnt[q];
        if (cq < 0 || len > kSlab) continue;
        const int id = lane < kSlab ? s_list[q][lane] : kDrop;
        int rank = 0;
        const int ulen = __builtin_amdgcn_readfirstlane(len);
        for (int k = 0; k < ulen; k++) rank += __builtin_amdgcn_readlane(id, k) < id ? 1 : 0;
        if (id != kDrop) slab[(size_t)cq * kSlab + rank] = id;
        const int total = __popcll(__ballot(id != kDrop));
        if (lane == 0) count[cq] = total;
    }
    // colliders with more overlaps than their slab holds: exact counts, and which walk found them (bp_emit_large
    // takes the same: with a box that is not a number the two need not agree)
    auto list_large = [&](int cq, int total, int walk) {
        count[cq] = total;
        slab[(size_t)cq * kSlab] = walk;
        large[atomicAdd(nb_large, 1)] = cq;
    };
    auto walk_world = [&](int cq, int first, int step) {   // the lane's share
        const float4 amn = C.amin[cq], amx = C.amax[cq];
        const int w = C.world[cq];
        int found = 0;
        for (int o = wcoll[w] + first; o < wcoll[w + 1]; o += step)
            if (aabb_overlap(amn, amx, C.amin[o], C.amax[o]) && emits(C, cq, o, L)) found++;
        return found;
    };
    const int found = s_cnt[lane];
    const int of_world = query ? wcoll[world + 1] - wcoll[world] : 0;
    const unsigned long long over = __ballot(query && found > kSlab);
    const unsigned long long by_tiles = __ballot(found <= kLargeList && of_world > kTileWalk) & over;
    int turn = 0;
    for (unsigned long long m = by_tiles; m; m &= m - 1) {
        if ((turn++ & (nw - 1)) != wave) continue;
        const int cq = s_id[__ffsll(m) - 1], w = C.world[cq];
        const float4 amn = C.amin[cq], amx = C.amax[cq];
        int total = 0, walk = kWalkTiles;
        for (int T0 = 0; T0 < nt; T0 += kWave) {
            unsigned long long meets = __ballot(T0 + lane < nt && tile_meets(tmn, tmx, T0 + lane, amn, amx, w));
            for (; meets; meets &= meets - 1) {
                int o = 0;
                const bool hit = tile_hit(n, smn, smx, T0 + __ffsll(meets) - 1, amn, amx, w, o);
                total += __popcll(__ballot(hit && emits(C, cq, o, L)));
            }
        }
        if (total > kLargeList) {
            total = wave_sum(walk_world(cq, lane, kWave));
            walk = kWalkWorld;
        }
        if (lane == 0) list_large(cq, total, walk);
    }
    for (unsigned long long m = over & ~by_tiles; m; m &= m - 1) {   // the same in every wavefront
        const int cq = s_id[__ffsll(m) - 1];
        __syncthreads();
        if (tid == 0) s_total = 0;
        __syncthreads();
        const int mine = wave_sum(walk_world(cq, tid, blockDim.x));
        if (lane == 0 && mine) atomicAdd(&s_total, mine);
        __syncthreads();
        if (tid == 0) list_large(cq, s_total, kWalkWorld);
    }
}

// Partners from the slabs (eight lanes per collider) and the static colliders' lists to the segments of the
// key array.
__global__ void bp_emit(DevColliders C, int n, const int* count, const int* offset, const int* slab, uint64_t* out_keys,
                        int capacity, int* status) {
    constexpr int kLanes = 8;
    RP3DG_GRID_STRIDE(t, n * kLanes) {
        const int c = t / kLanes;
        const int base = offset[c], total = count[c];
        const bool fixed = C.is_static[c];
        const int* src = fixed ? C.ss_list + C.ss_offs[c] : slab + (size_t)c * kSlab;
        if (!fixed && total > 0 && src[0] < 0) continue;   // bp_emit_large's
        // past the capacity the table is truncated (and the step reports the overflow), but every entry
        // below it is written, since the merge reads all of them
        for (int k = t % kLanes; k < total; k += kLanes) {
            if (base + k < capacity) out_keys[base + k] = ((uint64_t)(uint32_t)c << 32) | (uint32_t)src[k];
            else atomicOr(status, STATUS_PAIR_OVERFLOW);
        }
    }
}

// Colliders with more overlaps than a slab, one workgroup each.  Up to kLargeList partners are collected from the tiles
// that the collider meets and ranked in LDS, in worlds of more than kTileWalk colliders; else they come sorted from a
// walk over its world in index order.  With that walk for all, the broadphase of 12,000 and 40,000 spheres of 64 pairs
// each took 0.93 and 7.0 ms, 0.33 and 0.93 as it is; with tiles for all that of 3,000 takes 0.48 and not 0.35.
__global__ __launch_bounds__(1024) void bp_emit_large(DevColliders C, int n, const float4* smn, const float4* smx,
                                                      const float4* tmn, const float4* tmx, const int* wcoll, NoColLists L,
                                                      const int* count, const int* offset, const int* slab,
                                                      uint64_t* out_keys, int capacity, const int* large,
                                                      const int* nb_large, int* status) {
    __shared__ int sm[17];
    __shared__ int4 s_list[kLargeList / 4];
    __shared__ int s_tile[1024];
    int* list = reinterpret_cast<int*>(s_list);
    const int nl = *nb_large, wave = threadIdx.x / kWave, nw = blockDim.x / kWave;
    for (int i = blockIdx.x; i < nl; i += gridDim.x) {
        const int c = large[i], w = C.world[c], total = count[c];
        const float4 amn = C.amin[c], amx = C.amax[c];
        int base = offset[c];
        auto put = [&](int pos, int o) {
            if (pos < capacity) out_keys[pos] = ((uint64_t)(uint32_t)c << 32) | (uint32_t)o;
            else atomicOr(status, STATUS_PAIR_OVERFLOW);
        };
        if (slab[(size_t)c * kSlab] == kWalkTiles) {
            constexpr int kNone = 0x7fffffff;
            const int nt = (n + kTile - 1) / kTile;
            if (threadIdx.x == 0) sm[0] = 0;
            for (int k = threadIdx.x; k < kLargeList; k += blockDim.x) list[k] = kNone;
            for (int T0 = 0; T0 < nt; T0 += blockDim.x) {   // the tiles it meets, shared out among the wavefronts
                const int T = T0 + threadIdx.x;
                if (threadIdx.x == 0) sm[1] = 0;
                __syncthreads();
                if (T < nt && tile_meets(tmn, tmx, T, amn, amx, w)) s_tile[atomicAdd(&sm[1], 1)] = T;
                __syncthreads();
                for (int k = wave; k < sm[1]; k += nw) {
                    int o = 0;
                    if (tile_hit(n, smn, smx, s_tile[k], amn, amx, w, o) && emits(C, c, o, L)) {
                        const int pos = atomicAdd(&sm[0], 1);
                        if (pos < kLargeList) list[pos] = o;
                    }
                }
                __syncthreads();
            }
            for (int k = threadIdx.x; k < total; k += blockDim.x) {
                const int o = list[k];
                int rank = 0;
                for (int j = 0; 4 * j < total; j++) {
                    const int4 x = s_list[j];
                    rank += (x.x < o ? 1 : 0) + (x.y < o ? 1 : 0) + (x.z < o ? 1 : 0) + (x.w < o ? 1 : 0);
                }
                put(base + rank, o);
            }
            __syncthreads();
            continue;
        }
        for (int o0 = wcoll[w]; o0 < wcoll[w + 1]; o0 += blockDim.x) {
            const int o = o0 + threadIdx.x;
            const bool hit = o < wcoll[w + 1] && aabb_overlap(amn, amx, C.amin[o], C.amax[o]) && emits(C, c, o, L);
            int found;
            const int pos = base + block_excl_scan(hit ? 1 : 0, sm, &found);
            if (hit) put(pos, o);
            base += found;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Batches of small worlds.  One workgroup per world group stages the fat AABBs of its
// colliders in LDS and every dynamic collider tests the boxes of all colliders of its own world in
// index order, so its partners come out sorted; the scan runs twice (count, then write after the
// prefix sum of the counts).  The pair set is bp_pairs' (the same
// AABB::testCollision on the same boxes, the same emitter rule and filters); the cost is
// sum over worlds of (colliders)^2 box tests in one launch for thousands of worlds.  LDS per collider: min (w = body | static << 31), max (w = filter bits).
// ---------------------------------------------------------------------------------------------
// pass 0 writes the partner count of every collider, pass 1 (after the scan) its sorted keys.
__global__ __launch_bounds__(256) void bp_world_scan(DevColliders C, const int* gworld, const int* wcoll,
                                                     const int* block_group, NoColLists L, int* count,
                                                     const int* offset, uint64_t* out_keys, int capacity, int pass,
                                                     int* status) {
    extern __shared__ float4 s_box[];   // [group colliders] min boxes, then [group colliders] max boxes
    const int g = block_group[blockIdx.x];
    const int gc0 = wcoll[gworld[g]], gc1 = wcoll[gworld[g + 1]];
    const int ncg = gc1 - gc0;
    float4* smn = s_box;
    float4* smx = s_box + ncg;
    for (int i = threadIdx.x; i < ncg; i += blockDim.x) {
        const int c = gc0 + i;
        float4 mn = C.amin[c], mx = C.amax[c];
        mn.w = __int_as_float(C.body[c] | (C.is_static[c] ? (int)0x80000000u : 0));
        mx.w = __uint_as_float(C.filter[c]);
        smn[i] = mn;
        smx[i] = mx;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < ncg; i += blockDim.x) {
        const int c = gc0 + i;
        const float4 amn = smn[i], amx = smx[i];
        const int bc = __float_as_int(amn.w);
        const int base = pass ? offset[c] : 0;
        if (bc < 0) {   // static colliders do not query (their static-static pairs are listed at upload)
            const int b = C.ss_offs[c], e = C.ss_offs[c + 1];
            if (!pass) {
                count[c] = e - b;
            } else {
                for (int q = b; q < e; q++)
                    if (base + q - b < capacity) out_keys[base + q - b] = ((uint64_t)(uint32_t)c << 32) | (uint32_t)C.ss_list[q];
                if (base + e - b > capacity) atomicOr(status, STATUS_PAIR_OVERFLOW);
            }
            continue;
        }
        const int w = C.world[c];
        const int j0 = wcoll[w] - gc0, j1 = wcoll[w + 1] - gc0;
        const uint32_t fc = __float_as_uint(amx.w);
        const bool concave = shape_is_concave(C.type[c]);   // concave vs concave pairs are not created
        const int n0 = L.offs[bc], n1 = L.offs[bc + 1];   // bodies this collider's body must not collide with
        int cnt = 0;
        for (int j = j0; j < j1; j++) {
            const float4 bmn = smn[j], bmx = smx[j];
            const int bo = __float_as_int(bmn.w);
            if (j == i || (bo >= 0 && j < i)) continue;
            if (!aabb_overlap(amn, amx, bmn, bmx)) continue;
            const int bb = bo & 0x7fffffff;
            if (bb == bc) continue;
            bool excluded = false;
            for (int k = n0; k < n1; k++) excluded |= L.list[k] == bb;
            if (excluded || !filters_pass(fc, __float_as_uint(bmx.w))) continue;
            if (concave && shape_is_concave(C.type[gc0 + j])) continue;
            if (pass) {
                if (base + cnt < capacity) out_keys[base + cnt] = ((uint64_t)(uint32_t)c << 32) | (uint32_t)(gc0 + j);
                else atomicOr(status, STATUS_PAIR_OVERFLOW);
            }
            cnt++;
        }
        if (!pass) count[c] = cnt;
    }
}

// ---------------------------------------------------------------------------------------------
// Pair table update.  Surviving pairs keep collider order, LastFrameCollisionInfo and the contact
// cache.  A new pair is oriented as OverlappingPairs::addPair receives it: collider1 is the moved
// shape whose broadphase query reported the pair first, i.e. the moved one, or the one that comes
// first in the moved-shape set iteration order (rank) when both moved this step.
// ---------------------------------------------------------------------------------------------

// CollisionDispatch::selectAlgorithm (CollisionDispatch.cpp:80-115) on CollisionShapeType
__device__ __forceinline__ int shape_kind(int t) { return t == SHAPE_SPHERE ? 0 : (t == SHAPE_CAPSULE ? 1 : 2); }
__device__ __forceinline__ int select_algo(int t1, int t2) {
    if (shape_is_concave(t1) || shape_is_concave(t2)) return ALGO_CONCAVE;   // OverlappingPairs.cpp:427-440
    int a = shape_kind(t1), b = shape_kind(t2);
    if (a > b) { const int tmp = a; a = b; b = tmp; }
    if (a == 0 && b == 0) return ALGO_SPHERE_SPHERE;
    if (a == 0 && b == 1) return ALGO_SPHERE_CAPSULE;
    if (a == 1 && b == 1) return ALGO_CAPSULE_CAPSULE;
    if (a == 0 && b == 2) return ALGO_SPHERE_POLY;
    if (a == 1 && b == 2) return ALGO_CAPSULE_POLY;
    return ALGO_POLY_POLY;
}

// nkeys_ptr: overlapping pairs found (clamped to the capacity; bp_emit and bp_world_scan flag an overflow).
// nold_ptr: size of the previous table O.  nnew_ptr / nb_pairs_ptr receive the size of the new table N.
// old_offs: first entry of every emitter's segment in the previous table (its keys are sorted and
// grouped by emitter, key >> 32), so a key is searched only within its emitter's few old entries.
__global__ void bp_merge(DevColliders C, const uint64_t* keys, const int* nkeys_ptr, int capacity, DevPairs O,
                         const int* nold_ptr, const int* old_offs, DevPairs N, int* nnew_ptr, int* nb_pairs_ptr) {
    const int nkeys = min(*nkeys_ptr, capacity);
    const int nold = *nold_ptr;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *nnew_ptr = nkeys;
        *nb_pairs_ptr = nkeys;
    }
    RP3DG_GRID_STRIDE(k, nkeys) {
        const uint64_t key = keys[k];
        N.key[k] = key;
        const int e = (int)(key >> 32);
        int lo = min(old_offs[e], nold), hi = min(old_offs[e + 1], nold) - 1, found = -1;
        while (lo <= hi) {
            const int mid = (lo + hi) >> 1;
            const uint64_t v = O.key[mid];
            if (v == key) { found = mid; break; }
            if (v < key) lo = mid + 1;
            else hi = mid - 1;
        }
        N.prev[k] = found;
        if (found >= 0) {
            // the contact cache stays in O; the narrowphase reads it there through N.prev
            N.col[k] = O.col[found];
            N.algo[k] = O.algo[found];
            N.lf[k] = O.lf[found];
            N.lfaxis[k] = O.lfaxis[found];
            N.evf[k] = O.evf[found];
            O.kept[found] = 1;
        } else {
            N.evf[k] = 0;
            const int a = (int)(key >> 32), b = (int)(key & 0xffffffffu);
            const int ma = C.moved[a], mb = C.moved[b];
            bool a_first;
            if (ma && !mb) a_first = true;
            else if (mb && !ma) a_first = false;
            else a_first = C.rank[a] < C.rank[b];
            const int c1 = a_first ? a : b, c2 = a_first ? b : a;
            N.col[k] = make_int2(c1, c2);
            N.algo[k] = select_algo(C.type[c1], C.type[c2]);
            N.lf[k] = 0u;
            N.lfaxis[k] = make_float4(0.f, 1.f, 0.f, 0.f);   // LastFrameCollisionInfo() default axis
            N.ncp[k] = 0;
            N.fimp[k] = make_float4(0.f, 0.f, 0.f, 0.f);
            N.fv1[k] = make_float4(0.f, 0.f, 0.f, 0.f);
            N.fv2[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
}

}  // namespace rp3dg
