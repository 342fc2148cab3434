// Searches shared by the query kernels (query.hip, silhouette.hip, batch.hip):
// closest point, closest silhouette and rays of a wave from one pool of pending
// nodes, and the chunks of a persistent launch.  Device code.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.hpp"
#include "traverse.hpp"

namespace snch {

namespace {

constexpr uint32_t LDS_PER_CU = 160 * 1024;

__device__ __forceinline__ uint32_t xcd_remap(uint32_t b, uint32_t nb)
{
    const uint32_t X = 8, q = nb / X, r = nb % X, x = b % X, k = b / X;
    return x * q + (x < r ? x : r) + k;
}

// wave-uniform copy of lane 0's value (a scalar register)
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// per-query visit counters (Counts), summed over the wave before one atomic per wave
__device__ __forceinline__ void flush_counts(const Counts& c, unsigned long long* stats)
{
    unsigned long long v[5] = {c.box, c.leaf, c.edge, c.node, c.cone};
#pragma unroll
    for (int k = 0; k < 5; ++k) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            v[k] += __shfl_xor(v[k], o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < 5; ++k)
            atomicAdd(stats + k, v[k]);
    }
}

// ------------------------------------------------------------ pooled search
// One wave answers up to 64 queries from a pool of pending nodes in LDS.  An
// item is (query slot, internal node) with the lower bound it was pushed
// with; a step pops the last 32 items, one pair of lanes each, and each lane
// tests one child of its item.  Surviving internal children are pushed, near
// ones on top, and surviving leaves go to a buffer that the wave evaluates 64
// at a time.  Each query's best answer and pruning bound live in LDS and are
// updated by atomic minima on (distance bits, id).  Against a stack per lane (one query per lane, the
// wave as slow as its slowest lane, a lane as slow as its chain of dependent
// loads) every lane has work until the wave's last query ends, a node's two
// children share one 64-B line per pair of lanes, and leaf code runs on full
// waves.  Queries enter as the pool runs low, CP_ADD or SIL_ADD at a time: with
// all 64 in flight at once the pool fills and pops one item at a time.
//
// Measured, one lane per query with a stack -> pool (each with all that is in
// this file now).  Closest point: 2^22 queries on 2^20 triangles 46 -> 18.5 ms,
// 65,536 on 20,480 triangles 2.1 -> 0.12 ms, 1,000 0.83 -> 0.03 ms (there a
// launch lasted as long as the longest chain of dependent loads, about 2 us a
// node).  Closest silhouette: 2^22 on 2^20 triangles 68 -> 20.7 ms, 10,007 on
// 90,000 triangles 4.3 -> 0.13 ms.  Pairs that keep their near child in
// registers instead of the pool: half as long again.  For those 2^22 queries,
// while they took 22.6 ms:
// SIL_ADD 12 / 20 / 26 / 32 / 40 / 64: 26.7 / 25.7 / 24.7 / 22.6 / 24.5 / 25.0
// ms; CP_ADD 16 to 24: within 1%; runs of 24 / 32 / 40 / 48 / 64 leaves: closest
// point 22.0 / 21.0 / 20.1 / 19.7 / 19.3, silhouette 25.2 / 25.2 / 25.7 / 25.9 /
// 25.9 (and 6% more of 10,007 with 64).
//
// The answer is that of the search one lane would make alone, near child
// first, each node's leaves at once, which skips a box as soon as its lower
// bound exceeds the best distance so far (lane_nearest below); rays that graze a
// face within rounding excepted (ray_leaves).  Where no
// rounding interferes that is the smallest (distance, id) of all leaves,
// whatever the order.  But a leaf's computed distance can lie below its box's
// computed lower bound by a few units in the last place of the coordinates
// ("hidden" leaves): among candidates that close, what the lone search finds
// first decides.  So the pool prunes with bounds widened by more than that
// rounding, which leaves no such candidate out, and where a hidden leaf has
// the smallest distance the lane repeats the search alone, from the widened
// bound (a few dozen nodes).  Closest point also bounds an answer by the boxes'
// minmaxdists, and there a leaf can be too far as well: the distance computed
// for a sliver or a degenerate triangle may be any multiple of the true one, or
// NaN, so that nothing within its box's minmaxdist is found.  A lane whose
// bound ended below its answer's own therefore searches alone too (cp_wave).
constexpr uint32_t CP_ADD = 20, SIL_ADD = 32;
constexpr uint32_t CP_LEAF_RUN = 64, SIL_LEAF_RUN = 40; // leaves that are worth a step of the wave
constexpr uint32_t LEAF_CAP = 64 + 64; // buffer entries: below a run's before a step, which adds at most 64

// smaller is better: the distance, then hidden candidates (so that an answer
// tells whether any attains it), then the smaller id (distances are not
// negative, ids are below 2^31)
__device__ __forceinline__ unsigned long long pack_best(float d, uint32_t id, bool hidden = false)
{
    return ((unsigned long long)__float_as_uint(d) << 32) | (hidden ? id : id | 0x80000000u);
}
// returns whether the answer is hidden
__device__ __forceinline__ bool unpack_best(unsigned long long v, float& d, uint32_t& id)
{
    const uint32_t w = (uint32_t)v;
    d = __uint_as_float((uint32_t)(v >> 32));
    id = w == INVALID ? INVALID : w & 0x7FFFFFFFu;
    return (w & 0x80000000u) == 0u;
}
// lanes of mask below this one
__device__ __forceinline__ uint32_t rank_in(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
// the value of the other lane of this lane's pair (lane ^ 1)
__device__ __forceinline__ float pair_other(float v)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0xB1, 0xF, 0xF, true));
}

// LDS of one wave, carved from the block's dynamic LDS: cap pool items (slot
// << 24 | node, and the upper half of the float bits of the bound it was
// pushed with: a lower bound of it), the leaf buffer (2 words per entry: slot
// << 24 | leaf, bound), and per query slot its answer, point and widened
// (squared) pruning bound
struct WaveLds {
    unsigned long long* best;
    uint32_t *pool, *leaf, *bound;
    uint16_t* pkey;
    float* q; // x, y, z rows of 64
    uint32_t cap;
    static constexpr uint32_t FIXED = 128 + 2 * LEAF_CAP + 64 + 192; // words besides the pool (and hard caps)
    __device__ __forceinline__ WaveLds(uint32_t* base, uint32_t cap_)
    {
        best = reinterpret_cast<unsigned long long*>(base);
        leaf = base + 128;
        bound = leaf + 2 * LEAF_CAP;
        q = reinterpret_cast<float*>(bound + 64);
        pool = base + FIXED;
        pkey = reinterpret_cast<uint16_t*>(pool + cap_);
        cap = cap_;
    }
    // squared hard caps, after the pool (hard-capped searches only)
    __device__ __forceinline__ float* cap2() const { return reinterpret_cast<float*>(pool + cap + cap / 2); }
    __device__ __forceinline__ v3 point(uint32_t s) const { return mk(q[s], q[64 + s], q[128 + s]); }
    __device__ __forceinline__ void start(uint32_t s, v3 p)
    {
        q[s] = p.x;
        q[64 + s] = p.y;
        q[128 + s] = p.z;
        best[s] = pack_best(F_INF, INVALID);
        bound[s] = __float_as_uint(F_INF);
    }
};
// a distance widened by more than the rounding of any distance to the scene
// from p (scale: the scene's largest coordinate; in 2D also the offset of the
// boxes), squared
template <int DIM>
__device__ __forceinline__ float widened(float d, v3 p, float scale)
{
    const float delta = (DIM == 3 ? 5e-7f : 2.0f * BVH_OFFSET) +
                        1e-6f * fmx(scale, fmx(dm::fabs_(p.x), fmx(dm::fabs_(p.y), dm::fabs_(p.z))));
    const float u = d * 1.000002f + delta;
    return u * u;
}
// the same by half as much: more than the rounding of a distance still (random
// slivers and needles, 3e8 queries at 1e-6 to 1e4 times their size: no leaf is
// hidden deeper), and less than that of a minmaxdist that equals the answer's
// distance (1.5 % of the queries beside a rough mesh) widened in full
template <int DIM>
__device__ __forceinline__ float half_widened(float d, v3 p, float scale)
{
    const float delta = (DIM == 3 ? 2.5e-7f : BVH_OFFSET) +
                        0.5e-6f * fmx(scale, fmx(dm::fabs_(p.x), fmx(dm::fabs_(p.y), dm::fabs_(p.z))));
    const float u = d * 1.000001f + delta;
    return u * u;
}
__device__ __forceinline__ float scene_scale(const TreeView& t)
{
    const box3 b = ldbox2(t.nbox, 0);
    return fmx(fmx(fmx(dm::fabs_(b.lo.x), dm::fabs_(b.hi.x)), fmx(dm::fabs_(b.lo.y), dm::fabs_(b.hi.y))),
               fmx(dm::fabs_(b.lo.z), dm::fabs_(b.hi.z)));
}
// words of dynamic LDS of a wave
constexpr uint32_t wave_lds_words(uint32_t cap, bool capped = false)
{
    return cap + cap / 2 + WaveLds::FIXED + (capped ? 64u : 0u);
}

// append (a, key) of the lanes with `yes` to a list of two-word entries (the
// callers' sizes never exceed the list: pool_take, LEAF_CAP)
__device__ __forceinline__ void list_push(uint32_t* list, uint32_t& size, bool yes, uint32_t a, float key)
{
    const uint64_t m = __builtin_amdgcn_ballot_w64(yes);
    const uint32_t at = size + rank_in(m);
    if (yes) {
        list[2 * at] = a;
        list[2 * at + 1] = __float_as_uint(key);
    }
    size += (uint32_t)__popcll(m);
}

// the same for pool items
template <class L>
__device__ __forceinline__ void pool_push(L& W, uint32_t& size, bool yes, uint32_t a, float key)
{
    const uint64_t m = __builtin_amdgcn_ballot_w64(yes);
    const uint32_t at = size + rank_in(m);
    if (yes) {
        W.pool[at] = a;
        W.pkey[at] = (uint16_t)(__float_as_uint(key) >> 16);
    }
    size += (uint32_t)__popcll(m);
}

// the children to descend to: those with `near` on top of the others.  One masked
// store instead of two pool_push: closest point 19.2 -> 18.5 ms for 2^22 queries on
// 2^20 triangles, rays the same; not for silhouettes, which measured the same.
template <class L>
__device__ __forceinline__ void pool_push2(L& W, uint32_t& size, bool yes, bool near, uint32_t a, float key)
{
    const uint64_t all = __builtin_amdgcn_ballot_w64(yes), top = __builtin_amdgcn_ballot_w64(yes && near);
    const uint32_t nfar = (uint32_t)__popcll(all & ~top);
    const uint32_t at = size + (near ? nfar + rank_in(top) : rank_in(all & ~top));
    if (yes) {
        W.pool[at] = a;
        W.pkey[at] = (uint16_t)(__float_as_uint(key) >> 16);
    }
    size += (uint32_t)__popcll(all);
}

// queries waiting to enter (todo: a slot per bit) into the pool, up to `add`
// of them
template <class L>
__device__ __forceinline__ void pool_feed(L& W, uint32_t& size, uint64_t& todo, uint32_t add)
{
    const uint32_t lane = threadIdx.x & 63;
    const bool in = ((todo >> lane) & 1ull) && rank_in(todo) < add;
    todo &= ~__builtin_amdgcn_ballot_w64(in);
    pool_push(W, size, in, lane << 24, 0.0f);
}

// how many items to pop so that their children fit: 32, fewer near the
// pool's end, and one at a time in its reserve of 64 (a depth-first search of
// one item needs at most one place per tree level)
__device__ __forceinline__ uint32_t pool_take(uint32_t size, uint32_t cap)
{
    const uint32_t room = cap - 64, k = min(32u, size);
    return size + k <= room ? k : size < room ? min(k, room - size) : 1u;
}

// ------------------------------------------------------------ closest point

// query_device(nearest) (query.cuh:238-318) by one lane: near child first,
// each node's leaves at once, with only nodes within the squared distance w.
// st: 128 words of LDS (a stack of 64 nodes and keys: a path of a Karras tree
// holds at most 64 internal nodes).
template <int DIM>
__device__ inline void lane_nearest(const TreeView& t, v3 p, float w, uint32_t* st, float& best, uint32_t& best_idx)
{
    best = F_INF;
    best_idx = INVALID;
    uint32_t sp = 0, node = 0;
    for (uint32_t it = 0; it < 2 * t.n_leaves + 64 && node < t.n_leaves - 1; ++it) {
        const NodeRec nr = load_node(t.tnode, node);
        const float Lmd = box_mindist(nr.L, p), Rmd = box_mindist(nr.R, p);
        const float Lmm = box_minmaxdist(nr.L, p), Rmm = box_minmaxdist(nr.R, p);
        const bool cL = Lmd <= Rmm, cR = Rmd <= Lmm; // query.cuh:279, :297
        uint32_t lf, lc, rf, rc;
        const bool lLeaf = as_leaf(nr.lref, 0u, lf, lc), rLeaf = as_leaf(nr.rref, 1u, rf, rc);
        if (cL && lLeaf && Lmd <= fmn(best, w))
            for (uint32_t k = 0; k < lc; ++k)
                cp_leaf<DIM>(t, lf + k, p, best, best_idx);
        if (cR && rLeaf && Rmd <= fmn(best, w))
            for (uint32_t k = 0; k < rc; ++k)
                cp_leaf<DIM>(t, rf + k, p, best, best_idx);
        const float b = fmn(best, w);
        const bool gL = cL && !lLeaf && Lmd <= b, gR = cR && !rLeaf && Rmd <= b;
        const bool lfirst = Lmd <= Rmd;
        if (gL && gR && sp < 64u) {
            st[2 * sp] = lfirst ? nr.rref : nr.lref;
            st[2 * sp + 1] = __float_as_uint(lfirst ? Rmd : Lmd);
            ++sp;
        }
        if (gL || gR) {
            node = gL && (lfirst || !gR) ? nr.lref : nr.rref;
            continue;
        }
        bool found = false;
        while (sp > 0 && !found) {
            --sp;
            node = st[2 * sp];
            found = __uint_as_float(st[2 * sp + 1]) <= b; // query.cuh:259
        }
        if (!found)
            break;
    }
}

// evaluates the last (up to 64) leaves of the wave's buffer; returns how many are left
template <bool STATS, int DIM>
__device__ __forceinline__ uint32_t cp_leaves(const TreeView& t, WaveLds& W, uint32_t nleaf, float scale, Counts& cnt)
{
    const uint32_t lane = threadIdx.x & 63, k = min(64u, nleaf);
    nleaf -= k;
    if (lane < k) {
        const uint32_t w = W.leaf[2 * (nleaf + lane)], slot = w >> 24;
        const float key = __uint_as_float(W.leaf[2 * (nleaf + lane) + 1]), b = __uint_as_float(W.bound[slot]);
        if (key <= b) {
            if (STATS)
                cnt.leaf += 1;
            const v3 p = W.point(slot);
            float d = F_INF;
            uint32_t id = INVALID;
            cp_leaf<DIM>(t, w & REF_MASK, p, d, id);
            if (id != INVALID && d <= b) {
                atomicMin(&W.best[slot], pack_best(d, id, key > d));
                atomicMin(&W.bound[slot], __float_as_uint(widened<DIM>(HwMath::sqrt(d), p, scale)));
            }
        }
    }
    return nleaf;
}

// query_device(nearest) (query.cuh:238-318) for the points in slots [0, nq)
// of a wave (WaveLds::start): W.best receives (squared distance, index).  Run
// by the whole wave.  Every box has geometry on (in 2D, within BVH_OFFSET of)
// each of its faces, so its minmaxdist bounds the answer from above: besides
// the reference's test against the sibling (query.cuh:279, :297) it lowers
// the query's bound before any leaf is reached.  Where a box's leaves are farther
// than it promises (slivers), the bound has passed over leaves that the answer
// may be among: a query that ends with its bound below its answer, or without
// an answer, is searched alone.
template <bool STATS, int DIM>
__device__ __forceinline__ void cp_wave(const TreeView& t, uint32_t nq, WaveLds& W, Counts& cnt, bool& overflow)
{
    const uint32_t lane = threadIdx.x & 63;
    if (t.n_leaves == 1) {
        if (lane < nq) {
            float d = F_INF;
            uint32_t id = INVALID;
            cp_leaf<DIM>(t, 0, W.point(lane), d, id);
            W.best[lane] = pack_best(d, id);
        }
        return;
    }
    const float scale = scene_scale(t);
    uint32_t size = 0, nleaf = 0;
    uint64_t todo = __builtin_amdgcn_ballot_w64(lane < nq);
    // every iteration pops a node of some query (each at most once) or
    // evaluates leaves; the bound only guards against a malformed tree
    const uint32_t cap_iters = 128u * t.n_leaves + 65536u;
    for (uint32_t it = 0;; ++it) {
        bool flush = nleaf >= CP_LEAF_RUN;
        if (!flush && size < 32u) {
            if (todo != 0ull)
                pool_feed(W, size, todo, CP_ADD);
            else if (nleaf > 0u)
                flush = true;
            else if (size == 0u)
                break;
        }
        if (flush) {
            nleaf = cp_leaves<STATS, DIM>(t, W, nleaf, scale, cnt);
            continue;
        }
        if (it >= cap_iters) {
            overflow = true;
            break;
        }
        const uint32_t k = pool_take(size, W.cap), side = lane & 1u;
        size -= k;
        uint32_t slot = 0, ref = 0;
        float md = F_INF, mm = F_INF, b = 0.0f;
        bool live = false;
        v3 p = mk(0.0f, 0.0f, 0.0f);
        if ((lane >> 1) < k) {
            const uint32_t at = size + (lane >> 1), w = W.pool[at], node = w & REF_MASK;
            slot = w >> 24;
            b = __uint_as_float(W.bound[slot]);
            live = __uint_as_float((uint32_t)W.pkey[at] << 16) <= b && node < t.n_leaves - 1;
            if (live) {
                p = W.point(slot);
                const ChildRec c = load_child(t.tnode, node, side);
                ref = c.ref;
                md = box_mindist(c.box, p);
                mm = box_minmaxdist_fast(c.box, p);
                if (STATS) {
                    cnt.node += side;
                    cnt.box += 1;
                }
            }
        }
        const float mo = pair_other(mm), m2 = fmn(mm, mo);
        if (live && m2 < b) {
            const float u = widened<DIM>(HwMath::sqrt(m2), p, scale);
            if (u < b) {
                if (side)
                    atomicMin(&W.bound[slot], __float_as_uint(u));
                b = u;
            }
        }
        uint32_t first, count;
        const bool go = live && md <= mo && md <= b, leaf = as_leaf(ref, side, first, count);
        const float other = pair_other(md);
        const bool lt = md < other, eq = md == other, near = lt || (eq && !side);
        pool_push2(W, size, go && !leaf, near, (slot << 24) | (ref & REF_MASK), md);
        list_push(W.leaf, nleaf, go && leaf, (slot << 24) | first, md);
        for (uint32_t j = 1; (t.flags & TREE_RUNS) && __ballot(go && leaf && j < count); ++j) {
            if (nleaf >= CP_LEAF_RUN)
                nleaf = cp_leaves<STATS, DIM>(t, W, nleaf, scale, cnt);
            list_push(W.leaf, nleaf, go && leaf && j < count, (slot << 24) | (first + j), md);
        }
    }
    // the pool is empty: its memory holds the stacks of the lone searches
    float d = F_INF, w = F_INF;
    uint32_t id = INVALID;
    bool alone = false;
    if (lane < nq) {
        const v3 p = W.point(lane);
        const bool hidden = unpack_best(W.best[lane], d, id);
        const float h = HwMath::sqrt(d);
        alone = hidden || id == INVALID || __uint_as_float(W.bound[lane]) < half_widened<DIM>(h, p, scale);
        if (id != INVALID)
            w = widened<DIM>(HwMath::sqrt(widened<DIM>(h, p, scale)), p, scale);
    }
    for (uint64_t todo = __ballot(alone); todo; todo = __ballot(alone)) {
        const uint32_t r = rank_in(todo);
        if (alone && r < W.cap / 128u) {
            const v3 p = W.point(lane);
            lane_nearest<DIM>(t, p, w, W.pool + 128 * r, d, id);
            W.best[lane] = pack_best(d, id);
            alone = false;
        }
    }
}

// ------------------------------------------------------------ silhouette

// query_device(nearest_silhouette) (query.cuh:325-423) by one lane: near child
// first, each node's leaves at once, with only nodes within the squared
// distance w, and internal nodes within the squared radius cap2.  st: 128
// words of LDS.
template <int DIM>
__device__ inline void lane_silhouette(const TreeView& t, v3 p, bool flip, float w, float cap2, uint32_t* st,
                                       float& best, uint32_t& best_e)
{
    best = F_INF;
    best_e = INVALID;
    Counts cnt;
    uint32_t sp = 0, node = 0;
    for (uint32_t it = 0; it < 2 * t.n_leaves + 64 && node < t.n_leaves - 1; ++it) {
        const NodeRec nr = load_node(t.tnode, node);
        const float Lmd = box_mindist(nr.L, p), Rmd = box_mindist(nr.R, p), b2 = fmn(best * best, w);
        const bool hL = Lmd <= b2 && cone_hit<DIM>(t, load_cone(t.tcone, node, 0u), p, nr.L, Lmd);
        const bool hR = Rmd <= b2 && cone_hit<DIM>(t, load_cone(t.tcone, node, 1u), p, nr.R, Rmd);
        uint32_t lf, lc, rf, rc;
        const bool lLeaf = as_leaf(nr.lref, 0u, lf, lc), rLeaf = as_leaf(nr.rref, 1u, rf, rc);
        if (hL && lLeaf)
            for (uint32_t k = 0; k < lc; ++k)
                sil_leaf<DIM>(t, lf + k, p, flip, best, best_e, cnt);
        if (hR && rLeaf)
            for (uint32_t k = 0; k < rc; ++k)
                sil_leaf<DIM>(t, rf + k, p, flip, best, best_e, cnt);
        const float nb2 = fmn(best * best, w);
        const bool gL = hL && !lLeaf && Lmd <= nb2 && Lmd <= cap2, gR = hR && !rLeaf && Rmd <= nb2 && Rmd <= cap2;
        const bool lfirst = Lmd <= Rmd;
        if (gL && gR && sp < 64u) {
            st[2 * sp] = lfirst ? nr.rref : nr.lref;
            st[2 * sp + 1] = __float_as_uint(lfirst ? Rmd : Lmd);
            ++sp;
        }
        if (gL || gR) {
            node = gL && (lfirst || !gR) ? nr.lref : nr.rref;
            continue;
        }
        bool found = false;
        while (sp > 0 && !found) {
            --sp;
            node = st[2 * sp];
            found = __uint_as_float(st[2 * sp + 1]) <= nb2; // query.cuh:347
        }
        if (!found)
            break;
    }
}

// a silhouette at distance d of a leaf with box bound key becomes a candidate of query `slot`
template <int DIM>
__device__ __forceinline__ void sil_found(WaveLds& W, uint32_t slot, v3 p, float scale, float key, float d, uint32_t id)
{
    atomicMin(&W.best[slot], pack_best(d, id, key > d * d));
    atomicMin(&W.bound[slot], __float_as_uint(widened<DIM>(d, p, scale)));
}

// evaluates the last (up to 64) leaves of the wave's buffer; returns how many
// are left.  3D: a leaf owns 0..3 edges; the wave lists the edges of all its
// leaves as slots and tests one per lane in rounds of 64.
template <bool STATS, int DIM>
__device__ __forceinline__ uint32_t sil_leaves(const TreeView& t, WaveLds& W, uint32_t nleaf, float scale, bool flip,
                                               Counts& cnt)
{
    const uint32_t lane = threadIdx.x & 63, k = min(64u, nleaf);
    nleaf -= k;
    uint32_t w = 0, es = 0, ec = 0;
    float key = F_INF;
    bool mine = false;
    if (lane < k) {
        w = W.leaf[2 * (nleaf + lane)];
        key = __uint_as_float(W.leaf[2 * (nleaf + lane) + 1]);
        mine = key <= __uint_as_float(W.bound[w >> 24]) && (w & REF_MASK) < t.n_leaves;
    }
    const uint32_t slot = w >> 24, j = w & REF_MASK;
    if (STATS && mine)
        cnt.leaf += 1;
    if (DIM == 2) {
        if (mine) {
            const v3 p = W.point(slot);
            float d = F_INF;
            uint32_t id = INVALID;
            Counts c;
            sil_leaf<DIM>(t, j, p, flip, d, id, c);
            if (STATS)
                cnt.edge += c.edge;
            if (id != INVALID && d * d <= __uint_as_float(W.bound[slot]))
                sil_found<DIM>(W, slot, p, scale, key, d, id);
        }
        return nleaf;
    }
    if (mine) {
        es = __float_as_uint(t.tleaf[3 * j + 1].w);
        ec = min(__float_as_uint(t.tleaf[3 * j + 2].w), 3u);
    }
    if (STATS)
        cnt.edge += ec;
    const uint64_t b0 = __builtin_amdgcn_ballot_w64((ec & 1u) != 0u), b1 = __builtin_amdgcn_ballot_w64((ec & 2u) != 0u);
    const uint32_t off = rank_in(b0) + 2u * rank_in(b1);
    const uint32_t total = (uint32_t)__popcll(b0) + 2u * (uint32_t)__popcll(b1);
    uint32_t* list = W.leaf + 2 * nleaf; // the popped entries' words: owner lane << 26 | edge
    for (uint32_t base = 0; base < total; base += 64) {
#pragma unroll
        for (uint32_t i = 0; i < 3; ++i) {
            const uint32_t at = off + i - base;
            if (i < ec && at < 64u)
                list[at] = (lane << 26) | (es + i);
        }
        const bool on = lane < min(64u, total - base);
        const uint32_t l = on ? list[lane] : 0u, e = l & 0x03FFFFFFu;
        const uint32_t s = (uint32_t)__shfl((int)slot, (int)(l >> 26), 64);
        const float kk = __shfl(key, (int)(l >> 26), 64);
        if (on) {
            const v3 p = W.point(s);
            const float b = __uint_as_float(W.bound[s]);
            const float4 A = t.tedge[4 * e], B = t.tedge[4 * e + 1];
            const v3 pa = mk(A.x, A.y, A.z), pb = mk(B.x, B.y, B.z);
            v3 cp;
            const float d = closest_point_segment(pa, pb, p, cp);
            if (d * d <= b) {
                bool sil = (__float_as_uint(B.w) & 3u) != 3u; // a boundary edge is always a silhouette
                if (!sil) {
                    const float4 N0 = t.tedge[4 * e + 2], N1 = t.tedge[4 * e + 3];
                    sil = is_silhouette_edge(pa, pb, mk(N0.x, N0.y, N0.z), mk(N1.x, N1.y, N1.z),
                                             mk(p.x - cp.x, p.y - cp.y, p.z - cp.z), d, flip);
                }
                if (sil)
                    sil_found<DIM>(W, s, p, scale, kk, d, __float_as_uint(A.w));
            }
        }
    }
    return nleaf;
}

// query_device(nearest_silhouette) (query.cuh:325-423) for the queries of a
// wave, a slot per bit of `all` (WaveLds::start): W.best receives (distance,
// silhouette id).  Run by the whole wave.
// MODE 0: plain.  MODE 1: `cap` (per lane) is a hint: the search within it
// first; a query with no answer there enters again without it (the pool
// spreads it over all lanes, so the rest of the wave does not wait for one
// lane).  Outputs equal MODE 0's.  MODE 2: `cap` is hard: internal nodes
// farther than it are not visited.
template <bool STATS, int DIM, int MODE>
__device__ __forceinline__ void sil_wave(const TreeView& t, uint64_t all, bool flip, float cap, WaveLds& W,
                                         Counts& cnt, bool& overflow)
{
    const uint32_t lane = threadIdx.x & 63;
    const bool valid = (all >> lane) & 1ull;
    if (t.n_leaves == 1) {
        if (valid) {
            const v3 p = W.point(lane);
            const box3 b = ldbox2(t.nbox, 0);
            const float4 c0 = t.ncone[0], c1 = t.ncone[1];
            float d = F_INF;
            uint32_t id = INVALID;
            if (cone_valid(c0.w) && overlap_dim<DIM>(c0, c1.x, p, b, box_mindist(b, p)))
                sil_leaf<DIM>(t, 0, p, flip, d, id, cnt);
            W.best[lane] = pack_best(d, id);
        }
        return;
    }
    if (!(cap >= 0.0f))
        cap = F_INF;
    const float scale = scene_scale(t);
    if (MODE == 1 && valid && cap < F_INF)
        W.bound[lane] = __float_as_uint(widened<DIM>(cap, W.point(lane), scale));
    if (MODE == 2 && valid)
        W.cap2()[lane] = cap * cap;
    uint32_t size = 0, nleaf = 0;
    uint64_t todo = all;
    bool hinted = MODE == 1;
    // every iteration pops a node of some query (each at most once, twice
    // with a hint) or evaluates leaves; the bound only guards against a
    // malformed tree
    const uint32_t cap_iters = 128u * t.n_leaves + 65536u;
    for (uint32_t it = 0;; ++it) {
        if (nleaf >= SIL_LEAF_RUN || (nleaf > 0u && todo == 0ull && size < 32u)) {
            nleaf = sil_leaves<STATS, DIM>(t, W, nleaf, scale, flip, cnt);
            continue;
        }
        if (size == 0u && todo == 0ull) {
            if (!hinted)
                break;
            // the queries without an answer within their hint enter again
            hinted = false;
            float d = F_INF;
            uint32_t id = INVALID;
            if (valid)
                unpack_best(W.best[lane], d, id);
            const bool again = valid && cap < F_INF && !(id != INVALID && d <= cap);
            if (again)
                W.bound[lane] = __float_as_uint(id != INVALID ? widened<DIM>(d, W.point(lane), scale) : F_INF);
            todo = __builtin_amdgcn_ballot_w64(again);
            continue;
        }
        if (it >= cap_iters) {
            overflow = true;
            break;
        }
        if (size < 32u && todo != 0ull)
            pool_feed(W, size, todo, SIL_ADD);
        const uint32_t k = pool_take(size, W.cap), side = lane & 1u;
        size -= k;
        uint32_t slot = 0, ref = 0;
        float md = F_INF;
        bool go = false;
        if ((lane >> 1) < k) {
            const uint32_t at = size + (lane >> 1), w = W.pool[at], node = w & REF_MASK;
            slot = w >> 24;
            const float b = __uint_as_float(W.bound[slot]);
            if (__uint_as_float((uint32_t)W.pkey[at] << 16) <= b && node < t.n_leaves - 1) {
                const v3 p = W.point(slot);
                const ChildRec c = load_child(t.tnode, node, side);
                const ConeRec cone = load_cone(t.tcone, node, side);
                ref = c.ref;
                md = box_mindist(c.box, p);
                go = md <= b && cone_hit<DIM>(t, cone, p, c.box, md);
                if (STATS) {
                    cnt.node += side;
                    cnt.cone += side;
                    cnt.box += 1;
                }
            }
        }
        uint32_t first, count;
        const bool leaf = as_leaf(ref, side, first, count);
        const float other = pair_other(md);
        const bool lt = md < other, eq = md == other, near = lt || (eq && !side);
        const bool down = go && !leaf && (MODE != 2 || md <= W.cap2()[slot]);
        pool_push(W, size, down && !near, (slot << 24) | (ref & REF_MASK), md);
        pool_push(W, size, down && near, (slot << 24) | (ref & REF_MASK), md);
        list_push(W.leaf, nleaf, go && leaf, (slot << 24) | first, md);
        for (uint32_t j = 1; (t.flags & TREE_RUNS) && __ballot(go && leaf && j < count); ++j) {
            if (nleaf >= SIL_LEAF_RUN)
                nleaf = sil_leaves<STATS, DIM>(t, W, nleaf, scale, flip, cnt);
            list_push(W.leaf, nleaf, go && leaf && j < count, (slot << 24) | (first + j), md);
        }
    }
    // hidden answers, and answers at distance 0, where the reference stops at
    // the first edge it meets (scene.cuh:791): the lone search decides
    float d = F_INF;
    uint32_t id = INVALID;
    const bool hidden = valid && unpack_best(W.best[lane], d, id);
    bool alone = hidden || (id != INVALID && !(d * d > 0.0f));
    for (uint64_t left = __ballot(alone); left; left = __ballot(alone)) {
        const uint32_t r = rank_in(left);
        if (alone && r < W.cap / 128u) {
            const v3 p = W.point(lane);
            lane_silhouette<DIM>(t, p, flip, widened<DIM>(HwMath::sqrt(__uint_as_float(W.bound[lane])), p, scale),
                                 MODE == 2 ? W.cap2()[lane] : F_INF, W.pool + 128 * r, d, id);
            W.best[lane] = pack_best(d, id);
            alone = false;
        }
    }
}

// ------------------------------------------------------------ rays

// LDS of a wave's rays: as WaveLds, with the origin, the reciprocal and the
// direction per query slot, and so a smaller pool, which does: a ray visits few
// nodes (20 on the 1M-triangle torus).  2^22 random rays at that torus / a camera's
// at the torus over a ground plane / random ones at 64 tori over it, in ms: as it
// is 1.00 / 2.62 / 4.84; a pool of 256 1.00 / 6.62 / 4.89, of 512 (21 waves per CU)
// 1.07 / 2.82 / 4.87; RAY_ADD 16 / 24 / 48 / 64: 1.00 / 2.86 / 5.22, 1.01 / 3.02 /
// 5.30, 1.02 / 2.87 / 5.31, 1.02 / 2.90 / 5.38; RAY_LEAF_RUN 16 / 40: 1.01 / 2.53 /
// 4.61, 1.01 / 2.77 / 5.21, but 2D rays (the soup of 2,000 segments: 0.72) 0.75 / 0.68.
constexpr uint32_t RAY_LEAF_RUN = 24, RAY_ADD = 32;
struct RayLds {
    unsigned long long* best; // (t, triangle)
    uint32_t *pool, *leaf, *bound;
    uint32_t *met, *close; // a bit per slot each, see ray_check
    uint16_t* pkey;
    float* q; // origin, reciprocal direction, direction: 9 rows of 64
    uint32_t cap;
    static constexpr uint32_t CAP = 384;
    static constexpr uint32_t WORDS = 128 + 2 * LEAF_CAP + 64 + 576 + CAP + CAP / 2;
    __device__ __forceinline__ explicit RayLds(uint32_t* base)
    {
        best = reinterpret_cast<unsigned long long*>(base);
        leaf = base + 128;
        bound = leaf + 2 * LEAF_CAP;
        q = reinterpret_cast<float*>(bound + 64);
        pool = bound + 640;
        pkey = reinterpret_cast<uint16_t*>(pool + CAP);
        met = leaf + 2 * LEAF_CAP - 4; // the leaf buffer is never that full
        close = met + 2;
        cap = CAP;
    }
    __device__ __forceinline__ v3 row3(uint32_t r, uint32_t s) const
    {
        return mk(q[64 * r + s], q[64 * r + 64 + s], q[64 * r + 128 + s]);
    }
    __device__ __forceinline__ v3 origin(uint32_t s) const { return row3(0, s); }
    __device__ __forceinline__ v3 inv(uint32_t s) const { return row3(3, s); }
    __device__ __forceinline__ v3 dir(uint32_t s) const { return row3(6, s); }
    __device__ __forceinline__ void start(uint32_t s, v3 o, v3 d, v3 i, float max_dist)
    {
        const v3 a[3] = {o, i, d};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            q[64 * (3 * k) + s] = a[k].x;
            q[64 * (3 * k + 1) + s] = a[k].y;
            q[64 * (3 * k + 2) + s] = a[k].z;
        }
        best[s] = pack_best(F_INF, INVALID);
        bound[s] = __float_as_uint(max_dist);
    }
};
static_assert(RAY_LEAF_RUN - 1 + 64 <= LEAF_CAP - 2, "room for the bits behind the leaves");
// LDS is dealt in pieces of 1,280 B: one word more would leave 21 waves per CU (9 % more time)
static_assert(RayLds::WORDS * sizeof(uint32_t) <= 5 * 1280, "25 waves per CU");
static_assert(RayLds::WORDS % 2 == 0, "8-byte aligned answers");

// the scene's hit test of the leaf at sorted position j: t, (u, v) and the original index
template <int DIM>
__device__ __forceinline__ bool ray_leaf(const TreeView& t, uint32_t j, v3 ro, v3 rd, float& th, float& uh, float& vh,
                                         uint32_t& id)
{
    if (j >= t.n_leaves)
        return false;
    const float4 a = t.tleaf[3 * j], b = t.tleaf[3 * j + 1];
    id = __float_as_uint(a.w);
    vh = 0.0f;
    if (DIM == 3) {
        const float4 c = t.tleaf[3 * j + 2];
        return ray_triangle(ro, rd, mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), mk(c.x, c.y, c.z), th, uh, vh);
    }
    return ray_segment(ro, rd, mk(a.x, a.y, 0.0f), mk(b.x, b.y, 0.0f), th, uh);
}

// query_device(ray_intersect) (query.cuh:79-169) by one lane: near child
// first, a node's leaves at once in that order.  st: 128 words of LDS.
template <int DIM>
__device__ inline void lane_ray(const TreeView& t, v3 ro, v3 rd, v3 inv, float max_dist, uint32_t* st, float& tbest,
                                uint32_t& bidx)
{
    tbest = F_INF;
    bidx = INVALID;
    auto leaf = [&](uint32_t j) {
        float th, uh, vh;
        uint32_t id;
        if (ray_leaf<DIM>(t, j, ro, rd, th, uh, vh, id) && th < max_dist && (th < tbest || (th == tbest && id < bidx))) {
            tbest = th;
            bidx = id;
        }
    };
    uint32_t sp = 0, node = 0;
    for (uint32_t it = 0; it < 2 * t.n_leaves + 64 && node < t.n_leaves - 1; ++it) {
        const NodeRec nr = load_node(t.tnode, node);
        float Ld = F_INF, Rd = F_INF;
        const bool bL = box_ray(nr.L, ro, inv, max_dist, Ld), bR = box_ray(nr.R, ro, inv, max_dist, Rd);
        const bool Lh = bL && Ld <= tbest, Rh = bR && Rd <= tbest;
        uint32_t lf, lc, rf, rc;
        const bool lLeaf = as_leaf(nr.lref, 0u, lf, lc), rLeaf = as_leaf(nr.rref, 1u, rf, rc);
        const bool rfirst = Lh && Rh && Rd < Ld; // nearer child first, as query.cuh:136-149
        if (rfirst) {
            if (Rh && rLeaf)
                for (uint32_t k = 0; k < rc; ++k)
                    leaf(rf + k);
            if (Lh && lLeaf && Ld <= tbest)
                for (uint32_t k = 0; k < lc; ++k)
                    leaf(lf + k);
        } else {
            if (Lh && lLeaf)
                for (uint32_t k = 0; k < lc; ++k)
                    leaf(lf + k);
            if (Rh && rLeaf && Rd <= tbest)
                for (uint32_t k = 0; k < rc; ++k)
                    leaf(rf + k);
        }
        const bool gL = Lh && !lLeaf && Ld <= tbest, gR = Rh && !rLeaf && Rd <= tbest;
        const bool lnear = bL && (!bR || !(Rd < Ld));
        if (gL && gR && sp < 64u) {
            st[2 * sp] = lnear ? nr.rref : nr.lref;
            st[2 * sp + 1] = __float_as_uint(lnear ? Rd : Ld);
            ++sp;
        }
        if (gL || gR) {
            node = gL && (lnear || !gR) ? nr.lref : nr.rref;
            continue;
        }
        bool found = false;
        while (sp > 0 && !found) {
            --sp;
            node = st[2 * sp];
            found = __uint_as_float(st[2 * sp + 1]) <= tbest; // query.cuh:106
        }
        if (!found)
            break;
    }
}

// 2D: a segment is hit up to 1e-3 of its length past its ends, where its box ends
// BVH_OFFSET past them: a ray may hit a segment longer than 1 (at most the
// scene's diagonal) up to this much before it enters its box, by the distance
// along the ray's reciprocals, and at most the time it takes across the scene.
// 2^20 rays on 20,000 segments of a curve: 0.242 -> 0.249 ms, on 2,000 of a soup
// 0.69 -> 0.74.
__device__ __forceinline__ float past_end(v3 inv, float scale)
{
    auto finite = [](float x) { return dm::fabs_(x) < F_INF ? dm::fabs_(x) : 0.0f; };
    const float length = 2.83f * scale, r = 1.01e-3f * length;
    return fmn(r * fmx(finite(inv.x), finite(inv.y)),
               (length + r + 4.0f * BVH_OFFSET) * 1.00001f * fmn(dm::fabs_(inv.x), dm::fabs_(inv.y)));
}

// tests the last (up to 64) leaves of the wave's buffer; returns how many are
// left.  A hit at t becomes a candidate of its ray, whose bound falls to a
// little more than t (the rounding of box and triangle parameters: see the
// hidden leaves above; in 2D past_end too); any hit ends the ray with ANY.  Where a ray grazes a
// sliver, rounding knows no such bound: a triangle is hit while its determinant
// is FLT_EPSILON, and the parameter computed for it may be any amount before its
// box.  The lone search reports such a hit if it happens to meet that leaf before
// the true one; here a leaf whose box lies well behind a hit found is left out.
// In 50M simulated rays aimed along slivers the two differ in 110, and in all of
// them this search has the hit that 64 bits give.  A bound wide enough for the
// largest such error gives the lone search's answer and costs 2 % on 2^20 even
// triangles, 80 % on a rough sphere and three quarters of the speed where a
// ground plane joins small meshes.
template <bool STATS, int DIM, bool ANY>
__device__ __forceinline__ uint32_t ray_leaves(const TreeView& t, RayLds& W, uint32_t nleaf, float scale, Counts& cnt)
{
    const uint32_t lane = threadIdx.x & 63, k = min(64u, nleaf);
    nleaf -= k;
    if (lane < k) {
        const uint32_t w = W.leaf[2 * (nleaf + lane)], slot = w >> 24;
        const float key = __uint_as_float(W.leaf[2 * (nleaf + lane) + 1]), b = __uint_as_float(W.bound[slot]);
        if (key <= b) {
            if (STATS)
                cnt.leaf += 1;
            const v3 o = W.origin(slot);
            float th, uh, vh;
            uint32_t id;
            if (ray_leaf<DIM>(t, w & REF_MASK, o, W.dir(slot), th, uh, vh, id) && th < b) {
                th += 0.0f; // -0 counts as 0
                atomicMin(&W.best[slot], pack_best(th, id, key > th));
                if (ANY)
                    W.bound[slot] = 0x7FC00000u; // NaN: no key is below it
                else
                    atomicMin(&W.bound[slot],
                              __float_as_uint(th * 1.0001f +
                                              1e-5f * fmx(scale, fmx(dm::fabs_(o.x),
                                                                     fmx(dm::fabs_(o.y), dm::fabs_(o.z)))) +
                                              (DIM == 2 ? past_end(W.inv(slot), scale) : 0.0f)));
            }
        }
    }
    return nleaf;
}

// The same leaves for rays whose answer is hidden, which enter once more to see
// whether the lone search could have missed it: it meets the answer's leaf unless
// something else that it may have found lies before that leaf's box.  So a ray
// needs the lone search only if another hit lies within half of what its bound is
// widened by (close), or the answer's box lies farther than that (not met).  On
// flat faces along the axes half of the hits are hidden and few need it.  1024 x
// 1024 rays of an image on a floor of 8,192 triangles and two boxes, alone for
// every hidden answer -> so: 0.37 -> 0.15 ms (one ray per lane for all: 0.11), in a
// room 0.47 -> 0.18 (0.26), a mesh of 2^20 triangles above a ground plane seen from a
// camera 6.7 -> 2.7 (4.3); where few answers are hidden it costs nothing measurable.
template <int DIM>
__device__ __forceinline__ uint32_t ray_check(const TreeView& t, RayLds& W, uint32_t nleaf, float scale)
{
    const uint32_t lane = threadIdx.x & 63, k = min(64u, nleaf);
    nleaf -= k;
    if (lane < k) {
        const uint32_t w = W.leaf[2 * (nleaf + lane)], slot = w >> 24;
        const float key = __uint_as_float(W.leaf[2 * (nleaf + lane) + 1]);
        const v3 o = W.origin(slot);
        float best, th, uh, vh;
        uint32_t best_id, id;
        unpack_best(W.best[slot], best, best_id);
        // (twice half is within the whole, so that no hidden hit this close is left out)
        const float near = best * 1.00004f + 4e-6f * fmx(scale, fmx(dm::fabs_(o.x), fmx(dm::fabs_(o.y), dm::fabs_(o.z))));
        if (ray_leaf<DIM>(t, w & REF_MASK, o, W.dir(slot), th, uh, vh, id) && (id == best_id ? key : th) <= near)
            atomicOr(&(id == best_id ? W.met : W.close)[slot >> 5], 1u << (slot & 31u));
    }
    return nleaf;
}

// query_device(ray_intersect) (query.cuh:79-169) for the rays of a wave, a
// slot per bit of `all` (RayLds::start): W.best receives (t, triangle).  Run
// by the whole wave.  A ray with a negative or NaN max_dist hits nothing.
template <bool STATS, int DIM, bool ANY>
__device__ __forceinline__ void ray_wave(const TreeView& t, uint64_t all, float max_dist, RayLds& W, Counts& cnt,
                                         bool& overflow)
{
    const uint32_t lane = threadIdx.x & 63, side = lane & 1u;
    const bool valid = ((all >> lane) & 1ull) && max_dist >= 0.0f;
    uint32_t size = 0, nleaf = 0;
    const float scale = scene_scale(t);
    const uint32_t cap_iters = 128u * t.n_leaves + 65536u;
    // the rays of `todo` from the root on, their leaves in batches to `leaves`
    auto search = [&](uint64_t todo, auto leaves) {
        for (uint32_t it = 0;; ++it) {
            bool flush = nleaf >= RAY_LEAF_RUN;
            if (!flush && size < 32u) {
                if (todo != 0ull)
                    pool_feed(W, size, todo, RAY_ADD);
                else if (nleaf > 0u)
                    flush = true;
                else if (size == 0u)
                    break;
            }
            if (flush) {
                leaves();
                continue;
            }
            if (it >= cap_iters) {
                overflow = true;
                break;
            }
            const uint32_t k = pool_take(size, W.cap);
            size -= k;
            uint32_t slot = 0, ref = 0;
            float dist = F_INF;
            bool go = false;
            if ((lane >> 1) < k) {
                const uint32_t at = size + (lane >> 1), w = W.pool[at], node = w & REF_MASK;
                slot = w >> 24;
                const float b = __uint_as_float(W.bound[slot]);
                if (__uint_as_float((uint32_t)W.pkey[at] << 16) <= b && node < t.n_leaves - 1) {
                    const ChildRec c = load_child(t.tnode, node, side);
                    ref = c.ref;
                    go = box_ray(c.box, W.origin(slot), W.inv(slot), b, dist);
                    if (STATS) {
                        cnt.node += side;
                        cnt.box += 1;
                    }
                }
            }
            dist = go ? dist : F_INF;
            uint32_t first, count;
            const bool leaf = as_leaf(ref, side, first, count);
            const float other = pair_other(dist);
            const bool lt = dist < other, eq = dist == other, near = lt || (eq && !side);
            pool_push2(W, size, go && !leaf, near, (slot << 24) | (ref & REF_MASK), dist);
            list_push(W.leaf, nleaf, go && leaf, (slot << 24) | first, dist);
            for (uint32_t j = 1; (t.flags & TREE_RUNS) && __ballot(go && leaf && j < count); ++j) {
                if (nleaf >= RAY_LEAF_RUN)
                    leaves();
                list_push(W.leaf, nleaf, go && leaf && j < count, (slot << 24) | (first + j), dist);
            }
        }
    };
    auto test = [&] { nleaf = ray_leaves<STATS, DIM, ANY>(t, W, nleaf, scale, cnt); };
    if (t.n_leaves == 1) { // the only leaf is tested without its box, as in the reference
        list_push(W.leaf, nleaf, valid && lane < 32u, lane << 24, 0.0f);
        if (nleaf)
            test();
        list_push(W.leaf, nleaf, valid && lane >= 32u, lane << 24, 0.0f);
        if (nleaf)
            test();
        return;
    }
    search(__builtin_amdgcn_ballot_w64(valid), test);
    if (ANY)
        return;
    float d = F_INF;
    uint32_t id = INVALID;
    bool alone = valid && unpack_best(W.best[lane], d, id);
    const uint64_t hidden = __ballot(alone);
    if (hidden == 0ull)
        return;
    if (lane < 4u)
        W.met[lane] = 0u; // and close
    search(hidden, [&] { nleaf = ray_check<DIM>(t, W, nleaf, scale); });
    if (alone) {
        alone = !((W.met[lane >> 5] >> (lane & 31u)) & 1u) || ((W.close[lane >> 5] >> (lane & 31u)) & 1u);
        W.best[lane] = pack_best(d, id);
    }
    for (uint64_t left = __ballot(alone); left; left = __ballot(alone)) {
        const uint32_t r = rank_in(left);
        if (alone && r < W.cap / 128u) {
            lane_ray<DIM>(t, W.origin(lane), W.dir(lane), W.inv(lane), max_dist, W.pool + 128 * r, d, id);
            W.best[lane] = pack_best(d + 0.0f, id);
            alone = false;
        }
    }
}

// ------------------------------------------------------------ launches

// the next chunk of nchunks for a wave of a persistent launch: its XCD's
// contiguous range first (x0: the block's XCD), then the other XCDs' ranges;
// xi counts the ranges exhausted (wave-uniform).  ctr: [0, 8) the ranges'
// counters (zero at launch).  INVALID when none is left.
__device__ __forceinline__ uint32_t take_chunk(uint32_t* ctr, uint32_t nchunks, uint32_t x0, uint32_t& xi)
{
    while (xi < 8u) {
        const uint32_t xx = (x0 + xi) & 7u;
        const uint32_t lo = (uint32_t)((uint64_t)nchunks * xx / 8u);
        const uint32_t hi = (uint32_t)((uint64_t)nchunks * (xx + 1u) / 8u);
        uint32_t k = 0;
        if ((threadIdx.x & 63u) == 0)
            k = atomicAdd(ctr + xx, 1u);
        k = uniform(k);
        if (k < hi - lo)
            return lo + k;
        ++xi;
    }
    return INVALID;
}
constexpr uint32_t CHUNK_CTR_WORDS = 8;

// How the queries of a launch over n are dealt to its waves: the queries per wave
// (64, or fewer where that would leave resident waves without work), and in bits
// 8 and up the logarithm of the run length, the queries in sequence in the
// visiting order that one wave gets.  Neighbours cost alike, and the costliest
// lie together (around the centre of a sphere): a wave that gets 64 of them in
// one run works on long after the others are done, while runs of one spread
// them over all waves.  Runs share tree records between their queries, though.
// Run length 1 where each resident wave has at most one chunk, twice that for
// each doubling of the chunks per wave, up to 2^most.  For 2^22 queries: closest
// point, 2^20 / 20,480 triangles, in runs of 1 / 4 / 64: 20.7 / 20.2 / 22.7 and
// 3.7 / 3.4 / 4.2 ms; silhouette, torus of 2^20 / sphere of 327,680, in runs of
// 1 / 16 / 64: 55 / 25 / 26 and 64 / 363 / 586 ms.  Rays come in the
// caller's order: 2^22 random ones do not care (1.00 ms in runs of 4 to 64, 1.16
// in runs of 1), 2048 x 2048 of an image do (0.38 ms in runs of 1 to 32, 0.58 in
// runs of 64; 632 x 632: 0.11 and 0.18), so 2^least = 4 and 2^most = 16.
struct Runs {
    uint32_t least, most;
};
constexpr Runs CP_RUNS{0, 2}, SIL_RUNS{0, 4}, RAY_RUNS{2, 4};
__host__ __device__ __forceinline__ uint32_t deal_queries(uint32_t n, uint32_t waves, Runs r)
{
    const uint32_t w = waves > 0u ? waves : 1u, k = n / w + (n % w ? 1u : 0u);
    if (k <= 64u)
        return k < 1u ? 1u : k;
    uint32_t run = r.least;
    while (run < r.most && (k >> (6u + run)) > 0u)
        ++run;
    return 64u | run << 8;
}

// Calls f(slot, valid) with the queries of each chunk of this wave.  One chunk
// per wave where there are waves enough; else (ctr, a persistent launch) the
// waves take chunks as they get free.
template <class F>
__device__ __forceinline__ void for_chunks(uint32_t n, uint32_t deal, uint32_t* ctr, F f)
{
    const uint32_t lane = threadIdx.x & 63, wpb = blockDim.x >> 6, w = threadIdx.x >> 6;
    const uint32_t qpw = deal & 255u, run = deal >> 8;
    const uint32_t waves = gridDim.x * wpb, nchunks = n / qpw + (n % qpw ? 1u : 0u);
    const uint32_t first = ((lane >> run) * nchunks << run) + (lane & ((1u << run) - 1u));
    auto chunk = [&](uint32_t c) {
        const uint32_t slot = first + (c << run);
        f(slot, lane < qpw && slot < n);
    };
    if (nchunks <= waves || !ctr) {
        const uint32_t c = uniform(xcd_remap(blockIdx.x, gridDim.x) * wpb + w);
        if (c < nchunks)
            chunk(c);
        return;
    }
    uint32_t xi = 0;
    for (uint32_t c = take_chunk(ctr, nchunks, blockIdx.x % 8u, xi); c != INVALID;
         c = take_chunk(ctr, nchunks, blockIdx.x % 8u, xi))
        chunk(c);
}

inline uint32_t nblocks(uint32_t n, uint32_t bs) { return (n + bs - 1) / bs; }

// grid of a search launch: a wave per chunk, or (persist) as many waves as
// are resident (wave_words words of LDS each, at most `per_simd` on a SIMD)
struct SearchGrid {
    dim3 grid, block;
    uint32_t deal; // deal_queries, or 0: from the count on the device
    size_t lds;
    bool persist;
};
inline SearchGrid search_grid(uint32_t n, uint32_t block, uint32_t wave_words, uint32_t n_cu, uint32_t per_simd,
                              bool may_persist, bool n_on_device, Runs runs)
{
    SearchGrid g;
    const uint32_t wpb = block / 64;
    g.lds = sizeof(uint32_t) * wpb * wave_words;
    const uint32_t per_cu = std::max(1u, std::min((uint32_t)(LDS_PER_CU / g.lds), per_simd * 4u / wpb));
    const uint32_t resident = n_cu * per_cu;
    g.deal = n_on_device ? 0u : deal_queries(n, resident * wpb, runs);
    const uint32_t blocks = nblocks(nblocks(n, g.deal ? g.deal & 255u : 1u), wpb);
    g.persist = may_persist && blocks > resident;
    g.grid = dim3(g.persist ? resident : blocks);
    g.block = dim3(block);
    return g;
}


} // namespace

#define SNCH_DISPATCH_DIM(dim, ...) \
    do {                            \
        if ((dim) == 3) {           \
            constexpr int DIM = 3;  \
            __VA_ARGS__;            \
        } else {                    \
            constexpr int DIM = 2;  \
            __VA_ARGS__;            \
        }                           \
    } while (0)

} // namespace snch
