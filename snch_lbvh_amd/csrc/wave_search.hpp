// Searches shared by the query kernels (query.hip, silhouette.hip, batch.hip):
// the restart-trail stack, closest point and closest silhouette for the lanes
// of a wave, and the chunks of a persistent launch.  Device code.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.hpp"
#include "traverse.hpp"

namespace snch {

namespace {

constexpr int SS = 16; // LDS stack entries per lane (rays)
constexpr uint32_t LDS_PER_CU = 160 * 1024;

__device__ __forceinline__ uint32_t xcd_remap(uint32_t b, uint32_t nb)
{
    const uint32_t X = 8, q = nb / X, r = nb % X, x = b % X, k = b / X;
    return x * q + (x < r ? x : r) + k;
}

// wave-uniform copy of lane 0's value (a scalar register)
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// A short stack with a restart trail (Laine 2010, "Restart trail for
// stackless BVH traversal"), for searches whose pruning bound only tightens:
// SSZ 4-B entries in a circular LDS column, and nothing in private memory.
// An entry is node << 8 | q for trees of at most 2^24 leaves (internal node
// ids < 2^24); q is an 8-bit lower bound of the key (a non-negative squared
// distance): the key's float bits >> 20 (exponent and 3 mantissa bits, the
// key truncated to 8 steps per octave) minus a base chosen per tree so that
// the 255 levels span 31 octaves below the squared scene diagonal; keys
// below that range store 0 (decoded as 0), keys above saturate at 255, so
// the decoded value never exceeds the key and a popped entry is never
// skipped wrongly.  A push onto a full stack overwrites the oldest
// entry (the shallowest level); the lost far children are found again
// through the trail and revisited from the root.  Per lane, one bit per tree
// level (root 0; a path holds at most 64 internal nodes):
//   T  at this level the near child is finished and the far child taken;
//   S  at this level only one child was descended (nothing left behind);
//   M  the levels whose far child sits in the stack (levels grow from the
//      stack's bottom to its top, so the top entry's level is M's highest).
// A level of the current path with neither T nor S set, and not in M, left
// its far child behind; when the stack runs empty the deepest such level j
// gets T and the search restarts from the root: levels above j follow the
// trail (T: far child; else near, re-pushing a surviving far child), and
// level j takes its far child.  Children survive only if they pass the
// pruning tests, which can only fail more often as the bound tightens, so a
// subtree left by the trail holds nothing new.
template <int BS, int SSZ>
struct TrailStack {
    uint32_t* lds;
    uint32_t top; // position of the next push (mod SSZ)
    uint32_t qbase;
    uint64_t T, S, M;
    uint32_t lv; // level of the current node

    __device__ __forceinline__ void init(uint32_t* base, uint32_t qb)
    {
        lds = base;
        qbase = qb;
        reset();
    }
    __device__ __forceinline__ void reset()
    {
        top = 0;
        T = S = M = 0ull;
        lv = 0;
    }
    __device__ __forceinline__ uint32_t enc(uint32_t n, float d) const
    {
        const uint32_t v = __float_as_uint(d) >> 20;
        const uint32_t q = v > qbase ? min(v - qbase, 255u) : 0u;
        return (n << 8) | q;
    }
    // the lower bound stored in an entry
    __device__ __forceinline__ float key(uint32_t e) const
    {
        const uint32_t q = e & 255u;
        return q ? __uint_as_float((q + qbase) << 20) : 0.0f;
    }
    __device__ __forceinline__ void push(uint32_t n, float d, uint32_t k)
    {
        lds[(top % SSZ) * BS] = enc(n, d);
        ++top;
        if (__popcll(M) >= SSZ)
            M &= M - 1ull; // the oldest entry was just overwritten
        M |= 1ull << k;
    }
    // pop the top entry (M != 0): its node and decoded key; the current
    // path ends at its level, whose near child is finished
    __device__ __forceinline__ void pop(uint32_t& n, float& d)
    {
        --top;
        const uint32_t e = lds[(top % SSZ) * BS];
        n = e >> 8;
        d = key(e);
        const uint32_t k = 63u - (uint32_t)__clzll(M);
        const uint64_t kb = 1ull << k;
        M &= ~kb;
        T = (T & (kb - 1ull)) | kb;
        S &= kb - 1ull;
        lv = k;
    }
    // the stack is empty: restart from the root for the deepest level of the
    // current path that left its far child behind; false when there is none
    __device__ __forceinline__ bool restart()
    {
        const uint64_t path = lv >= 63u ? ~1ull : ((2ull << lv) - 1ull) & ~1ull; // levels 1..lv
        const uint64_t Z = ~(T | S) & path;
        if (!Z)
            return false;
        const uint32_t j = 63u - (uint32_t)__clzll(Z);
        const uint64_t jb = 1ull << j;
        T = (T & (jb - 1ull)) | jb;
        S &= jb - 1ull;
        top = 0;
        lv = 0;
        return true;
    }
    // choose the child to descend from the current node (children at level
    // lv + 1), given which of the near (N) and far (F) children survive;
    // false: nothing to descend
    __device__ __forceinline__ bool descend(bool gN, bool gF, uint32_t nN, uint32_t nF, float dF, uint32_t& node)
    {
        if (!gN && !gF)
            return false;
        const uint32_t k = lv + 1u; // at most 63: the caller stops deeper paths
        const uint64_t kb = 1ull << k;
        if (T & kb) { // near finished before: the far child, if it survives
            if (!gF)
                return false;
            node = nF;
        } else if (gN && gF) {
            push(nF, dF, k);
            node = nN;
        } else if (gN) {
            S |= kb;
            node = nN;
        } else if (gF) { // off the trail: the near child no longer survives
            T = (T & (kb - 1ull)) | kb;
            S &= kb - 1ull;
            node = nF;
        } else {
            return false;
        }
        lv = k;
        return true;
    }
};

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
// waves.  Queries enter as the pool runs low: POOL_ADD at a time keeps few
// queries, and so few pending nodes, in flight (all 64 at once fill the pool
// and leave it popping one item at a time: 218 instead of 33 ms on the case
// below, with one lane per item; 4 or 16 at a time 33.5 and 34.6).
//
// Closest point, one lane per query with a stack -> pool: 2^22 queries on
// 2^20 triangles 46 -> 26 ms (VALU issue 0.78 of the SIMD cycles, 582 nodes
// per query), 65,536 on 20,480 triangles 2.1 -> 0.18 ms, 1,000 on 20,480
// triangles 0.83 -> 0.03 ms (there a launch lasted as long as the longest
// chain of dependent loads, about 2 us a node).
//
// The answer is that of the search one lane would make alone, near child
// first, each node's leaves at once, which skips a box as soon as its lower
// bound exceeds the best distance so far (lane_nearest below).  Where no
// rounding interferes that is the smallest (distance, id) of all leaves,
// whatever the order.  But a leaf's computed distance can lie below its box's
// computed lower bound by a few units in the last place of the coordinates
// ("hidden" leaves): among candidates that close, what the lone search finds
// first decides.  So the pool prunes with bounds widened by more than that
// rounding, which leaves no such candidate out, and where a hidden leaf has
// the smallest distance the lane repeats the search alone, from the widened
// bound (a few dozen nodes).
constexpr uint32_t POOL_ADD = 8;
constexpr uint32_t LEAF_CAP = 128; // leaf buffer entries: below 64 before a step, which adds at most 64

// smaller is better: the distance, ties to the smaller id (distances are not negative)
__device__ __forceinline__ unsigned long long pack_best(float d, uint32_t id)
{
    return ((unsigned long long)__float_as_uint(d) << 32) | id;
}
__device__ __forceinline__ void unpack_best(unsigned long long v, float& d, uint32_t& id)
{
    d = __uint_as_float((uint32_t)(v >> 32));
    id = (uint32_t)v;
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

// LDS of one wave, carved from the block's dynamic LDS: cap pool items (2
// words each: slot << 24 | node, key), the leaf buffer (2 words per entry:
// slot << 24 | leaf, key), and per query slot its answer, point, widened
// (squared) bound and the smallest distance of a hidden leaf
struct WaveLds {
    unsigned long long* best;
    uint32_t *pool, *leaf, *bound, *hidden;
    float* q; // x, y, z rows of 64
    uint32_t cap;
    static constexpr uint32_t FIXED = 128 + 2 * LEAF_CAP + 128 + 192; // words besides the pool
    __device__ __forceinline__ WaveLds(uint32_t* base, uint32_t cap_)
    {
        best = reinterpret_cast<unsigned long long*>(base);
        pool = base + 128;
        leaf = pool + 2 * cap_;
        bound = leaf + 2 * LEAF_CAP;
        hidden = bound + 64;
        q = reinterpret_cast<float*>(hidden + 64);
        cap = cap_;
    }
    __device__ __forceinline__ v3 point(uint32_t s) const { return mk(q[s], q[64 + s], q[128 + s]); }
    __device__ __forceinline__ void start(uint32_t s, v3 p)
    {
        q[s] = p.x;
        q[64 + s] = p.y;
        q[128 + s] = p.z;
        best[s] = pack_best(F_INF, INVALID);
        bound[s] = hidden[s] = __float_as_uint(F_INF);
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
__device__ __forceinline__ float scene_scale(const TreeView& t)
{
    const box3 b = ldbox2(t.nbox, 0);
    return fmx(fmx(fmx(dm::fabs_(b.lo.x), dm::fabs_(b.hi.x)), fmx(dm::fabs_(b.lo.y), dm::fabs_(b.hi.y))),
               fmx(dm::fabs_(b.lo.z), dm::fabs_(b.hi.z)));
}
// words of dynamic LDS of a wave with `depth` pool items per lane pair
inline uint32_t wave_lds_words(uint32_t depth) { return 2 * 32 * depth + WaveLds::FIXED; }

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
                atomicMin(&W.best[slot], pack_best(d, id));
                atomicMin(&W.bound[slot], __float_as_uint(widened<DIM>(HwMath::sqrt(d), p, scale)));
                if (key > d)
                    atomicMin(&W.hidden[slot], __float_as_uint(d));
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
// the query's bound before any leaf is reached.
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
    uint32_t size = 0, nleaf = 0, next = 0;
    // every iteration pops a node of some query (each at most once) or
    // evaluates leaves; the bound only guards against a malformed tree
    const uint32_t cap_iters = 128u * t.n_leaves + 65536u;
    for (uint32_t it = 0;; ++it) {
        const bool fed = next >= nq;
        if (nleaf >= 64u || (nleaf > 0u && fed && size < 32u)) {
            nleaf = cp_leaves<STATS, DIM>(t, W, nleaf, scale, cnt);
            continue;
        }
        if (size == 0u && fed)
            break;
        if (it >= cap_iters) {
            overflow = true;
            break;
        }
        if (size < 32u && !fed) {
            const uint32_t add = min(POOL_ADD, nq - next);
            list_push(W.pool, size, lane < add, (next + lane) << 24, 0.0f);
            next += add;
        }
        const uint32_t k = pool_take(size, W.cap), side = lane & 1u;
        size -= k;
        uint32_t slot = 0, ref = 0;
        float md = F_INF, mm = F_INF, b = 0.0f;
        bool live = false;
        v3 p = mk(0.0f, 0.0f, 0.0f);
        if ((lane >> 1) < k) {
            const uint32_t at = size + (lane >> 1), w = W.pool[2 * at], node = w & REF_MASK;
            slot = w >> 24;
            b = __uint_as_float(W.bound[slot]);
            live = __uint_as_float(W.pool[2 * at + 1]) <= b && node < t.n_leaves - 1;
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
        list_push(W.pool, size, go && !leaf && !near, (slot << 24) | (ref & REF_MASK), md);
        list_push(W.pool, size, go && !leaf && near, (slot << 24) | (ref & REF_MASK), md);
        list_push(W.leaf, nleaf, go && leaf, (slot << 24) | first, md);
        for (uint32_t j = 1; (t.flags & TREE_RUNS) && __ballot(go && leaf && j < count); ++j) {
            if (nleaf >= 64u)
                nleaf = cp_leaves<STATS, DIM>(t, W, nleaf, scale, cnt);
            list_push(W.leaf, nleaf, go && leaf && j < count, (slot << 24) | (first + j), md);
        }
    }
    // the pool is empty: its memory holds the stacks of the lone searches
    bool alone = false;
    if (lane < nq) {
        const uint32_t d = (uint32_t)(W.best[lane] >> 32);
        alone = d < __float_as_uint(F_INF) && W.hidden[lane] == d;
    }
    for (uint64_t todo = __ballot(alone); todo; todo = __ballot(alone)) {
        const uint32_t r = rank_in(todo);
        if (alone && r < W.cap / 64u) {
            const v3 p = W.point(lane);
            float d;
            uint32_t id;
            lane_nearest<DIM>(t, p, widened<DIM>(HwMath::sqrt(__uint_as_float(W.bound[lane])), p, scale),
                              W.pool + 128 * r, d, id);
            W.best[lane] = pack_best(d, id);
            alone = false;
        }
    }
}

// ------------------------------------------------------------ silhouette

// Per-wave LDS of the flattened leaf tests: one round of 64 edge slots (the
// edge, then its distance with the sign bit set when it is not a silhouette),
// the owner lane of each slot, and each owner's query point and bound.
struct EdgeLds {
    uint32_t edge[64];
    float d[64];
    uint8_t owner[64];
    float px[64], py[64], pz[64], bound[64];
};

// The leaf tests of the lanes with `mine` set, spread over every lane of the
// wave that runs this (all looping lanes, wave-uniformly): each owner lists
// the edges of its (at most two) leaves as a run of slots, and in rounds of
// 64 slots every lane computes the distance and the silhouette test of one,
// then each owner applies its results in its original edge order, so ties and
// the reference's early-out at distance 0 (scene.cuh:791) come out as in
// sil_leaf.  3D, leaves of one primitive each.
__device__ __forceinline__ void sil_leaves_wave(const TreeView& t, EdgeLds& L, bool mine, uint32_t la, bool ha,
                                                uint32_t lb, bool hb, v3 p, bool flip, float& best,
                                                uint32_t& best_e, Counts& cnt)
{
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    uint32_t ea = 0, eb = 0, sa = 0, sb = 0;
    if (mine && ha && la < t.n_leaves) {
        sa = __float_as_uint(t.tleaf[3 * la + 1].w);
        ea = __float_as_uint(t.tleaf[3 * la + 2].w);
    }
    if (mine && hb && lb < t.n_leaves) {
        sb = __float_as_uint(t.tleaf[3 * lb + 1].w);
        eb = __float_as_uint(t.tleaf[3 * lb + 2].w);
    }
    ea = min(ea, 3u);
    eb = min(eb, 3u);
    const uint32_t my = ea + eb; // 0..6
    const uint64_t b0 = __ballot(my & 1u), b1 = __ballot(my & 2u), b2 = __ballot(my & 4u);
    const uint32_t off = (uint32_t)__popcll(b0 & lt) + 2u * (uint32_t)__popcll(b1 & lt) + 4u * (uint32_t)__popcll(b2 & lt);
    const uint32_t total = (uint32_t)__popcll(b0) + 2u * (uint32_t)__popcll(b1) + 4u * (uint32_t)__popcll(b2);
    if (mine) {
        L.px[lane] = p.x;
        L.py[lane] = p.y;
        L.pz[lane] = p.z;
        L.bound[lane] = best;
        cnt.leaf += (ha ? 1u : 0u) + (hb ? 1u : 0u);
        cnt.edge += my;
    }
    const uint64_t helpers = __ballot(true);
    const uint32_t hr = (uint32_t)__popcll(helpers & lt), nh = (uint32_t)__popcll(helpers);
    bool stop = false; // best reached 0: the owner's remaining edges are skipped
    for (uint32_t base = 0; base < total; base += 64) {
        // this round's slots [base, base + 64) of every owner
        for (uint32_t k = 0; mine && k < my; ++k) {
            const uint32_t sl = off + k;
            if (sl >= base && sl < base + 64) {
                L.edge[sl - base] = k < ea ? sa + k : sb + (k - ea);
                L.owner[sl - base] = (uint8_t)lane;
            }
        }
        // every lane of the wave (LDS operations of one wave complete in order)
        const uint32_t n_round = min(64u, total - base);
        for (uint32_t r = hr; r < n_round; r += nh) {
            const uint32_t e = L.edge[r], o = L.owner[r];
            const v3 q = mk(L.px[o], L.py[o], L.pz[o]);
            const float b = L.bound[o], mr2 = b * b;
            const float4 A = t.tedge[4 * e], B = t.tedge[4 * e + 1];
            const uint32_t fl = __float_as_uint(B.w);
            const v3 pa = mk(A.x, A.y, A.z), pb = mk(B.x, B.y, B.z);
            v3 cp;
            const float d = closest_point_segment(pa, pb, q, cp);
            bool sil = (fl & 3u) != 3u; // a boundary edge is always a silhouette
            if (!sil && d * d <= mr2) {
                const float4 N0 = t.tedge[4 * e + 2], N1 = t.tedge[4 * e + 3];
                sil = is_silhouette_edge(pa, pb, mk(N0.x, N0.y, N0.z), mk(N1.x, N1.y, N1.z),
                                         mk(q.x - cp.x, q.y - cp.y, q.z - cp.z), d, flip);
            }
            L.d[r] = sil ? d : -d; // d >= 0: the sign bit carries "not a silhouette"
        }
        for (uint32_t k = 0; mine && !stop && k < my; ++k) {
            const uint32_t sl = off + k;
            if (sl < base || sl >= base + 64)
                continue;
            const float mr2 = best * best;
            if (!(0.0f < mr2)) {
                stop = true; // min_radius_squared (0) >= max_radius_squared
                break;
            }
            const float sd = L.d[sl - base];
            const float d = dm::fabs_(sd);
            if (d * d > mr2 || dm::signbit_(sd))
                continue;
            const uint32_t e = k < ea ? sa + k : sb + (k - ea);
            const uint32_t id = __float_as_uint(t.tedge[4 * e].w);
            if (d < best || (d == best && id < best_e)) {
                best = d;
                best_e = id;
            }
        }
    }
}


// query_device(nearest_silhouette) (query.cuh:325-423) for one query point.
// best / best_e receive the answer.  The stack is a TrailStack: SSZ entries
// in LDS and no private memory.  A finite radius `cap` prunes internal nodes
// farther than cap as well.  When the search within cap ends with
// best <= cap, every node that could hold a silhouette at least as close has
// been visited; otherwise (HINT) it searches again from the root with no cap
// and the bound found so far, or (hard cap, !HINT) it stops.  With index
// tie-breaking the answer equals the uncapped search.
template <int BS, int SSZ, bool STATS, int DIM, bool HINT, bool PARK>
__device__ __forceinline__ void sil_query(const TreeView& t, v3 p, bool flip, float cap, uint32_t* stk_col,
                                          EdgeLds* elds, float& best, uint32_t& best_e, Counts& cnt,
                                          bool& overflow)
{
    best = F_INF;
    best_e = INVALID;
    if (t.n_leaves == 1) {
        const box3 b = ldbox2(t.nbox, 0);
        const float4 c0 = t.ncone[0], c1 = t.ncone[1];
        if (cone_valid(c0.w) && overlap_dim<DIM>(c0, c1.x, p, b, box_mindist(b, p)))
            sil_leaf<DIM>(t, 0, p, flip, best, best_e, cnt);
        return;
    }
    if (!(cap >= 0.0f))
        cap = F_INF;
    float cap2 = cap * cap;
    TrailStack<BS, SSZ> st;
    st.init(stk_col, t.qbase);
    uint32_t node = 0;
    // a pass visits each internal node at most once; restarts add the paths
    // above lost far children (a few per query); the bound only guards
    // against an inconsistent tree, and hitting it is reported as an overflow
    const uint32_t cap_iters = 8 * t.n_leaves + 8192;
    uint32_t it = 0;
    // A lane whose node has leaf children to evaluate parks them (phase
    // `leaves`) until a quarter of the wave's looping lanes, or all of them,
    // are parked; the parked lanes then evaluate their leaves together and
    // decide the node's internal children with the bound found, exactly as
    // if the leaves had been evaluated at once.  The leaf code then runs on
    // many lanes at a time instead of on the few that reached a leaf (about
    // 5 of 64 on the 1M-triangle torus: 99.6 -> 89 ms).  Hard-capped searches
    // (!HINT: short, as in walk on stars) evaluate leaves at once.
    bool leaves = false;
    float Lmd = 0.0f, Rmd = 0.0f;
    bool hL = false, hR = false, lLeaf = false, rLeaf = false;
    uint32_t lref = 0, rref = 0, lf = 0, lc = 0, rf = 0, rc = 0;
    for (; it < cap_iters && node < t.n_leaves - 1;) {
        bool decide = false;
        if (!leaves) {
            ++it;
            const NodeRec nr = load_node(t.tnode, node);
            Lmd = box_mindist(nr.L, p);
            Rmd = box_mindist(nr.R, p);
            const float b2 = best * best;
            hL = Lmd <= b2;
            hR = Rmd <= b2;
            if (STATS) {
                cnt.node += 1;
                cnt.box += 2;
            }
            if (hL || hR) {
                if (STATS)
                    cnt.cone += 1;
                const float4 CL = t.tcone[4 * node], CR = t.tcone[4 * node + 1], Cr = t.tcone[4 * node + 2];
                // query.cuh:366-367
                if (DIM == 3 && (t.flags & TREE_FAST_CONE)) {
                    const float4 SC = t.tcone[4 * node + 3];
                    hL = hL && cone_valid(CL.w) &&
                         cone_overlap_fast(mk(CL.x, CL.y, CL.z), CL.w, SC.x, SC.y, Cr.x, p, nr.L, Lmd);
                    hR = hR && cone_valid(CR.w) &&
                         cone_overlap_fast(mk(CR.x, CR.y, CR.z), CR.w, SC.z, SC.w, Cr.y, p, nr.R, Rmd);
                } else {
                    hL = hL && cone_valid(CL.w) && overlap_dim<DIM>(CL, Cr.x, p, nr.L, Lmd);
                    hR = hR && cone_valid(CR.w) && overlap_dim<DIM>(CR, Cr.y, p, nr.R, Rmd);
                }
            }
            lref = nr.lref;
            rref = nr.rref;
            lLeaf = as_leaf(nr.lref, 0u, lf, lc);
            rLeaf = as_leaf(nr.rref, 1u, rf, rc);
            leaves = (hL && lLeaf) || (hR && rLeaf);
            decide = !leaves;
        }
        const uint64_t parked = __ballot(leaves), looping = __ballot(true);
        if (parked &&
            (!PARK || 4u * (uint32_t)__popcll(parked) >= (uint32_t)__popcll(looping) || parked == looping)) {
            // wave-uniform: the parked lanes' leaves are tested now
            const bool la = hL && lLeaf, ra = hR && rLeaf;
            const bool runs = __ballot(leaves && ((la && lc > 1) || (ra && rc > 1))) != 0;
            if (DIM == 3 && elds && !runs) {
                sil_leaves_wave(t, *elds, leaves, lf, la, rf, ra, p, flip, best, best_e, cnt);
            } else if (leaves) {
                if (la)
                    for (uint32_t k = 0; k < lc; ++k)
                        sil_leaf<DIM>(t, lf + k, p, flip, best, best_e, cnt);
                if (ra)
                    for (uint32_t k = 0; k < rc; ++k)
                        sil_leaf<DIM>(t, rf + k, p, flip, best, best_e, cnt);
            }
            decide = decide || leaves;
            leaves = false;
        }
        if (!decide)
            continue;
        // internal children to descend: within the bound and the cap
        const float nb2 = best * best;
        const bool gL = hL && !lLeaf && Lmd <= nb2 && Lmd <= cap2;
        const bool gR = hR && !rLeaf && Rmd <= nb2 && Rmd <= cap2;
        if ((gL || gR) && st.lv >= 63u) {
            overflow = true; // deeper than a Karras tree can be
            break;
        }
        const bool lfirst = Lmd <= Rmd;
        if (st.descend(lfirst ? gL : gR, lfirst ? gR : gL, lfirst ? lref : rref, lfirst ? rref : lref,
                       lfirst ? Rmd : Lmd, node))
            continue;
        bool found = false;
        while (st.M) {
            uint32_t nn;
            float dd;
            st.pop(nn, dd);
            if (dd <= best * best) { // query.cuh:347
                node = nn;
                found = true;
                break;
            }
        }
        if (found)
            continue;
        if (st.restart()) {
            node = 0;
            continue;
        }
        // the search within the cap is over: settled, or (HINT) search again
        // from the root with no cap and the bound found so far
        if (cap2 == F_INF || (best_e != INVALID && best <= cap) || !HINT)
            break;
        cap2 = F_INF;
        st.reset();
        node = 0;
    }
    overflow = overflow || it >= cap_iters;
}

// the next 64-query chunk of nchunks for a one-wave block of a persistent
// launch: its own XCD's contiguous range first (x0: the block's XCD), then
// the other XCDs' ranges; xi counts the ranges exhausted (wave-uniform).
// ctr: [0, 8) the ranges' counters.  INVALID when none is left.
__device__ __forceinline__ uint32_t take_chunk(uint32_t* ctr, uint32_t nchunks, uint32_t x0, uint32_t& xi)
{
    while (xi < 8u) {
        const uint32_t xx = (x0 + xi) & 7u;
        const uint32_t lo = (uint32_t)((uint64_t)nchunks * xx / 8u);
        const uint32_t hi = (uint32_t)((uint64_t)nchunks * (xx + 1u) / 8u);
        uint32_t k = 0;
        if (threadIdx.x == 0)
            k = atomicAdd(ctr + xx, 1u);
        k = uniform(k);
        if (k < hi - lo)
            return lo + k;
        ++xi;
    }
    return INVALID;
}

inline uint32_t nblocks(uint32_t n, uint32_t bs) { return (n + bs - 1) / bs; }

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
