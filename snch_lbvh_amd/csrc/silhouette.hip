// Closest-silhouette kernels (query.cuh:325-423): one block per chunk of
// queries, the persistent launches, and their dispatch.
#include "wave_search.hpp"

namespace snch {

namespace {

// MODE 0: plain search.  MODE 1: search within the radius seed[qi] first; a
// query not settled there searches again from the root with no cap and the
// bound found so far (bit-identical to MODE 0).  MODE 2: search within the
// radius only (a hard cap).  Keeping the second search in the same launch
// lets the rare unsettled queries (the costliest ones) overlap with the rest
// of the grid; a separate second launch over them measured ~30 ms slower on
// the 1M-triangle torus, all of it the tail of those few queries.  The plain
// kernel is held to 80 VGPRs (6 waves per SIMD), the others to 96.
template <int BS, bool STATS, int DIM, int MODE, int SSZ>
__global__ __launch_bounds__(BS, MODE == 0 && !STATS ? 6 : 5) void k_closest_silhouette(TreeView t, const float* __restrict__ q, uint32_t n,
                                                           uint32_t nq, int flip, const float* __restrict__ seed,
                                                           uint32_t* __restrict__ out_e, float* __restrict__ out_d,
                                                           const uint32_t* __restrict__ perm,
                                                           uint32_t* __restrict__ err, unsigned long long* stats)
{
    __shared__ uint32_t stk[SSZ * BS];
    __shared__ EdgeLds elds[DIM == 3 ? BS / 64 : 1];
    const uint32_t slot = xcd_remap(blockIdx.x, gridDim.x) * BS + threadIdx.x;
    Counts cnt;
    if (t.n_dev)
        n = min(n, *t.n_dev);
    const uint32_t qi = slot < n ? (perm ? perm[slot] : slot) : nq;
    if (qi >= nq) {
        if (STATS)
            flush_counts(cnt, stats);
        return;
    }
    float cap = MODE != 0 ? seed[qi] : F_INF;
    if (!(cap >= 0.0f))
        cap = F_INF;
    float best;
    uint32_t best_e;
    bool ovf = false;
    const v3 p = load_point<DIM>(q, qi);
    sil_query<BS, SSZ, STATS, DIM, MODE != 2, MODE != 2>(t, p, flip != 0, cap, stk + threadIdx.x,
                                                         DIM == 3 ? &elds[threadIdx.x / 64] : nullptr, best,
                                                         best_e, cnt, ovf);
    if (ovf && err)
        atomicOr(err, 1u);
    if (out_e)
        out_e[qi] = best_e;
    out_d[qi] = best;
    if (STATS)
        flush_counts(cnt, stats);
}

// Seeded search with re-queued unsettled queries.  A wave's time is that of
// its slowest lane, so a query not settled within its seed radius, searched
// again in place, holds 63 settled lanes idle.  Here the launch is
// persistent: each wave takes 64-query chunks of the visiting order (each
// XCD a contiguous range of chunks first, then the other XCDs' ranges) and
// searches them within their seeds (a hard cap); a query not settled there is
// appended to a queue.  A wave that finds no chunk left takes up to 64 queued
// queries at a time and searches them with no cap, until it finds the queue
// empty.  Every appended entry is taken: its appender itself goes on to drain
// the queue after its last append.  A taken slot may still be being written
// by its appender, which has reserved it and is running, so the wait for it
// is short (and bounded).  Each XCD appends to its own queue and drains it
// first: its waves work through a contiguous stretch of the visiting order,
// so a wave of its queued queries stays in one region of the scene, whose
// nodes its L2 holds (one queue for all mixed the regions of all eight).
// ctr: [0, 8) next chunk of each XCD's range, [8 + 2x] and [9 + 2x] head and
// tail of XCD x's queue (RQ_CTR_WORDS words in all); queue: 8 queues of n
// entries, RQ_EMPTY at launch.  Results equal the unseeded search's.
constexpr uint32_t RQ_EMPTY = 0xFFFFFFFFu;
constexpr uint32_t RQ_SPIN = 1u << 20;
constexpr uint32_t RQ_CTR_WORDS = 24;

__global__ __launch_bounds__(256) void k_requeue_init(uint32_t* __restrict__ ctr, uint32_t* __restrict__ queue,
                                                      uint32_t n)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < RQ_CTR_WORDS)
        ctr[i] = 0u;
    for (uint32_t k = i; k < n; k += gridDim.x * 256)
        queue[k] = RQ_EMPTY;
}

template <int SSZ, bool STATS, int DIM>
__global__ __launch_bounds__(64, STATS ? 5 : 6) void k_sil_requeue(TreeView t, const float* __restrict__ q,
                                                                 uint32_t n, int flip, const float* __restrict__ seed,
                                                                 uint32_t* __restrict__ out_e,
                                                                 float* __restrict__ out_d,
                                                                 const uint32_t* __restrict__ perm, uint32_t* ctr,
                                                                 uint32_t* queue, uint32_t* __restrict__ err,
                                                                 unsigned long long* stats)
{
    __shared__ uint32_t stk[SSZ * 64];
    __shared__ EdgeLds elds[1];
    const uint32_t lane = threadIdx.x;
    const uint32_t nchunks = (n + 63) / 64;
    const uint32_t x0 = blockIdx.x % 8u; // blocks are dispatched round-robin over the 8 XCDs
    uint32_t xi = 0;                     // ranges exhausted so far, own range first (wave-uniform)
    uint32_t di = 0;                     // queues found empty while draining, own XCD's first
    bool draining = false, ovf = false;
    Counts cnt;
    for (;;) {
        uint32_t qi = INVALID;
        float cap = F_INF;
        if (!draining) {
            uint32_t c = INVALID;
            while (xi < 8u) {
                const uint32_t xx = (x0 + xi) & 7u;
                const uint32_t lo = (uint32_t)((uint64_t)nchunks * xx / 8u);
                const uint32_t hi = (uint32_t)((uint64_t)nchunks * (xx + 1u) / 8u);
                uint32_t k = 0;
                if (lane == 0)
                    k = atomicAdd(ctr + xx, 1u);
                k = uniform(k);
                if (k < hi - lo) {
                    c = lo + k;
                    break;
                }
                ++xi;
            }
            if (c == INVALID) {
                draining = true;
                continue;
            }
            const uint32_t slot = c * 64u + lane;
            if (slot < n) {
                qi = perm ? perm[slot] : slot;
                cap = seed[qi];
                if (!(cap >= 0.0f))
                    cap = F_INF;
            }
        } else {
            // take up to 64 queued queries of queue dq (this XCD's first):
            // [base, base + k) below its tail
            const uint32_t dq = (x0 + di) & 7u;
            uint32_t* head = ctr + 8 + 2 * dq;
            uint32_t base = 0, k = 0, empty = 0;
            if (lane == 0) {
                uint32_t h = __hip_atomic_load(head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                for (uint32_t tries = 0; tries < 64u; ++tries) {
                    const uint32_t tl = __hip_atomic_load(head + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (h >= tl) {
                        empty = 1u;
                        break;
                    }
                    const uint32_t want = min(64u, tl - h);
                    const uint32_t old = atomicCAS(head, h, h + want); // a failure means another wave took some
                    if (old == h) {
                        base = h;
                        k = want;
                        break;
                    }
                    h = old;
                }
            }
            if (uniform(empty)) {
                if (++di >= 8u)
                    break;
                continue;
            }
            base = uniform(base);
            k = uniform(k);
            if (k == 0u)
                continue; // contended: try again
            if (lane < k) {
                uint32_t v = RQ_EMPTY;
                for (uint32_t s = 0; s < RQ_SPIN && v == RQ_EMPTY; ++s) {
                    v = __hip_atomic_load(queue + (size_t)dq * n + base + lane, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
                    if (v == RQ_EMPTY)
                        __builtin_amdgcn_s_sleep(2);
                }
                if (v < n)
                    qi = v;
                else
                    ovf = true; // not expected: the slot's writer had reserved it
            }
        }
        float best = F_INF;
        uint32_t best_e = INVALID;
        if (qi < n)
            sil_query<64, SSZ, STATS, DIM, false, true>(t, load_point<DIM>(q, qi), flip != 0, cap, stk + lane,
                                                        DIM == 3 ? elds : nullptr, best, best_e, cnt, ovf);
        const bool unsettled = qi < n && cap < F_INF && !(best_e != INVALID && best <= cap);
        if (qi < n && !unsettled) {
            if (out_e)
                out_e[qi] = best_e;
            out_d[qi] = best;
        }
        const uint64_t um = __ballot(unsettled);
        if (um) {
            uint32_t b = 0;
            if (lane == 0)
                b = atomicAdd(ctr + 9 + 2 * x0, (uint32_t)__popcll(um)); // this XCD's queue
            b = uniform(b);
            // rank among the unsettled lanes below this one
            const uint32_t r = __builtin_amdgcn_mbcnt_hi((uint32_t)(um >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)um, 0u));
            if (unsettled)
                __hip_atomic_store(queue + (size_t)x0 * n + b + r, qi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (ovf && err)
        atomicOr(err, 1u);
    if (STATS)
        flush_counts(cnt, stats);
}

// Plain search on a persistent launch: each wave takes 64-query chunks of the
// visiting order, its own XCD's contiguous range of chunks first, then the
// other XCDs' ranges, until none is left.  A wave's time is that of its
// slowest lane, and waves of one launch differ widely; taking chunks as waves
// free up balances that over the whole launch, and the per-XCD ranges keep
// the queries an XCD searches close together in space (its L2 holds their
// nodes).  On the 1M-triangle torus, 4M queries: 75.3 -> 70.7 ms against one
// 64-query block per chunk.  Handing the few lanes left in a wave to fresh
// waves (suspend, resume from the trail) was measured slower: 81-90 ms with
// the suspended queries kept in visiting order, ~140 ms in suspension order.
// CAPPED: the search within the radius seed[qi] only (as k_closest_silhouette's
// MODE 2; walk on stars), over the first min(n, *t.n_dev) queries when the
// count is on the device.  ctr: [0, 8) the chunk counters of the XCD ranges
// (zero at launch).
template <int SSZ, bool STATS, int DIM, bool CAPPED>
__global__ __launch_bounds__(64, STATS || CAPPED ? 5 : 6) void k_sil_persist(TreeView t, const float* __restrict__ q,
                                                                 uint32_t n, int flip, const float* __restrict__ seed,
                                                                 uint32_t* __restrict__ out_e,
                                                                 float* __restrict__ out_d,
                                                                 const uint32_t* __restrict__ perm, uint32_t* ctr,
                                                                 uint32_t* __restrict__ err,
                                                                 unsigned long long* stats)
{
    __shared__ uint32_t stk[SSZ * 64];
    __shared__ EdgeLds elds[1];
    const uint32_t lane = threadIdx.x;
    if (CAPPED && t.n_dev)
        n = min(n, *t.n_dev);
    const uint32_t nchunks = (n + 63) / 64;
    const uint32_t x0 = blockIdx.x % 8u; // blocks are dispatched round-robin over the 8 XCDs
    uint32_t xi = 0;                     // ranges exhausted so far, own range first (wave-uniform)
    bool ovf = false;
    Counts cnt;
    for (;;) {
        const uint32_t c = take_chunk(ctr, nchunks, x0, xi);
        if (c == INVALID)
            break;
        const uint32_t slot = c * 64u + lane;
        const uint32_t qi = slot < n ? (perm ? perm[slot] : slot) : INVALID;
        if (qi < n) {
            float best;
            uint32_t best_e;
            float cap = F_INF;
            if (CAPPED) {
                cap = seed[qi];
                if (!(cap >= 0.0f))
                    cap = F_INF;
            }
            // hard-capped searches are short: leaves are tested at once (no parking)
            sil_query<64, SSZ, STATS, DIM, false, !CAPPED>(t, load_point<DIM>(q, qi), flip != 0, cap, stk + lane,
                                                           DIM == 3 ? elds : nullptr, best, best_e, cnt, ovf);
            if (out_e)
                out_e[qi] = best_e;
            out_d[qi] = best;
        }
    }
    if (ovf && err)
        atomicOr(err, 1u);
    if (STATS)
        flush_counts(cnt, stats);
}

} // namespace

template <int BS, int DIM, int SSZ>
static void launch_sil_cfg(const TreeView& t, const float* q, uint32_t n, int flip, const float* seed, bool capped,
                           uint32_t* sil, float* dist, const uint32_t* perm, unsigned long long* stats,
                           uint32_t* err, hipStream_t st)
{
    const dim3 g(nblocks(n, BS)), b(BS);
#define SNCH_SIL(S_, M_, ...) \
    hipLaunchKernelGGL((k_closest_silhouette<BS, S_, DIM, M_, SSZ>), g, b, 0, st, __VA_ARGS__)
    if (!seed) {
        if (stats)
            SNCH_SIL(true, 0, t, q, n, n, flip, seed, sil, dist, perm, err, stats);
        else
            SNCH_SIL(false, 0, t, q, n, n, flip, seed, sil, dist, perm, err, stats);
    } else if (capped) {
        if (stats)
            SNCH_SIL(true, 2, t, q, n, n, flip, seed, sil, dist, perm, err, stats);
        else
            SNCH_SIL(false, 2, t, q, n, n, flip, seed, sil, dist, perm, err, stats);
    } else {
        if (stats)
            SNCH_SIL(true, 1, t, q, n, n, flip, seed, sil, dist, perm, err, stats);
        else
            SNCH_SIL(false, 1, t, q, n, n, flip, seed, sil, dist, perm, err, stats);
    }
#undef SNCH_SIL
}

template <int BS, int DIM>
static void launch_sil_bs(const TreeView& t, const float* q, uint32_t n, int flip, const float* seed, bool capped,
                          uint32_t* sil, float* dist, uint32_t depth, const uint32_t* perm,
                          unsigned long long* stats, uint32_t* err, hipStream_t st)
{
    if (DIM == 2 || depth == 16) // scene<2> uses the default depth only
        launch_sil_cfg<BS, DIM, 16>(t, q, n, flip, seed, capped, sil, dist, perm, stats, err, st);
    else if (depth == 8)
        launch_sil_cfg<BS, DIM, 8>(t, q, n, flip, seed, capped, sil, dist, perm, stats, err, st);
    else if (depth == 24)
        launch_sil_cfg<BS, DIM, 24>(t, q, n, flip, seed, capped, sil, dist, perm, stats, err, st);
    else
        launch_sil_cfg<BS, DIM, 32>(t, q, n, flip, seed, capped, sil, dist, perm, stats, err, st);
}

hipError_t launch_closest_silhouette(const TreeView& t, int dim, const float* q, uint32_t n, int flip,
                                     const float* seed, bool capped, uint32_t* sil, float* dist, uint32_t block,
                                     uint32_t depth, const uint32_t* perm, uint64_t* stats, hipStream_t st,
                                     uint32_t* err)
{
    if (n == 0)
        return hipSuccess;
    auto* sp = reinterpret_cast<unsigned long long*>(stats);
    if (!err)
        err = traversal_error_word();
    SNCH_DISPATCH_DIM(dim, {
        switch (block) {
        case 128: launch_sil_bs<128, DIM>(t, q, n, flip, seed, capped, sil, dist, depth, perm, sp, err, st); break;
        case 256: launch_sil_bs<256, DIM>(t, q, n, flip, seed, capped, sil, dist, depth, perm, sp, err, st); break;
        case 512: launch_sil_bs<512, DIM>(t, q, n, flip, seed, capped, sil, dist, depth, perm, sp, err, st); break;
        default: launch_sil_bs<64, DIM>(t, q, n, flip, seed, capped, sil, dist, depth, perm, sp, err, st); break;
        }
    });
    return hipGetLastError();
}

template <int DIM, bool STATS>
static void launch_sil_requeue_cfg(const TreeView& t, const float* q, uint32_t n, int flip, const float* seed,
                                   uint32_t* sil, float* dist, const uint32_t* perm, unsigned long long* stats,
                                   uint32_t* ctr, uint32_t* queue, uint32_t n_cu, uint32_t* err, hipStream_t st)
{
    // as many one-wave blocks as are resident at once; more would only wait
    static int per_cu = 0;
    if (per_cu == 0 &&
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_sil_requeue<16, STATS, DIM>, 64, 0) != hipSuccess)
        per_cu = 1;
    const uint32_t grid = std::max(1u, std::min(n_cu * (uint32_t)std::max(per_cu, 1), (n + 63) / 64));
    hipLaunchKernelGGL((k_sil_requeue<16, STATS, DIM>), dim3(grid), dim3(64), 0, st, t, q, n, flip, seed, sil, dist,
                       perm, ctr, queue, err, stats);
}

hipError_t launch_closest_silhouette_requeue(const TreeView& t, int dim, const float* q, uint32_t n, int flip,
                                             const float* seed, uint32_t* sil, float* dist, const uint32_t* perm,
                                             uint64_t* stats, uint32_t* ctr, uint32_t* queue, uint32_t n_cu,
                                             hipStream_t st, uint32_t* err)
{
    if (n == 0)
        return hipSuccess;
    auto* sp = reinterpret_cast<unsigned long long*>(stats);
    if (!err)
        err = traversal_error_word();
    hipLaunchKernelGGL(k_requeue_init, dim3(std::min(nblocks(n, 256), 1024u)), dim3(256), 0, st, ctr, queue, 8 * n);
    SNCH_DISPATCH_DIM(dim, {
        if (sp)
            launch_sil_requeue_cfg<DIM, true>(t, q, n, flip, seed, sil, dist, perm, sp, ctr, queue, n_cu, err, st);
        else
            launch_sil_requeue_cfg<DIM, false>(t, q, n, flip, seed, sil, dist, perm, sp, ctr, queue, n_cu, err, st);
    });
    return hipGetLastError();
}

template <int DIM, bool STATS, bool CAPPED>
static void launch_sil_persist_cfg(const TreeView& t, const float* q, uint32_t n, int flip, const float* seed,
                                   uint32_t* sil, float* dist, const uint32_t* perm, unsigned long long* stats,
                                   uint32_t* ctr, uint32_t n_cu, uint32_t* err, hipStream_t st)
{
    // as many one-wave blocks as are resident at once; more would only wait
    static int per_cu = 0;
    if (per_cu == 0 && hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_sil_persist<16, STATS, DIM, CAPPED>,
                                                                     64, 0) != hipSuccess)
        per_cu = 1;
    const uint32_t grid = std::max(1u, std::min(n_cu * (uint32_t)std::max(per_cu, 1), (n + 63) / 64));
    hipLaunchKernelGGL((k_sil_persist<16, STATS, DIM, CAPPED>), dim3(grid), dim3(64), 0, st, t, q, n, flip, seed, sil,
                       dist, perm, ctr, err, stats);
}

hipError_t launch_closest_silhouette_persist(const TreeView& t, int dim, const float* q, uint32_t n, int flip,
                                             const float* seed, uint32_t* sil, float* dist, const uint32_t* perm,
                                             uint64_t* stats, uint32_t* ctr, uint32_t n_cu, hipStream_t st,
                                             uint32_t* err)
{
    if (n == 0)
        return hipSuccess;
    auto* sp = reinterpret_cast<unsigned long long*>(stats);
    if (!err)
        err = traversal_error_word();
    hipLaunchKernelGGL(k_requeue_init, dim3(1), dim3(256), 0, st, ctr, nullptr, 0u); // the chunk counters
    SNCH_DISPATCH_DIM(dim, {
        if (sp && seed)
            launch_sil_persist_cfg<DIM, true, true>(t, q, n, flip, seed, sil, dist, perm, sp, ctr, n_cu, err, st);
        else if (sp)
            launch_sil_persist_cfg<DIM, true, false>(t, q, n, flip, seed, sil, dist, perm, sp, ctr, n_cu, err, st);
        else if (seed)
            launch_sil_persist_cfg<DIM, false, true>(t, q, n, flip, seed, sil, dist, perm, sp, ctr, n_cu, err, st);
        else
            launch_sil_persist_cfg<DIM, false, false>(t, q, n, flip, seed, sil, dist, perm, sp, ctr, n_cu, err, st);
    });
    return hipGetLastError();
}

} // namespace snch
