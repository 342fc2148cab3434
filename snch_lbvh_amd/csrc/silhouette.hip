// Closest-silhouette kernel (query.cuh:325-423) and its dispatch.
#include "wave_search.hpp"

namespace snch {

namespace {

// MODE 0: plain search.  MODE 1: seed[qi] is a pruning hint.  MODE 2: a hard
// cap (sil_wave).  A large launch is persistent: as many waves as are
// resident take chunks of 64 queries as they get free, each XCD from its own
// range of chunks first (its L2 holds that region's nodes).
template <bool STATS, int DIM, int MODE>
__global__ __launch_bounds__(512, STATS ? 4 : 6) void k_silhouette(TreeView t, const float* __restrict__ q, uint32_t n,
                                                                   uint32_t deal, uint32_t cap_items, int flip,
                                                                   const float* __restrict__ seed,
                                                                   uint32_t* __restrict__ out_e,
                                                                   float* __restrict__ out_d,
                                                                   const uint32_t* __restrict__ perm, uint32_t* ctr,
                                                                   uint32_t* __restrict__ err,
                                                                   unsigned long long* stats)
{
    extern __shared__ __align__(16) uint32_t smem[];
    const uint32_t lane = threadIdx.x & 63;
    WaveLds W(smem + (threadIdx.x >> 6) * wave_lds_words(cap_items, MODE == 2), cap_items);
    if (t.n_dev)
        n = min(n, *t.n_dev);
    if (deal == 0u)
        deal = deal_queries(n, gridDim.x * (blockDim.x >> 6), SIL_RUNS);
    bool ovf = false;
    Counts cnt;
    for_chunks(n, deal, ctr, [&](uint32_t slot, bool valid) {
        const uint32_t qi = valid ? (perm ? min(perm[slot], n - 1) : slot) : 0u;
        if (valid)
            W.start(lane, load_point<DIM>(q, qi));
        const float cap = MODE != 0 && valid ? seed[qi] : F_INF;
        sil_wave<STATS, DIM, MODE>(t, __ballot(valid), flip != 0, cap, W, cnt, ovf);
        if (valid) {
            float best;
            uint32_t best_e;
            unpack_best(W.best[lane], best, best_e);
            if (out_e)
                out_e[qi] = best_e;
            out_d[qi] = best;
        }
    });
    if (ovf && err)
        atomicOr(err, 1u);
    if (STATS)
        flush_counts(cnt, stats);
}

__global__ void k_clear_chunks(uint32_t* __restrict__ ctr)
{
    if (threadIdx.x < CHUNK_CTR_WORDS)
        ctr[threadIdx.x] = 0u;
}

} // namespace

bool silhouette_persists(uint32_t n, uint32_t block, uint32_t depth, bool hard, uint32_t n_cu)
{
    return search_grid(n, block, wave_lds_words(pool_cap(depth), hard), n_cu, 6, true, false, SIL_RUNS).persist;
}

hipError_t clear_chunks(uint32_t* ctr, hipStream_t st)
{
    hipLaunchKernelGGL(k_clear_chunks, dim3(1), dim3(64), 0, st, ctr);
    return hipGetLastError();
}

hipError_t launch_closest_silhouette(const TreeView& t, int dim, const float* q, uint32_t n, int flip,
                                     const float* seed, bool capped, uint32_t* sil, float* dist, uint32_t block,
                                     uint32_t depth, const uint32_t* perm, uint64_t* stats, uint32_t* ctr,
                                     uint32_t n_cu, hipStream_t st, uint32_t* err)
{
    if (n == 0)
        return hipSuccess;
    auto* sp = reinterpret_cast<unsigned long long*>(stats);
    if (!err)
        err = traversal_error_word();
    const bool hard = seed && capped;
    const SearchGrid g = search_grid(n, block, wave_lds_words(pool_cap(depth), hard), n_cu, 6, ctr != nullptr,
                                      t.n_dev != nullptr, SIL_RUNS);
    uint32_t* c = g.persist ? ctr : nullptr;
#define SNCH_SIL(S_, M_)                                                                                             \
    hipLaunchKernelGGL((k_silhouette<S_, DIM, M_>), g.grid, g.block, g.lds, st, t, q, n, g.deal, pool_cap(depth), flip, \
                       seed, sil, dist, perm, c, err, sp)
    SNCH_DISPATCH_DIM(dim, {
        if (!seed) {
            if (sp)
                SNCH_SIL(true, 0);
            else
                SNCH_SIL(false, 0);
        } else if (capped) {
            if (sp)
                SNCH_SIL(true, 2);
            else
                SNCH_SIL(false, 2);
        } else {
            if (sp)
                SNCH_SIL(true, 1);
            else
                SNCH_SIL(false, 1);
        }
    });
#undef SNCH_SIL
    return hipGetLastError();
}

} // namespace snch
