// Batched queries: one persistent launch over the queries of every mesh of a
// batch.
#include <vector>

#include "wave_search.hpp"

namespace snch {

namespace {

// ------------------------------------------------------------ batches
// One persistent launch over the queries of every mesh of a batch, given as
// one concatenated query array; the queries of each mesh are cut into chunks of `qpw` (a multiple of 64), and chunks are handed out in
// schedule order (meshes with deeper trees first) through one atomic counter.
// Queries of mesh m are [qoff[m], qoff[m + 1]).
// Each wave takes a chunk, answers it 64 queries at a time against that
// mesh's tree, and takes the next, until the counter passes the last chunk:
// every wave reaches that exit.
struct BatchTable {
    const TreeView* views;  // per mesh
    const uint32_t* qoff;   // per mesh, n_meshes + 1 entries
    const uint32_t* sched;  // schedule entry -> mesh
    const uint32_t* cstart; // schedule entry -> first chunk (n_sched + 1 entries)
    const uint32_t* perm;   // optional visiting order of all queries (null: input order)
    uint32_t* counter;
    uint32_t n_sched, total_chunks, qpw;
};

// SEEDED (closest silhouette): seed[qi] is the query's pruning radius (a
// learned bound); the search within it is exact, a query not settled there
// searches again from the root, so results equal the unseeded ones
template <int BS, int SSZ, int KIND, bool SEEDED>
__global__ __launch_bounds__(BS, 5) void k_batch(BatchTable bt, const float* __restrict__ q, int flip,
                                              const float* __restrict__ seed, uint32_t* __restrict__ out_idx,
                                              float* __restrict__ out_dist, uint32_t* __restrict__ err)
{
    // closest point: a pool per wave; closest silhouette: a stack per lane
    constexpr uint32_t POOL_WORDS = 2 * 32 * SSZ + WaveLds::FIXED;
    __shared__ __align__(16) uint32_t stk[KIND == 0 ? POOL_WORDS * (BS / 64) : SSZ * BS];
    __shared__ EdgeLds elds[KIND == 0 ? 1 : BS / 64];
    const uint32_t lane = threadIdx.x & 63;
    bool ovf = false;
    Counts cnt;
    for (uint32_t guard = 0; guard < bt.total_chunks + 1; ++guard) {
        uint32_t c = 0;
        if (lane == 0)
            c = atomicAdd(bt.counter, 1u);
        c = __shfl(c, 0, 64);
        if (c >= bt.total_chunks)
            break;
        uint32_t lo = 0, hi = bt.n_sched; // last entry with cstart <= c
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (bt.cstart[mid] <= c)
                lo = mid;
            else
                hi = mid;
        }
        const uint32_t m = bt.sched[lo];
        const TreeView tv = bt.views[m];
        const uint32_t q0 = bt.qoff[m] + (c - bt.cstart[lo]) * bt.qpw;
        const uint32_t q1 = min(q0 + bt.qpw, bt.qoff[m + 1]);
        for (uint32_t base = q0; base < q1; base += 64) {
            const uint32_t slot = base + lane;
            const bool valid = slot < q1;
            if (KIND != 0 && !valid)
                continue;
            const uint32_t qi = valid ? (bt.perm ? bt.perm[slot] : slot) : 0u;
            const v3 p = valid ? load_point<3>(q, qi) : mk(0.0f, 0.0f, 0.0f);
            float best = F_INF;
            uint32_t bi = INVALID;
            if (KIND == 0) {
                WaveLds W(stk + (threadIdx.x / 64) * POOL_WORDS, 32 * SSZ);
                if (valid)
                    W.start(lane, p);
                cp_wave<false, 3>(tv, min(64u, q1 - base), W, cnt, ovf);
                if (!valid)
                    continue;
                unpack_best(W.best[lane], best, bi);
                best = dm::sqrt_(best);
            } else {
                float cap = SEEDED ? seed[qi] : F_INF;
                if (!(cap >= 0.0f))
                    cap = F_INF;
                sil_query<BS, SSZ, false, 3, SEEDED, true>(tv, p, flip != 0, cap, stk + threadIdx.x,
                                                           &elds[KIND == 0 ? 0 : threadIdx.x / 64], best, bi, cnt,
                                                           ovf);
            }
            if (out_idx)
                out_idx[qi] = bi;
            out_dist[qi] = best;
        }
    }
    if (ovf && err)
        atomicOr(err, 1u);
}

// Morton code of each query in its own mesh's root box (batches)
__global__ __launch_bounds__(256) void k_batch_codes(const TreeView* __restrict__ views,
                                                     const uint32_t* __restrict__ qmesh, const float* __restrict__ q,
                                                     uint32_t n, uint32_t* __restrict__ codes,
                                                     uint32_t* __restrict__ idx)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    const TreeView& t = views[qmesh[i]];
    const float4 lo = t.nbox[0], hi = t.nbox[1];
    const v3 p = load_point<3>(q, i);
    codes[i] = morton3(mk((p.x - lo.x) / (hi.x - lo.x), (p.y - lo.y) / (hi.y - lo.y), (p.z - lo.z) / (hi.z - lo.z)));
    idx[i] = i;
}

__global__ void k_zero_counter(uint32_t* c) { *c = 0u; }

// mesh of each query of a batch (last m with qoff[m] <= i)
__global__ __launch_bounds__(256) void k_query_mesh(const uint32_t* __restrict__ qoff, uint32_t M, uint32_t n,
                                                    uint32_t* __restrict__ qmesh)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    uint32_t lo = 0, hi = M;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (qoff[mid] <= i)
            lo = mid;
        else
            hi = mid;
    }
    qmesh[i] = lo;
}

} // namespace

template <int BS, int SSZ, int KIND, bool SEEDED>
static hipError_t launch_batch_cfg(const BatchTable& bt, const float* q, int flip, const float* seed,
                                   uint32_t* out_idx, float* out_dist, uint32_t n_cu, hipStream_t st)
{
    int per_cu = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_batch<BS, SSZ, KIND, SEEDED>, BS, 0);
    if (e != hipSuccess)
        return e;
    const uint32_t waves = n_cu * (uint32_t)std::max(per_cu, 1) * (BS / 64);
    // no more waves than chunks
    const uint32_t grid = std::max(1u, std::min(n_cu * (uint32_t)std::max(per_cu, 1),
                                                (std::min(waves, bt.total_chunks) + BS / 64 - 1) / (BS / 64)));
    hipLaunchKernelGGL((k_batch<BS, SSZ, KIND, SEEDED>), dim3(grid), dim3(BS), 0, st, bt, q, flip, seed, out_idx,
                       out_dist, traversal_error_word());
    return hipGetLastError();
}

template <int BS, int KIND, bool SEEDED>
static hipError_t launch_batch_bs(const BatchTable& bt, uint32_t ssz, const float* q, int flip, const float* seed,
                                  uint32_t* out_idx, float* out_dist, uint32_t n_cu, hipStream_t st)
{
    switch (ssz) {
    case 8: return launch_batch_cfg<BS, 8, KIND, SEEDED>(bt, q, flip, seed, out_idx, out_dist, n_cu, st);
    case 24: return launch_batch_cfg<BS, 24, KIND, SEEDED>(bt, q, flip, seed, out_idx, out_dist, n_cu, st);
    case 32: return launch_batch_cfg<BS, 32, KIND, SEEDED>(bt, q, flip, seed, out_idx, out_dist, n_cu, st);
    default: return launch_batch_cfg<BS, 16, KIND, SEEDED>(bt, q, flip, seed, out_idx, out_dist, n_cu, st);
    }
}

template <int KIND, bool SEEDED>
static hipError_t launch_batch_kind(const BatchTable& bt, uint32_t bs, uint32_t ssz, const float* q, int flip,
                                    const float* seed, uint32_t* out_idx, float* out_dist, uint32_t n_cu,
                                    hipStream_t st)
{
    switch (bs) {
    case 64: return launch_batch_bs<64, KIND, SEEDED>(bt, ssz, q, flip, seed, out_idx, out_dist, n_cu, st);
    case 128: return launch_batch_bs<128, KIND, SEEDED>(bt, ssz, q, flip, seed, out_idx, out_dist, n_cu, st);
    case 512: return launch_batch_bs<512, KIND, SEEDED>(bt, ssz, q, flip, seed, out_idx, out_dist, n_cu, st);
    default: return launch_batch_bs<256, KIND, SEEDED>(bt, ssz, q, flip, seed, out_idx, out_dist, n_cu, st);
    }
}

hipError_t launch_batch(const snch_scene* s, int kind, const float* q, const uint32_t* q_off_host, int flip,
                        uint32_t* out_idx, float* out_dist, const BatchConfig& cfg, hipStream_t st,
                        const float* seed)
{
    const uint32_t M = s->n_meshes;
    BatchState& b = s->batch;
    const uint32_t n = q_off_host[M];
    if (n == 0)
        return hipSuccess;
    const uint32_t qpw = cfg.queries_per_wave;
    // schedule: meshes with more leaves (deeper trees, costlier queries) first
    std::vector<uint32_t> order(M);
    for (uint32_t m = 0; m < M; ++m)
        order[m] = m;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t c) {
        return s->mesh_off[a + 1] - s->mesh_off[a] > s->mesh_off[c + 1] - s->mesh_off[c];
    });
    // host table: qoff (M + 1) | sched (M) | cstart (M + 1)
    b.host_tab.assign(3 * (size_t)M + 2, 0);
    uint32_t* h_qoff = b.host_tab.data();
    uint32_t* h_sched = h_qoff + M + 1;
    uint32_t* h_cstart = h_sched + M;
    for (uint32_t m = 0; m <= M; ++m)
        h_qoff[m] = q_off_host[m];
    uint32_t ns = 0, total = 0;
    for (uint32_t k = 0; k < M; ++k) {
        const uint32_t m = order[k], cnt = q_off_host[m + 1] - q_off_host[m];
        if (cnt == 0)
            continue;
        h_sched[ns] = m;
        h_cstart[ns] = total;
        total += (cnt + qpw - 1) / qpw;
        ++ns;
    }
    h_cstart[ns] = total;
    hipError_t e;
    if ((e = b.tab.ensure(sizeof(uint32_t) * b.host_tab.size())) != hipSuccess ||
        (e = b.counter.ensure(64)) != hipSuccess)
        return e;
    uint32_t* d_tab = b.tab.as<uint32_t>();
    if ((e = hipMemcpyAsync(d_tab, b.host_tab.data(), sizeof(uint32_t) * b.host_tab.size(), hipMemcpyHostToDevice,
                            st)) != hipSuccess)
        return e;
    BatchTable bt;
    bt.views = b.views.as<TreeView>();
    bt.qoff = d_tab;
    bt.sched = d_tab + M + 1;
    bt.cstart = d_tab + 2 * M + 1;
    bt.perm = nullptr;
    bt.counter = b.counter.as<uint32_t>();
    bt.n_sched = ns;
    bt.total_chunks = total;
    bt.qpw = qpw;
    if (cfg.coherent) {
        QueryScratch& w = b.order;
        if ((e = w.codes.ensure(sizeof(uint32_t) * n)) != hipSuccess ||
            (e = w.idx.ensure(sizeof(uint32_t) * n)) != hipSuccess ||
            (e = w.codes_alt.ensure(sizeof(uint32_t) * n)) != hipSuccess ||
            (e = w.idx_alt.ensure(sizeof(uint32_t) * n)) != hipSuccess ||
            (e = b.qmesh.ensure(sizeof(uint32_t) * n)) != hipSuccess)
            return e;
        hipLaunchKernelGGL(k_query_mesh, dim3(nblocks(n, 256)), dim3(256), 0, st, d_tab, M, n,
                           b.qmesh.as<uint32_t>());
        hipLaunchKernelGGL(k_batch_codes, dim3(nblocks(n, 256)), dim3(256), 0, st, bt.views, b.qmesh.as<uint32_t>(),
                           q, n, w.codes.as<uint32_t>(), w.idx.as<uint32_t>());
        int mesh_bits = 0;
        while (mesh_bits < 32 && ((M - 1) >> mesh_bits) != 0)
            ++mesh_bits;
        bool in_alt = false;
        if ((e = radix_sort_pairs(w.codes.as<uint32_t>(), w.idx.as<uint32_t>(), w.codes_alt.as<uint32_t>(),
                                  w.idx_alt.as<uint32_t>(), n, 30, w.hist, st, &in_alt,
                                  M > 1 ? b.qmesh.as<uint32_t>() : nullptr, M > 1 ? mesh_bits : 0)) != hipSuccess)
            return e;
        bt.perm = in_alt ? w.idx_alt.as<uint32_t>() : w.idx.as<uint32_t>();
    }
    hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(1), 0, st, bt.counter);
    const uint32_t n_cu = s->ctx && s->ctx->n_cu > 0 ? (uint32_t)s->ctx->n_cu : 256u;
    if (kind == 0)
        return launch_batch_kind<0, false>(bt, cfg.block_size, cfg.stack_depth, q, flip, nullptr, out_idx, out_dist,
                                           n_cu, st);
    if (seed)
        return launch_batch_kind<1, true>(bt, cfg.block_size, cfg.stack_depth, q, flip, seed, out_idx, out_dist, n_cu,
                                          st);
    return launch_batch_kind<1, false>(bt, cfg.block_size, cfg.stack_depth, q, flip, nullptr, out_idx, out_dist, n_cu,
                                       st);
}

} // namespace snch
