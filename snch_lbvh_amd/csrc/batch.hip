// Batched queries: one persistent launch over the queries of every mesh of a
// batch.
#include <vector>

#include "wave_search.hpp"

namespace snch {

namespace {

// ------------------------------------------------------------ batches
// One persistent launch over the queries of every mesh of a batch, given as
// one concatenated query array, those of mesh m being [qoff[m], qoff[m + 1]).
// The queries of a mesh are dealt to steps of up to 64 (deal_queries, by the
// size of the whole batch), and chunks of `spc` steps are handed out in
// schedule order (meshes with deeper trees first) through one atomic counter.
// Each wave takes a chunk, answers it step by step against that mesh's tree,
// and takes the next, until the counter passes the last chunk: every wave
// reaches that exit.
// Steps of 64 neighbours leave the few that hold a mesh's costliest queries to
// run on alone, and most waves of a small batch idle: 24 meshes of up to 200,000
// triangles and 1,379,128 silhouette queries 36.1 ms so, 11.0 dealt; 10 meshes,
// 201,121 queries 13.1 and 3.4 (closest points 3.1 and 2.1, 1.23 and 0.59).
struct BatchTable {
    const TreeView* views;  // per mesh
    const uint32_t* qoff;   // per mesh, n_meshes + 1 entries
    const uint32_t* sched;  // schedule entry -> mesh
    const uint32_t* cstart; // schedule entry -> first chunk (n_sched + 1 entries)
    const uint32_t* perm;   // optional visiting order of all queries (null: input order)
    uint32_t* counter;
    uint32_t n_sched, total_chunks, deal, spc;
};

// KIND 0: closest point.  1: closest silhouette.  2: closest silhouette with
// a per-query pruning hint seed[qi]; results equal the unseeded ones
template <int KIND>
__global__ __launch_bounds__(512, 6) void k_batch(BatchTable bt, uint32_t cap, const float* __restrict__ q, int flip,
                                                  const float* __restrict__ seed, uint32_t* __restrict__ out_idx,
                                                  float* __restrict__ out_dist, uint32_t* __restrict__ err)
{
    extern __shared__ __align__(16) uint32_t smem[];
    const uint32_t lane = threadIdx.x & 63;
    WaveLds W(smem + (threadIdx.x >> 6) * wave_lds_words(cap), cap);
    bool ovf = false;
    Counts cnt;
    for (uint32_t guard = 0; guard < bt.total_chunks + 1; ++guard) {
        uint32_t c = 0;
        if (lane == 0)
            c = atomicAdd(bt.counter, 1u);
        c = uniform(c);
        if (c >= bt.total_chunks)
            break;
        uint32_t lo = 0, hi = bt.n_sched; // last entry with cstart <= c
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (uniform(bt.cstart[mid]) <= c)
                lo = mid;
            else
                hi = mid;
        }
        const uint32_t m = uniform(bt.sched[lo]);
        const TreeView tv = bt.views[m];
        const uint32_t q0 = uniform(bt.qoff[m]), nq = uniform(bt.qoff[m + 1]) - q0;
        const uint32_t per = bt.deal & 255u, run = bt.deal >> 8, nsteps = (nq + per - 1u) / per;
        const uint32_t first = ((lane >> run) * nsteps << run) + (lane & ((1u << run) - 1u));
        const uint32_t s0 = (c - uniform(bt.cstart[lo])) * bt.spc, s1 = min(s0 + bt.spc, nsteps);
        for (uint32_t step = s0; step < s1; ++step) {
            const uint32_t rel = first + (step << run), slot = q0 + rel;
            const bool valid = lane < per && rel < nq;
            const uint32_t qi = valid ? (bt.perm ? bt.perm[slot] : slot) : 0u;
            if (valid)
                W.start(lane, load_point<3>(q, qi));
            if (KIND == 0)
                cp_wave<false, 3>(tv, (uint32_t)__popcll(__ballot(valid)), W, cnt, ovf); // valid: a prefix of the lanes
            else
                sil_wave<false, 3, KIND - 1>(tv, __ballot(valid), flip != 0, KIND == 2 && valid ? seed[qi] : F_INF, W,
                                             cnt, ovf);
            if (valid) {
                float best;
                uint32_t bi;
                unpack_best(W.best[lane], best, bi);
                if (out_idx)
                    out_idx[qi] = bi;
                out_dist[qi] = KIND == 0 ? dm::sqrt_(best) : best;
            }
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

hipError_t launch_batch(const snch_scene* s, int kind, const float* q, const uint32_t* q_off_host, int flip,
                        uint32_t* out_idx, float* out_dist, const BatchConfig& cfg, hipStream_t st,
                        const float* seed)
{
    const uint32_t M = s->n_meshes;
    BatchState& b = s->batch;
    const uint32_t n = q_off_host[M];
    if (n == 0)
        return hipSuccess;
    // as many waves as are resident, and no more than chunks
    const uint32_t wpb = cfg.block_size / 64, cap = pool_cap(cfg.stack_depth);
    const size_t lds = sizeof(uint32_t) * wpb * wave_lds_words(cap);
    const uint32_t per_cu = std::max(1u, std::min((uint32_t)(LDS_PER_CU / lds), 24u / wpb));
    const uint32_t deal = deal_queries(n, s->n_cu() * per_cu * wpb, kind == 0 ? CP_RUNS : SIL_RUNS);
    const uint32_t spc = std::max(1u, cfg.queries_per_wave / 64u), per_chunk = spc * (deal & 255u);
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
        total += cnt / per_chunk + (cnt % per_chunk ? 1u : 0u);
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
    bt.deal = deal;
    bt.spc = spc;
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
    const dim3 g(std::max(1u, std::min(s->n_cu() * per_cu, nblocks(total, wpb)))), blk(cfg.block_size);
#define SNCH_BATCH(K_)                                                                                               \
    hipLaunchKernelGGL((k_batch<K_>), g, blk, lds, st, bt, cap, q, flip, seed, out_idx, out_dist, traversal_error_word())
    if (kind == 0)
        SNCH_BATCH(0);
    else if (seed)
        SNCH_BATCH(2);
    else
        SNCH_BATCH(1);
#undef SNCH_BATCH
    return hipGetLastError();
}

} // namespace snch
