// Query kernels for triangle scenes on gfx950: closest primitive, closest
// silhouette, ray (closest hit / any hit) and SampleTriangleInSphere.
//
// The reference runs one thread per query (query_device, query.cuh:79-423, and
// sample_object_in_sphere, sample.cuh:23-92).  Here the searches run up to 64
// queries per wave from a pool; the sampler and the generic overlap and line
// queries keep one lane per query.  Differences in HOW, not WHAT:
//  * Node layout: one 64-B record per internal node holds both children's
//    boxes and references, 32 B each; the silhouette query reads a cone record
//    from a separate stream, so the closest-point and ray queries never touch
//    it.
//  * The searches run a wave's queries from one pool of pending nodes in LDS
//    (wave_search.hpp).  The generic overlap and line queries, which must emit
//    hits in the reference's visit order, keep 16 LDS entries per lane over a
//    private overflow array (the tree depth is at most 64, so it never loses
//    one).
//  * Order: the nearer child is descended first and the farther is pushed,
//    and a child is skipped when its lower bound exceeds the best answer so
//    far.  The reference's own pruning predicates (minmaxdist for closest
//    point, cone overlap for silhouettes, slab tests for rays) are evaluated
//    unchanged; the added bound checks are conservative.
//  * Ties: among candidates at exactly the same distance the smallest index
//    wins (the reference keeps the last visited one for closest point and
//    silhouette, query.cuh:286/:383, and the first for rays, :115).  The
//    answer is then a function of the candidate set alone, independent of
//    visit order, block size or a seeded search radius.
//  * Blocks are remapped so that each of the 8 XCDs processes one contiguous
//    range of queries (blocks are dispatched round-robin over XCDs).
#include "wave_search.hpp"

namespace snch {

namespace {

constexpr int SS = 16;  // LDS stack entries per lane (generic queries)
constexpr int OVF = 64; // private overflow entries per lane (generic queries)

// ------------------------------------------------------------ closest point
template <bool STATS, int DIM>
__global__ __launch_bounds__(512, 6) void k_closest_point(TreeView t, const float* __restrict__ q, uint32_t n,
                                                          uint32_t deal, uint32_t cap, uint32_t* __restrict__ out_idx,
                                                          float* __restrict__ out_dist,
                                                          const uint32_t* __restrict__ perm, uint32_t* ctr,
                                                          uint32_t* __restrict__ err, unsigned long long* stats)
{
    extern __shared__ __align__(16) uint32_t smem[];
    const uint32_t lane = threadIdx.x & 63;
    WaveLds W(smem + (threadIdx.x >> 6) * wave_lds_words(cap), cap);
    if (t.n_dev)
        n = min(n, *t.n_dev);
    if (deal == 0u)
        deal = deal_queries(n, gridDim.x * (blockDim.x >> 6), CP_RUNS);
    bool ovf = false;
    Counts cnt;
    for_chunks(n, deal, ctr, [&](uint32_t slot, bool valid) {
        const uint32_t qi = valid ? (perm ? min(perm[slot], n - 1) : slot) : 0u;
        if (valid)
            W.start(lane, load_point<DIM>(q, qi));
        cp_wave<STATS, DIM>(t, (uint32_t)__popcll(__ballot(valid)), W, cnt, ovf);
        if (valid) {
            float best;
            uint32_t best_idx;
            unpack_best(W.best[lane], best, best_idx);
            out_idx[qi] = best_idx;
            out_dist[qi] = dm::sqrt_(best);
        }
    });
    if (ovf && err)
        atomicOr(err, 1u);
    if (STATS)
        flush_counts(cnt, stats);
}

// ------------------------------------------------------------ ray
// out_uv: the hit's barycentrics (2D: the segment parameter), from the hit
// test of the triangle found
template <bool STATS, int DIM, bool ANY>
__global__ __launch_bounds__(64, 6) void k_ray(TreeView t, const float4* __restrict__ V, const int32_t* __restrict__ F,
                                               const float* __restrict__ o, const float* __restrict__ d,
                                               const float* __restrict__ tmax, uint32_t n, uint32_t deal,
                                               uint8_t* __restrict__ out_hit, float* __restrict__ out_t,
                                               float* __restrict__ out_uv, uint32_t* __restrict__ out_idx,
                                               uint32_t* ctr, uint32_t* __restrict__ err, unsigned long long* stats)
{
    __shared__ __align__(16) uint32_t smem[RayLds::WORDS];
    const uint32_t lane = threadIdx.x & 63;
    RayLds W(smem);
    if (t.n_dev)
        n = min(n, *t.n_dev);
    if (deal == 0u)
        deal = deal_queries(n, gridDim.x, RAY_RUNS);
    bool ovf = false;
    Counts cnt;
    for_chunks(n, deal, ctr, [&](uint32_t qi, bool valid) {
        float max_dist = F_INF;
        v3 ro = mk(0.0f, 0.0f, 0.0f), rd = ro;
        if (valid) {
            ro = load_point<DIM>(o, qi);
            rd = load_point<DIM>(d, qi);
            if (tmax)
                max_dist = tmax[qi];
            // aabb.cuh:308-311 (2D: z slab inert)
            W.start(lane, ro, rd, mk(1.0f / rd.x, 1.0f / rd.y, 1.0f / rd.z), max_dist);
        }
        ray_wave<STATS, DIM, ANY>(t, __ballot(valid), max_dist, W, cnt, ovf);
        if (!valid)
            return;
        float tbest;
        uint32_t idx;
        unpack_best(W.best[lane], tbest, idx);
        const bool found = idx != INVALID;
        if (out_hit)
            out_hit[qi] = found ? 1 : 0;
        if (ANY)
            return;
        float u = 0.0f, v = 0.0f;
        if (found && (out_uv || out_t)) {
            const v3 o2 = W.origin(lane), d2 = W.dir(lane);
            if (DIM == 3) {
                const float4 a = V[F[3 * idx]], b = V[F[3 * idx + 1]], c = V[F[3 * idx + 2]];
                ray_triangle(o2, d2, mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), mk(c.x, c.y, c.z), tbest, u, v);
            } else {
                const float4 a = V[F[2 * idx]], b = V[F[2 * idx + 1]];
                ray_segment(o2, d2, mk(a.x, a.y, 0.0f), mk(b.x, b.y, 0.0f), tbest, u);
            }
        }
        if (out_t)
            out_t[qi] = tbest;
        if (out_uv) {
            if (DIM == 3) {
                out_uv[2 * qi] = u;
                out_uv[2 * qi + 1] = v;
            } else {
                out_uv[qi] = u; // segment parameter s
            }
        }
        if (out_idx)
            out_idx[qi] = idx;
    });
    if (ovf && err)
        atomicOr(err, 1u);
    if (STATS)
        flush_counts(cnt, stats);
}

// ------------------------------------------------------------ sampling
// sample.cuh:23-92: a single root-to-leaf descent, bit-identical to the
// reference's FP32 arithmetic (u rescaled at each level).
template <int DIM>
__global__ __launch_bounds__(256) void k_sample(TreeView t, const float4* __restrict__ V,
                                                const int32_t* __restrict__ F, const float* __restrict__ cc,
                                                const float* __restrict__ rr, const float* __restrict__ uu,
                                                uint32_t n, int32_t* __restrict__ out_idx,
                                                float* __restrict__ out_pdf, float* __restrict__ out_pt)
{
    const uint32_t qi = xcd_remap(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (t.n_dev)
        n = min(n, *t.n_dev);
    if (qi >= n)
        return;
    const v3 c = load_point<DIM>(cc, qi);
    int32_t obj;
    float pdf;
    v3 pt;
    sample_one<DIM>(t, V, F, c, rr[qi], uu[3 * qi], uu[3 * qi + 1], uu[3 * qi + 2], obj, pdf, pt);
    out_idx[qi] = obj;
    out_pdf[qi] = pdf;
    if (out_pt) {
        if (DIM == 3) {
            out_pt[3 * qi] = pt.x;
            out_pt[3 * qi + 1] = pt.y;
            out_pt[3 * qi + 2] = pt.z;
        } else {
            out_pt[2 * qi] = pt.x;
            out_pt[2 * qi + 1] = pt.y;
        }
    }
}

template <int DIM>
__global__ __launch_bounds__(256) void k_sample_on_object(const float4* __restrict__ V, const int32_t* __restrict__ F,
                                                          uint32_t nF, const int32_t* __restrict__ idx,
                                                          const float* __restrict__ uv, uint32_t n,
                                                          float* __restrict__ out_pt)
{
    const uint32_t qi = blockIdx.x * 256 + threadIdx.x;
    if (qi >= n)
        return;
    const int32_t o = idx[qi];
    v3 pt = mk(0.0f, 0.0f, 0.0f);
    if (o >= 0 && (uint32_t)o < nF) {
        if (DIM == 3) {
            const float4 a = V[F[3 * o]], b = V[F[3 * o + 1]], d = V[F[3 * o + 2]];
            pt = sample_triangle(mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), mk(d.x, d.y, d.z), uv[2 * qi],
                                 uv[2 * qi + 1]);
        } else {
            const float4 a = V[F[2 * o]], b = V[F[2 * o + 1]];
            const float u1 = uv[2 * qi];
            pt = mk(a.x + u1 * (b.x - a.x), a.y + u1 * (b.y - a.y), 0.0f);
        }
    }
    if (DIM == 3) {
        out_pt[3 * qi] = pt.x;
        out_pt[3 * qi + 1] = pt.y;
        out_pt[3 * qi + 2] = pt.z;
    } else {
        out_pt[2 * qi] = pt.x;
        out_pt[2 * qi + 1] = pt.y;
    }
}

// ------------------------------------------------------------ overlap / line
// query_device(bvh, overlaps(box), out, max) (query.cuh:176-231) and
// query_device(bvh, line_intersect(line), element_test, out, max)
// (query.cuh:12-77): every primitive whose leaf box meets the query box
// (aabb.cuh:54-82) or the infinite line (slab test, aabb.cuh:330-364; the
// element test is the scene's ray test without t >= 0), emitted in the
// reference's order: pop a node, test its left then its right child, emit a
// leaf at once, push an internal child.  The first max_out ids (and line
// parameters) land in the query's row; count = all found.  The node ids are
// the reference's, so the order is the reference's bit for bit.
template <int BS, int SSZ>
struct IdStack {
    uint32_t* lds; // this lane's column: entry s at lds[s * BS]
    int sp;
    uint32_t ov[OVF];
    bool overflow;
    __device__ __forceinline__ void init(uint32_t* base)
    {
        lds = base;
        sp = 0;
        overflow = false;
    }
    __device__ __forceinline__ void push(uint32_t n)
    {
        const int s = sp % SSZ;
        if (sp >= SSZ) {
            if (sp - SSZ >= OVF) {
                overflow = true;
                return;
            }
            ov[sp - SSZ] = lds[s * BS];
        }
        lds[s * BS] = n;
        ++sp;
    }
    __device__ __forceinline__ uint32_t pop()
    {
        --sp;
        const int s = sp % SSZ;
        const uint32_t n = lds[s * BS];
        if (sp >= SSZ)
            lds[s * BS] = ov[sp - SSZ];
        return n;
    }
};

template <int DIM>
__device__ __forceinline__ bool overlap_box(const box3& b, const box3& q)
{
    if (b.hi.x < q.lo.x || q.hi.x < b.lo.x || b.hi.y < q.lo.y || q.hi.y < b.lo.y)
        return false;
    return DIM == 2 || !(b.hi.z < q.lo.z || q.hi.z < b.lo.z);
}

template <int DIM>
__device__ __forceinline__ bool line_box(const box3& b, v3 o, v3 inv)
{
    float t1 = (b.lo.x - o.x) * inv.x, t2 = (b.hi.x - o.x) * inv.x;
    float tmin = fmn(t1, t2), tmax = fmx(t1, t2);
    t1 = (b.lo.y - o.y) * inv.y;
    t2 = (b.hi.y - o.y) * inv.y;
    tmin = fmx(tmin, fmn(t1, t2));
    tmax = fmn(tmax, fmx(t1, t2));
    if (DIM == 3) {
        t1 = (b.lo.z - o.z) * inv.z;
        t2 = (b.hi.z - o.z) * inv.z;
        tmin = fmx(tmin, fmn(t1, t2));
        tmax = fmn(tmax, fmx(t1, t2));
    }
    return tmax >= tmin;
}

template <int BS, int DIM, int KIND>
__global__ __launch_bounds__(BS) void k_generic(TreeView t, const float* __restrict__ qa, const float* __restrict__ qb,
                                                uint32_t n, uint32_t max_out, uint32_t* __restrict__ out_count,
                                                uint32_t* __restrict__ out_idx, float* __restrict__ out_t,
                                                uint32_t* __restrict__ err)
{
    __shared__ uint32_t stk[SS * BS];
    const uint32_t qi = xcd_remap(blockIdx.x, gridDim.x) * BS + threadIdx.x;
    if (qi >= n)
        return;
    // KIND 0: the box [qa, qb]; KIND 1: the line through qa along qb
    const v3 a = load_point<DIM>(qa, qi), b = load_point<DIM>(qb, qi);
    box3 qbox;
    qbox.lo = a;
    qbox.hi = b;
    const v3 inv = mk(1.0f / b.x, 1.0f / b.y, DIM == 3 ? 1.0f / b.z : 0.0f); // line(o, dir) (aabb.cuh:288-294)
    uint32_t found = 0;
    const size_t row = (size_t)qi * max_out;
    auto hit_box = [&](const box3& bx) { return KIND == 0 ? overlap_box<DIM>(bx, qbox) : line_box<DIM>(bx, a, inv); };
    auto emit = [&](uint32_t j) {
        if (j >= t.n_leaves)
            return;
        const float4 la = t.tleaf[3 * j], lb = t.tleaf[3 * j + 1];
        float tt = 0.0f;
        bool ok = true;
        if (KIND == 1) {
            float uh, vh;
            if (DIM == 3) {
                const float4 lc = t.tleaf[3 * j + 2];
                ok = line_triangle(a, b, mk(la.x, la.y, la.z), mk(lb.x, lb.y, lb.z), mk(lc.x, lc.y, lc.z), tt, uh, vh);
            } else {
                ok = line_segment(a, b, mk(la.x, la.y, 0.0f), mk(lb.x, lb.y, 0.0f), tt, uh);
            }
        }
        if (!ok)
            return;
        if (found < max_out) {
            out_idx[row + found] = __float_as_uint(la.w);
            if (KIND == 1 && out_t)
                out_t[row + found] = tt;
        }
        ++found;
    };
    if (t.n_leaves == 1) {
        if (hit_box(ldbox2(t.nbox, 0)))
            emit(0);
    } else {
        IdStack<BS, SS> st;
        st.init(stk + threadIdx.x);
        st.push(0);
        // each internal node is pushed at most once
        for (uint32_t it = 0; it < t.n_leaves && st.sp > 0; ++it) {
            const NodeRec nr = load_node(t.tnode, st.pop());
            if (hit_box(nr.L)) {
                if (nr.lref & LEAF_BIT)
                    emit(nr.lref & REF_MASK);
                else
                    st.push(nr.lref & REF_MASK);
            }
            if (hit_box(nr.R)) {
                if (nr.rref & LEAF_BIT)
                    emit(nr.rref & REF_MASK);
                else
                    st.push(nr.rref & REF_MASK);
            }
        }
        if (st.overflow && err)
            atomicOr(err, 1u);
    }
    out_count[qi] = found;
}

// Morton code of each query point in the root box (clamped to it), used to
// visit queries in spatial order: neighbouring lanes then walk mostly the
// same nodes, which keeps a wave's memory accesses and branches together
template <int DIM>
__global__ __launch_bounds__(256) void k_query_codes(const float4* __restrict__ nbox, const float* __restrict__ q,
                                                     uint32_t n, uint32_t* __restrict__ codes,
                                                     uint32_t* __restrict__ idx)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    const float4 lo = nbox[0], hi = nbox[1];
    const v3 p = load_point<DIM>(q, i);
    const float x = (p.x - lo.x) / (hi.x - lo.x), y = (p.y - lo.y) / (hi.y - lo.y);
    codes[i] = DIM == 3 ? morton3(mk(x, y, (p.z - lo.z) / (hi.z - lo.z))) : morton2(x, y);
    idx[i] = i;
}

} // namespace

hipError_t query_order(const TreeView& t, int dim, const float* q, uint32_t n, QueryScratch& w, hipStream_t st,
                       const uint32_t** perm)
{
    *perm = nullptr;
    if (n < 2)
        return hipSuccess;
    hipError_t e;
    if ((e = w.codes.ensure(sizeof(uint32_t) * n)) != hipSuccess || (e = w.idx.ensure(sizeof(uint32_t) * n)) ||
        (e = w.codes_alt.ensure(sizeof(uint32_t) * n)) || (e = w.idx_alt.ensure(sizeof(uint32_t) * n)))
        return e;
    SNCH_DISPATCH_DIM(dim, hipLaunchKernelGGL(k_query_codes<DIM>, dim3(nblocks(n, 256)), dim3(256), 0, st, t.nbox,
                                              q, n, w.codes.as<uint32_t>(), w.idx.as<uint32_t>()));
    bool in_alt = false;
    if ((e = radix_sort_pairs(w.codes.as<uint32_t>(), w.idx.as<uint32_t>(), w.codes_alt.as<uint32_t>(),
                              w.idx_alt.as<uint32_t>(), n, 30, w.hist, st, &in_alt)) != hipSuccess)
        return e;
    *perm = in_alt ? w.idx_alt.as<uint32_t>() : w.idx.as<uint32_t>();
    return hipGetLastError();
}

size_t query_order_scratch_bytes(uint32_t n)
{
    return sizeof(uint32_t) * 4 * (size_t)n + radix_sort_scratch_bytes(n, 4);
}

hipError_t query_order_in(const TreeView& t, int dim, const float* q, uint32_t n, uint32_t* words, hipStream_t st,
                          const uint32_t** perm, uint32_t* err)
{
    *perm = nullptr;
    if (n < 2)
        return hipSuccess;
    uint32_t *codes = words, *idx = words + n, *codes_alt = words + 2 * (size_t)n, *idx_alt = words + 3 * (size_t)n;
    SNCH_DISPATCH_DIM(dim, hipLaunchKernelGGL(k_query_codes<DIM>, dim3(nblocks(n, 256)), dim3(256), 0, st, t.nbox,
                                              q, n, codes, idx));
    bool in_alt = false;
    const hipError_t e = radix_sort_pairs_in(codes, idx, codes_alt, idx_alt, n, 30, words + 4 * (size_t)n, st,
                                             &in_alt, err);
    if (e != hipSuccess)
        return e;
    *perm = in_alt ? idx_alt : idx;
    return hipGetLastError();
}

hipError_t launch_closest_point(const TreeView& t, int dim, const float* q, uint32_t n, uint32_t* idx, float* dist,
                                uint32_t block, uint32_t depth, const uint32_t* perm, uint64_t* stats, uint32_t* ctr,
                                uint32_t n_cu, hipStream_t st)
{
    if (n == 0)
        return hipSuccess;
    auto* sp = reinterpret_cast<unsigned long long*>(stats);
    const SearchGrid g = search_grid(n, block, wave_lds_words(pool_cap(depth)), n_cu, 6, ctr != nullptr,
                                      t.n_dev != nullptr, CP_RUNS);
    uint32_t* c = g.persist ? ctr : nullptr;
    SNCH_DISPATCH_DIM(dim, {
        if (stats)
            hipLaunchKernelGGL((k_closest_point<true, DIM>), g.grid, g.block, g.lds, st, t, q, n, g.deal,
                               pool_cap(depth), idx, dist, perm, c, traversal_error_word(), sp);
        else
            hipLaunchKernelGGL((k_closest_point<false, DIM>), g.grid, g.block, g.lds, st, t, q, n, g.deal,
                               pool_cap(depth), idx, dist, perm, c, traversal_error_word(), sp);
    });
    return hipGetLastError();
}

hipError_t launch_ray(const TreeView& t, int dim, const float4* V, const int32_t* F, const float* o, const float* d,
                      const float* tmax, uint32_t n, int any_hit, uint8_t* hit, float* tout, float* uv, uint32_t* idx,
                      uint64_t* stats, uint32_t* ctr, uint32_t n_cu, hipStream_t st)
{
    if (n == 0)
        return hipSuccess;
    auto* sp = reinterpret_cast<unsigned long long*>(stats);
    const SearchGrid g = search_grid(n, 64, RayLds::WORDS, n_cu, 6, ctr != nullptr, t.n_dev != nullptr, RAY_RUNS);
    uint32_t* c = g.persist ? ctr : nullptr;
#define SNCH_RAY(S_, A_)                                                                                             \
    hipLaunchKernelGGL((k_ray<S_, DIM, A_>), g.grid, g.block, 0, st, t, V, F, o, d, tmax, n, g.deal, hit, tout, uv, idx, \
                       c, traversal_error_word(), sp)
    SNCH_DISPATCH_DIM(dim, {
        if (any_hit) {
            if (stats)
                SNCH_RAY(true, true);
            else
                SNCH_RAY(false, true);
        } else if (stats) {
            SNCH_RAY(true, false);
        } else {
            SNCH_RAY(false, false);
        }
    });
#undef SNCH_RAY
    return hipGetLastError();
}

hipError_t launch_sample(const TreeView& t, int dim, const float4* V, const int32_t* F, const float* c,
                         const float* r, const float* u, uint32_t n, int32_t* idx, float* pdf, float* pt,
                         hipStream_t st)
{
    if (n == 0)
        return hipSuccess;
    SNCH_DISPATCH_DIM(dim, hipLaunchKernelGGL(k_sample<DIM>, dim3(nblocks(n, 256)), dim3(256), 0, st, t, V, F, c, r,
                                              u, n, idx, pdf, pt));
    return hipGetLastError();
}

hipError_t launch_generic(const TreeView& t, int dim, int kind, const float* qa, const float* qb, uint32_t n,
                          uint32_t max_out, uint32_t* count, uint32_t* idx, float* tout, hipStream_t st)
{
    if (n == 0)
        return hipSuccess;
    uint32_t* err = traversal_error_word();
    SNCH_DISPATCH_DIM(dim, {
        if (kind == 0)
            hipLaunchKernelGGL((k_generic<64, DIM, 0>), dim3(nblocks(n, 64)), dim3(64), 0, st, t, qa, qb, n, max_out,
                               count, idx, tout, err);
        else
            hipLaunchKernelGGL((k_generic<64, DIM, 1>), dim3(nblocks(n, 64)), dim3(64), 0, st, t, qa, qb, n, max_out,
                               count, idx, tout, err);
    });
    return hipGetLastError();
}

hipError_t launch_sample_on_object(int dim, const float4* V, const int32_t* F, uint32_t nF, const int32_t* idx,
                                   const float* uv, uint32_t n, float* pt, hipStream_t st)
{
    if (n == 0)
        return hipSuccess;
    SNCH_DISPATCH_DIM(dim, hipLaunchKernelGGL(k_sample_on_object<DIM>, dim3(nblocks(n, 256)), dim3(256), 0, st, V,
                                              F, nF, idx, uv, n, pt));
    return hipGetLastError();
}

} // namespace snch
