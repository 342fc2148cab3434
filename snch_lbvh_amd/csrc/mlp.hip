// Learned distance bound: a Fourier-feature MLP on BF16 MFMA (gfx950).
//
//   x -> xhat = (x - c) / h              (scene box -> [-1, 1]^3)
//   f = [sin(B xhat), cos(B xhat)]       (B: 32 x 3, N(0, sigma^2) radians per
//                                         normalised unit, fixed)
//   z1 = W1 f + b1, a1 = silu(z1)        (64 -> 128)
//   z2..z4 likewise                      (128 -> 128, three layers)
//   o = w5 . a4 + b5                     (128 -> 1)
// The network regresses o ~ log(min(d / D, 1) + 1e-3) where d is a query's
// exact closest-silhouette distance and D the scene box diagonal; the seed
// radius is r0 = ((exp(o) - 1e-3) * (1 + rel) + abs) * D.  The exact
// traversal verifies every answer (query.hip), so the network only changes
// how fast a query runs, never its result.
//
// Kernels:
//   k_mlp_infer   out^T = W x^T per layer on v_mfma_f32_16x16x32_bf16 (gfx950's
//                 K = 32 BF16 MFMA): the weights are the A operand, staged in
//                 LDS once per block (112 KB) and shared by its 16 waves; the
//                 activations are the B operand and never leave registers: a
//                 layer's accumulator tiles are turned into the next layer's
//                 B fragments in place, because the hidden features are
//                 numbered so that the output layout of two 16-row tiles is
//                 the B layout of one 32-deep K block (see infer_index);
//                 each wave takes P tiles of 16 points, so every weight
//                 fragment read from LDS feeds P MFMAs (one wave = 16 P points)
//   k_mlp_train   forward + backward over 64-point tiles, one persistent
//                 workgroup of 16 waves per CU: waves (w, 0) and (w, 1) own
//                 output rows 16 w .. 16 w + 15 of every layer, for half of
//                 the points each; they keep their pre-activations, and the
//                 gradient of half of the rows' columns each (56 accumulators
//                 per lane) over all tiles, in registers, and write it once
//   k_mlp_reduce  sums the workgroups' gradients
//   k_mlp_adam    the same, and Adam on FP32 master weights; writes the BF16
//                 copies in the two MFMA fragment orders (infer_index and
//                 back_index)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "internal.hpp"

namespace snch {
namespace mlpk {

constexpr int NFREQ = 32, NIN = 64, H = 128;
constexpr int OFF_W[4] = {0, 8320, 24832, 41344};
constexpr int OFF_B[4] = {8192, 24704, 41216, 57728};
constexpr int KIN[4] = {64, 128, 128, 128};
constexpr int OFF_W5 = 57856, OFF_B5 = 57984, NPARAM = 57985;
constexpr int SW_OFF[4] = {0, 8192, 24576, 40960}; // offsets in the bf16 fragment arrays
constexpr int NSW = 57344;
constexpr float LOG_EPS = 1e-3f;
#ifndef MLP_INFER_WAVES
#define MLP_INFER_WAVES 16 // waves per inference block (they share one LDS copy of the weights)
#endif
#ifndef MLP_INFER_TILES
#define MLP_INFER_TILES 2 // 16-point tiles per wave at a time (reuse of each weight fragment)
#endif

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));
struct v4s8 {
    v4s lo, hi;
};

__host__ __device__ __forceinline__ unsigned short f2bf(float f)
{
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    u += 0x7FFFu + ((u >> 16) & 1u); // round to nearest even (finite inputs)
    return (unsigned short)(u >> 16);
}
__host__ __device__ __forceinline__ float bf2f(unsigned short h) { return __builtin_bit_cast(float, (uint32_t)h << 16); }

// D (16 x 16) += A (16 x 32) B (32 x 16); lane l = 16 g + r holds A[r][8 g + j],
// B[8 g + j][r] (j = 0..7) and D[4 g + i][r] (i = 0..3)
__device__ __forceinline__ v4f mma32(v8bf a, v8bf b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// the same in two steps of 16: positions j < 4 of all lanes, then j >= 4 (sums
// in the order of the features, see k_mlp_train)
__device__ __forceinline__ v4f mma16x2(v8bf a, v8bf b, v4f c)
{
    const v4s8 x = __builtin_bit_cast(v4s8, a), y = __builtin_bit_cast(v4s8, b);
    c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x.lo, y.lo, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x.hi, y.hi, c, 0, 0, 0);
}

// fragment index of W_l[n][k] for k_mlp_infer: the A operand of tile (mt, kb)
// (16 output rows x 32 inputs) is 64 lanes x 8 BF16, lane 16 g + r holding
// row 16 mt + r.  Layer 0 reads the features in order (position 8 g + j of
// block kb is input 32 kb + 8 g + j).  Layers 1-3 read the previous layer's
// outputs as its accumulators leave them: lane 16 g + r of output tiles 2 kb
// and 2 kb + 1 holds rows 4 g + i of each, so position 8 g + j of block kb is
// input 32 kb + 4 g + j (j < 4) or 32 kb + 16 + 4 g + j - 4 (j >= 4).
__host__ __device__ __forceinline__ int infer_index(int l, int n, int k)
{
    const int KB = KIN[l] >> 5, mt = n >> 4, r = n & 15, kb = k >> 5, kl = k & 31;
    int g, j;
    if (l == 0) {
        g = kl >> 3;
        j = kl & 7;
    } else {
        g = (kl & 15) >> 2;
        j = (kl & 3) + (kl >= 16 ? 4 : 0);
    }
    return SW_OFF[l] + (((mt * KB + kb) * 64 + 16 * g + r) << 3) + j;
}

// fragment index of W_0[n][k] for k_mlp_train: the same, with the features
// ordered within a block as the hidden layers' inputs are
__host__ __device__ __forceinline__ int train0_index(int n, int k)
{
    const int kl = k & 31, g = (kl & 15) >> 2, j = (kl & 3) + (kl >= 16 ? 4 : 0);
    return ((((n >> 4) * (NIN >> 5) + (k >> 5)) * 64 + 16 * g + (n & 15)) << 3) + j;
}

// fragment index of W_l[n][k], l >= 1, for the deltas W_l^T delta_l of
// k_mlp_train: the A operand of tile (kt, nb) (16 inputs x 32 outputs), lane
// 16 g + r holding input 16 kt + r, outputs in the order of infer_index
__host__ __device__ __forceinline__ int back_index(int l, int n, int k)
{
    const int kt = k >> 4, r = k & 15, nb = n >> 5, nl = n & 31, g = (nl & 15) >> 2, j = (nl & 3) + (nl >= 16 ? 4 : 0);
    return SW_OFF[l] + (((kt * (H >> 5) + nb) * 64 + 16 * g + r) << 3) + j;
}

struct Frame {
    float cx, cy, cz, ihx, ihy, ihz, invD;
    float tau; // loss asymmetry: weight 2 tau on under-prediction, 2 (1 - tau) on over-prediction
};

// ------------------------------------------------------------------ infer
// One hidden layer L for P tiles of 16 points: acc = W_L bop (+ bias, SiLU);
// the results become the next layer's B operand in place (L < 3) or are dotted
// with the output weights (L = 3: o = partial w5 . a4 of this lane's rows).
// A function per layer keeps every register array statically indexed.
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
// two floats as one word of two round-to-nearest-even BF16 halves (low first):
// one v_cvt_pk_bf16_f32 on gfx950
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{lo, hi}, v2bf));
}
// SiLU for the inference path: the hardware exp and reciprocal (about 1 ulp,
// far inside the BF16 rounding its result gets)
__device__ __forceinline__ float silu_fast(float z) { return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

template <int L, int P>
__device__ __forceinline__ void infer_layer(const v4u* sW, const float* sB, v4u (&bop)[P][4], float (&o)[P],
                                            int lane, int g)
{
    constexpr int KB = KIN[L] >> 5;
    v4f acc[P][8];
#pragma unroll
    for (int pt = 0; pt < P; ++pt)
#pragma unroll
        for (int mt = 0; mt < 8; ++mt)
            acc[pt][mt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int mt = 0; mt < 8; ++mt) {
            const v8bf a = __builtin_bit_cast(v8bf, sW[(SW_OFF[L] >> 3) + (mt * KB + kb) * 64 + lane]);
#pragma unroll
            for (int pt = 0; pt < P; ++pt)
                acc[pt][mt] = mma32(a, __builtin_bit_cast(v8bf, bop[pt][kb]), acc[pt][mt]);
        }
    // bias + SiLU; lane (g, r) holds outputs 16 mt + 4 g + i of point r
#pragma unroll
    for (int pt = 0; pt < P; ++pt) {
        float s = 0.0f;
#pragma unroll
        for (int mt = 0; mt < 8; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 16 * mt + 4 * g + i;
                acc[pt][mt][i] = silu_fast(acc[pt][mt][i] + sB[L * H + row]);
                if (L == 3)
                    s += sB[4 * H + row] * acc[pt][mt][i];
            }
        o[pt] = s;
        if (L < 3) { // tiles 2 kb and 2 kb + 1 become K block kb of the next layer
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                const v4f a0 = acc[pt][2 * kb], a1 = acc[pt][2 * kb + 1];
                bop[pt][kb] = v4u{pack_bf16(a0[0], a0[1]), pack_bf16(a0[2], a0[3]), pack_bf16(a1[0], a1[1]),
                                  pack_bf16(a1[2], a1[3])};
            }
        }
    }
}

// mode 0: predicted distance; mode 1: seed radius.  NW waves per block share
// the LDS weights; each wave takes P tiles of 16 points at a time.
template <int NW, int P>
__global__ __launch_bounds__(NW * 64) void k_mlp_infer(const v4u* __restrict__ wisw, const float* __restrict__ theta,
                                                       const float* __restrict__ fourier, Frame fr,
                                                       const float* __restrict__ pts, uint32_t n, int mode, float rel,
                                                       float absm, float D, float* __restrict__ out)
{
    __shared__ v4u sW[NSW / 8];
    __shared__ float sB[4 * H + H + 1];
    __shared__ float sFour[3 * NFREQ];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, g = lane >> 4;
    for (int i = tid; i < NSW / 8; i += NW * 64)
        sW[i] = wisw[i];
    for (int i = tid; i < 4 * H; i += NW * 64)
        sB[i] = theta[OFF_B[i / H] + (i % H)];
    for (int i = tid; i < H; i += NW * 64)
        sB[4 * H + i] = theta[OFF_W5 + i];
    if (tid == 0)
        sB[5 * H] = theta[OFF_B5];
    for (int i = tid; i < 3 * NFREQ; i += NW * 64)
        sFour[i] = fourier[i];
    __syncthreads();
    const uint32_t ntiles = (n + 15) / 16;
    for (uint32_t t0 = ((uint32_t)blockIdx.x * NW + w) * P; t0 < ntiles; t0 += gridDim.x * NW * P) {
        // a compiler-level memory barrier: the weight fragments are the same in
        // every iteration, and without it the compiler hoists all 112 of their
        // LDS reads out of the loop (448 registers, spilled to scratch)
        asm volatile("" ::: "memory");
        // layer-0 B operand: features of point r of each tile, frequencies 8 g .. 8 g + 7
        v4u bop[P][4];
#pragma unroll
        for (int pt = 0; pt < P; ++pt) {
            const uint32_t p = (t0 + pt) * 16 + r;
            const bool valid = p < n;
            const float x = valid ? pts[3 * p] : 0.0f, y = valid ? pts[3 * p + 1] : 0.0f,
                        z = valid ? pts[3 * p + 2] : 0.0f;
            const float xh = (x - fr.cx) * fr.ihx, yh = (y - fr.cy) * fr.ihy, zh = (z - fr.cz) * fr.ihz;
            float sn[8], cs[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int fi = 8 * g + j;
                const float arg = sFour[3 * fi] * xh + sFour[3 * fi + 1] * yh + sFour[3 * fi + 2] * zh;
                sn[j] = __sinf(arg); // hardware sine and cosine (|arg| stays below ~40 rad):
                cs[j] = __cosf(arg); // errors far below the BF16 rounding of the features
            }
            bop[pt][0] = v4u{pack_bf16(sn[0], sn[1]), pack_bf16(sn[2], sn[3]), pack_bf16(sn[4], sn[5]),
                             pack_bf16(sn[6], sn[7])};
            bop[pt][1] = v4u{pack_bf16(cs[0], cs[1]), pack_bf16(cs[2], cs[3]), pack_bf16(cs[4], cs[5]),
                             pack_bf16(cs[6], cs[7])};
        }
        float o[P];
        infer_layer<0, P>(sW, sB, bop, o, lane, g);
        infer_layer<1, P>(sW, sB, bop, o, lane, g);
        infer_layer<2, P>(sW, sB, bop, o, lane, g);
        infer_layer<3, P>(sW, sB, bop, o, lane, g);
#pragma unroll
        for (int pt = 0; pt < P; ++pt) {
            float s = o[pt];
            s += __shfl_xor(s, 16, 64);
            s += __shfl_xor(s, 32, 64);
            const uint32_t p = (t0 + pt) * 16 + r;
            if (g == 0 && p < n) {
                float d = __expf(s + sB[5 * H]) - LOG_EPS;
                d = d > 0.0f ? d : 0.0f;
                out[p] = mode == 0 ? d * D : (d * (1.0f + rel) + absm) * D;
            }
        }
    }
}

// ------------------------------------------------------------------ train
constexpr int TP = 64;      // points per tile
constexpr int TW = 8;       // pairs of waves per workgroup: one per 16 hidden features
// LDS rows, one per point.  84 and 36 dwords: 16 bytes of 8 rows in a row lie
// in different banks of 64, and the 4 x 16 blocks that the transposing reads
// take in at most two cycles.
constexpr int ROW = 168, F_ROW = 72;

// F: features; A: the activations a1..a3; D: deltas of the current layer and of
// the one before (ping-pong).  All are in the K order of infer_index's hidden
// layers, so a row is a layer's MFMA operand; a weight gradient, a sum over
// points, reads its operands as columns (ds_read_b64_tr_b16).
struct TrainLds {
    unsigned short F[TP * F_ROW];
    unsigned short A[3][TP * ROW], D[2][TP * ROW];
    float out[TW][TP];
    float g[TP];
    float bias[4 * H], w5[H];
};

// 1 / (1 + e^-z), the reciprocal with a Newton step: as good as a division (the
// gradients are the same) and 0.065 ms of 0.62 less over 2^19 points
__device__ __forceinline__ float sigm(float z)
{
    const float d = fminf(1.0f + __expf(-z), 1e37f), q = __builtin_amdgcn_rcpf(d);
    return fmaf(fmaf(-d, q, 1.0f), q, q);
}
__device__ __forceinline__ float lane_xor(float v, int lane, int mask)
{
    return __int_as_float(__builtin_amdgcn_ds_bpermute((lane ^ mask) << 2, __float_as_int(v)));
}
__device__ __forceinline__ float bf_lo(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float bf_hi(uint32_t v) { return __uint_as_float(v & 0xFFFF0000u); }
__device__ __forceinline__ v4f unpack4(uint2 v) { return v4f{bf_lo(v.x), bf_hi(v.x), bf_lo(v.y), bf_hi(v.y)}; }
__device__ __forceinline__ v8bf frag(const unsigned short* p)
{
    return __builtin_bit_cast(v8bf, *reinterpret_cast<const v4u*>(p));
}

// column r of 16-feature block m over the points p0 + 8 g .. + 7 (lane 16 g + r).
// A transposing read gives lane r of 16 the column r of a 4 x 16 block whose row
// k the lanes 4 k .. 4 k + 3 point to, 4 values each.
template <int S>
__device__ __forceinline__ v8bf columns(unsigned short* rows, int m, int p0, int g, int r)
{
    unsigned short* a = rows + (p0 + 8 * g + (r >> 2)) * S + 32 * (m >> 1) + 8 * (r & 3) + 4 * (m & 1);
    typedef __attribute__((address_space(3))) v4s* ldsp;
    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ldsp)a),
              hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ldsp)(a + 4 * S));
    return __builtin_bit_cast(v8bf, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// four values of features 16 w + 4 g .. + 3 of point p, as BF16
__device__ __forceinline__ void put4(unsigned short* rows, int p, int w, int g, const v4f& v)
{
    *reinterpret_cast<uint2*>(rows + p * ROW + 32 * (w >> 1) + 8 * g + 4 * (w & 1)) =
        make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
}

// layer L forward for the wave's 16 rows and 32 points: pre-activations to z
// (BF16), activations to A[L] (not for the last layer)
template <int L>
__device__ __forceinline__ void train_forward(TrainLds& S, const v4u* __restrict__ wsw, int w, int h, int lane,
                                              uint2 (&z)[2])
{
    asm volatile("" : "+v"(lane));
    const int r = lane & 15, g = lane >> 4;
    constexpr int KB = KIN[L] >> 5;
    v8bf wf[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
        wf[kb] = __builtin_bit_cast(v8bf, wsw[(SW_OFF[L] >> 3) + (w * KB + kb) * 64 + lane]);
    const v4f b = *reinterpret_cast<const v4f*>(S.bias + L * H + 16 * w + 4 * g);
#pragma unroll
    for (int pt = 0; pt < 2; ++pt) {
        const int p = 32 * h + 16 * pt + r;
        const unsigned short* in = L == 0 ? S.F + p * F_ROW : S.A[L > 0 ? L - 1 : 0] + p * ROW;
        v4f acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
            acc = mma16x2(wf[kb], frag(in + 32 * kb + 8 * g), acc);
        z[pt] = make_uint2(pack_bf16(acc[0] + b[0], acc[1] + b[1]), pack_bf16(acc[2] + b[2], acc[3] + b[3]));
        if (L < 3) {
            v4f v = unpack4(z[pt]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[i] *= sigm(v[i]);
            put4(S.A[L < 3 ? L : 0], p, w, g, v);
        }
    }
}

// layer L backward: the wave's rows and half of the columns of dW_L
// (+= delta_L a_{L-1}^T), the rows of the bias gradient (wave L % 2 of the pair;
// per lane: this lane's points), then (L > 0) the deltas of layer L - 1 for its
// 16 inputs and 32 points, from D[cur] to D[cur ^ 1]
template <int L>
__device__ __forceinline__ void train_backward(TrainLds& S, const v4u* __restrict__ wtsw, int w, int h,
                                               int lane, const uint2 (&zprev)[2], v4f (&dw)[KIN[L] / 32],
                                               float& db)
{
    asm volatile("" : "+v"(lane));
    const int r = lane & 15, g = lane >> 4;
    constexpr int cur = (3 - L) & 1;
    v8bf wt[4];
    if (L > 0) {
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
            wt[nb] = __builtin_bit_cast(v8bf, wtsw[(SW_OFF[L] >> 3) + (w * 4 + nb) * 64 + lane]);
    }
    const v8bf d0 = columns<ROW>(S.D[cur], w, 0, g, r), d1 = columns<ROW>(S.D[cur], w, 32, g, r);
    if (h == (L & 1)) {
        const v4u e0 = __builtin_bit_cast(v4u, d0), e1 = __builtin_bit_cast(v4u, d1);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            db += (bf_lo(e0[k]) + bf_hi(e0[k])) + (bf_lo(e1[k]) + bf_hi(e1[k]));
    }
    unsigned short* in = L == 0 ? S.F : S.A[L > 0 ? L - 1 : 0];
#pragma unroll
    for (int nt = 0; nt < KIN[L] / 32; ++nt) {
        const int m = KIN[L] / 32 * h + nt;
        dw[nt] = mma32(d0, columns<(L > 0 ? ROW : F_ROW)>(in, m, 0, g, r), dw[nt]);
        dw[nt] = mma32(d1, columns<(L > 0 ? ROW : F_ROW)>(in, m, 32, g, r), dw[nt]);
    }
    if (L == 0)
        return;
#pragma unroll
    for (int pt = 0; pt < 2; ++pt) {
        const int p = 32 * h + 16 * pt + r;
        v4f acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
            acc = mma16x2(wt[nb], frag(S.D[cur] + p * ROW + 32 * nb + 8 * g), acc);
        // (sigm of the same value was taken in the forward pass: taken again, not kept)
        uint2 zp = zprev[pt];
        asm volatile("" : "+v"(zp.x), "+v"(zp.y));
        const v4f zf = unpack4(zp);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float s = sigm(zf[i]);
            acc[i] *= s * (1.0f + zf[i] * (1.0f - s));
        }
        put4(S.D[cur ^ 1], p, w, g, acc);
    }
}

// Gradient of the loss over n points.  A workgroup per 64 points that adds its
// 58k weight gradients to memory, one atomic each, is bound by those atomics
// (2^19 points: 4.1 ms, 42 TFLOP/s).  Here a workgroup stays on its CU for every
// n_cu-th tile and writes each gradient once, to its row of `part`: 0.53 ms,
// 325 TFLOP/s, of which the VALU (sigmoids, conversions) is busy over 60% and
// the rest is the eleven barriers of a tile.  Eight waves with twice the
// registers each take 6% longer; weights loaded a layer ahead spill, 3% longer.
// Rounding points: features, pre-activations, activations and deltas in BF16,
// everything else in FP32.  A pre-activation whose FP32 sum moves by an ulp may
// round to the other BF16, and so would 3e-5 of a gradient over 4000 points:
// the products feed 16 inputs at a time (K = 32 MFMAs: 6% less time).
__global__ __launch_bounds__(TW * 128, 4) void k_mlp_train(const v4u* __restrict__ wisw, const v4u* __restrict__ wtsw,
                                                          const float* __restrict__ theta,
                                                          const float* __restrict__ fourier, Frame fr,
                                                          const float* __restrict__ pts,
                                                          const float* __restrict__ dist, uint32_t n, float inv_batch,
                                                          float* __restrict__ part, float* __restrict__ loss_acc)
{
    __shared__ __align__(16) TrainLds S;
    int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int w = wave >> 1, h = wave & 1;
    if (tid < 4 * H)
        S.bias[tid] = theta[OFF_B[tid / H] + (tid % H)];
    else if (tid < 5 * H)
        S.w5[tid - 4 * H] = theta[OFF_W5 + tid - 4 * H];
    const float b5 = theta[OFF_B5];
    const v4f zero{0.0f, 0.0f, 0.0f, 0.0f};
    v4f dw0[2], dw1[4], dw2[4], dw3[4], dw5 = zero;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        dw1[k] = dw2[k] = dw3[k] = zero;
        if (k < 2)
            dw0[k] = zero;
    }
    float db0 = 0.0f, db1 = 0.0f, db2 = 0.0f, db3 = 0.0f, db5 = 0.0f, loss = 0.0f;
    const uint32_t ntiles = (n + TP - 1) / TP;
    for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        // weights are read, and addresses computed, anew for every tile: hoisted
        // out of the loop they would take 150 registers
        uint32_t o0 = 0;
        asm volatile("" : "+s"(o0), "+v"(tid));
        {
            // features: sixteen threads per point, two frequencies each
            const int pl = tid >> 4, f0 = 2 * (tid & 15);
            const uint32_t p = tile * TP + pl;
            const bool valid = p < n;
            const float x = valid ? pts[3 * (size_t)p] : 0.0f, y = valid ? pts[3 * (size_t)p + 1] : 0.0f,
                        z = valid ? pts[3 * (size_t)p + 2] : 0.0f;
            const float xh = (x - fr.cx) * fr.ihx, yh = (y - fr.cy) * fr.ihy, zh = (z - fr.cz) * fr.ihz;
            float sn[2], cs[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int fi = f0 + j;
                const float arg = fourier[o0 + 3 * fi] * xh + fourier[o0 + 3 * fi + 1] * yh + fourier[o0 + 3 * fi + 2] * zh;
                sincosf(arg, &sn[j], &cs[j]);
            }
            const uint32_t s2 = pack_bf16(sn[0], sn[1]), c2 = pack_bf16(cs[0], cs[1]);
            uint32_t* f = reinterpret_cast<uint32_t*>(S.F + pl * F_ROW + 8 * ((f0 & 15) >> 2) + 4 * (f0 >> 4) + (f0 & 3));
            f[0] = s2;
            f[NFREQ / 2] = c2;
        }
        __syncthreads();
        uint2 z0[2], z1[2], z2[2], z3[2];
        train_forward<0>(S, wtsw + o0, w, h, lane, z0);
        __syncthreads();
        train_forward<1>(S, wisw + o0, w, h, lane, z1);
        __syncthreads();
        train_forward<2>(S, wisw + o0, w, h, lane, z2);
        __syncthreads();
        train_forward<3>(S, wisw + o0, w, h, lane, z3);
        asm volatile("" : "+v"(lane));
        const int r = lane & 15, g = lane >> 4;
        // output: this wave's share of w5 . a4 of every point
        const float4 w5 = *reinterpret_cast<const float4*>(S.w5 + 16 * w + 4 * g);
#pragma unroll
        for (int pt = 0; pt < 2; ++pt) {
            const v4f v = unpack4(z3[pt]);
            float s = w5.x * (v[0] * sigm(v[0])) + w5.y * (v[1] * sigm(v[1])) + w5.z * (v[2] * sigm(v[2])) +
                      w5.w * (v[3] * sigm(v[3]));
            s += lane_xor(s, lane, 16);
            s += lane_xor(s, lane, 32);
            if (g == 0)
                S.out[w][32 * h + 16 * pt + r] = s;
        }
        __syncthreads();
        if (wave == 0) { // loss and dL/do of point `lane`
            const uint32_t p = tile * TP + lane;
            float err = 0.0f;
            if (p < n) {
                float o = 0.0f;
#pragma unroll
                for (int k = 0; k < TW; ++k)
                    o += S.out[k][lane];
                o += b5;
                float dn = dist[p] * fr.invD;
                dn = dn < 1.0f ? dn : 1.0f; // +inf (no silhouette) saturates
                err = o - __logf(dn + LOG_EPS);
            }
            // expectile loss w err^2: w = 2 tau when the prediction is below the
            // target, 2 (1 - tau) above it (tau = 0.5: the plain squared error;
            // tau > 0.5 pushes the prediction up, towards an upper bound)
            const float wgt = 2.0f * (err < 0.0f ? fr.tau : 1.0f - fr.tau);
            const float gp = 2.0f * wgt * err * inv_batch;
            S.g[lane] = gp;
            db5 += gp;
            loss += wgt * err * err;
        }
        __syncthreads();
        // output layer gradient and delta4
#pragma unroll
        for (int pt = 0; pt < 2; ++pt) {
            const int p = 32 * h + 16 * pt + r;
            const float gp = S.g[p];
            const v4f v = unpack4(z3[pt]);
            const float wv[4] = {w5.x, w5.y, w5.z, w5.w};
            v4f d;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float s = sigm(v[i]);
                dw5[i] += gp * (v[i] * s);
                d[i] = gp * wv[i] * (s * (1.0f + v[i] * (1.0f - s)));
            }
            put4(S.D[0], p, w, g, d);
        }
        asm volatile("" : "+v"(dw5[0]), "+v"(dw5[1]), "+v"(dw5[2]), "+v"(dw5[3]));
        __syncthreads();
        train_backward<3>(S, wtsw + o0, w, h, lane, z2, dw3, db3);
        __syncthreads();
        train_backward<2>(S, wtsw + o0, w, h, lane, z1, dw2, db2);
        __syncthreads();
        train_backward<1>(S, wtsw + o0, w, h, lane, z0, dw1, db1);
        __syncthreads();
        train_backward<0>(S, wtsw + o0, w, h, lane, z0, dw0, db0);
        // (the sums are done here, not carried over to the next tile)
        asm volatile("" : "+v"(dw5[0]), "+v"(dw5[1]), "+v"(dw5[2]), "+v"(dw5[3]), "+v"(db0), "+v"(db1), "+v"(db2),
                     "+v"(db3));
        __syncthreads(); // the next tile rewrites F
    }
    const int r = lane & 15, g = lane >> 4;
    // this workgroup's gradient: lane (g, r) holds dW rows 16 w + 4 g + i,
    // columns KIN / 2 h + 16 nt + r
    float* out = part + (size_t)blockIdx.x * NPARAM;
    auto put_w = [&](int l, int nt, const v4f& v) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            out[OFF_W[l] + (16 * w + 4 * g + i) * KIN[l] + KIN[l] / 2 * h + 16 * nt + r] = v[i];
    };
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        if (nt < 2)
            put_w(0, nt, dw0[nt]);
        put_w(1, nt, dw1[nt]);
        put_w(2, nt, dw2[nt]);
        put_w(3, nt, dw3[nt]);
    }
    auto put_b = [&](int l, float v) { // lane (g, r): row 16 w + r, the points 8 g .. 8 g + 7 and 32 more
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        if (g == 0)
            out[OFF_B[l] + 16 * w + r] = v;
    };
    if (h == 0) {
        put_b(0, db0);
        put_b(2, db2);
    } else {
        put_b(1, db1);
        put_b(3, db3);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float v = dw5[i];
#pragma unroll
        for (int o = 1; o < 16; o <<= 1)
            v += __shfl_xor(v, o, 64);
        if (r == 0)
            S.out[w][16 * h + 4 * g + i] = v;
    }
    __syncthreads();
    if (h == 0 && lane < 16)
        out[OFF_W5 + 16 * w + lane] = S.out[w][lane] + S.out[w][16 + lane];
    if (wave == 0) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            db5 += __shfl_xor(db5, o, 64);
            loss += __shfl_xor(loss, o, 64);
        }
        if (lane == 0) {
            out[OFF_B5] = db5;
            atomicAdd(loss_acc, loss);
        }
    }
}

// the sum of the workgroups' gradients of parameter i, in order
__device__ __forceinline__ float sum_parts(const float* __restrict__ part, uint32_t nparts, int i)
{
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t b = 0;
    for (; b + 4 <= nparts; b += 4)
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            s[k] += part[(size_t)(b + k) * NPARAM + i];
    for (; b < nparts; ++b)
        s[0] += part[(size_t)b * NPARAM + i];
    return (s[0] + s[1]) + (s[2] + s[3]);
}

__global__ __launch_bounds__(64) void k_mlp_reduce(const float* __restrict__ part, uint32_t nparts,
                                                   float* __restrict__ grad)
{
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i < NPARAM)
        grad[i] = sum_parts(part, nparts, i);
}

// Adam (Kingma & Ba 2015) on the FP32 master weights from the workgroups'
// gradients (nparts = 0: no update); refreshes the BF16 fragments
__global__ __launch_bounds__(64) void k_mlp_adam(float* __restrict__ theta, const float* __restrict__ part,
                                                 uint32_t nparts, float* __restrict__ m1, float* __restrict__ m2,
                                                 unsigned short* __restrict__ wtsw, unsigned short* __restrict__ wisw,
                                                 float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= NPARAM)
        return;
    float th = theta[i];
    if (nparts) {
        const float g = sum_parts(part, nparts, i);
        const float a = b1 * m1[i] + (1.0f - b1) * g;
        const float b = b2 * m2[i] + (1.0f - b2) * g * g;
        m1[i] = a;
        m2[i] = b;
        th -= lr * (a * c1) / (sqrtf(b * c2) + eps);
        theta[i] = th;
    }
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const int K = KIN[l];
        if (i >= OFF_W[l] && i < OFF_W[l] + H * K) {
            const int n = (i - OFF_W[l]) / K, k = (i - OFF_W[l]) % K;
            const unsigned short h = f2bf(th);
            wisw[infer_index(l, n, k)] = h;
            wtsw[l == 0 ? train0_index(n, k) : back_index(l, n, k)] = h;
        }
    }
}

__global__ void k_fill0(float* p, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n)
        p[i] = 0.0f;
}

} // namespace mlpk
} // namespace snch

using namespace snch;
using namespace snch::mlpk;

struct snch_mlp {
    snch_context* ctx = nullptr;
    Frame fr{};
    float D = 1.0f;
    DeviceBuffer theta, grad, m1, m2, wtsw, wisw, fourier, loss;
    DeviceBuffer part; // the workgroups' gradients (training only)
    std::vector<float> h_fourier;
    int step = 0;
};

namespace {

// one workgroup per CU
uint32_t train_workgroups(const snch_mlp* m) { return m->ctx && m->ctx->n_cu > 0 ? (uint32_t)m->ctx->n_cu : 256u; }

uint64_t splitmix(uint64_t& s)
{
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
double u01(uint64_t& s) { return ((splitmix(s) >> 11) + 0.5) * (1.0 / 9007199254740992.0); }

void launch_adam(snch_mlp* m, uint32_t nparts, float lr, float b1, float b2, float eps, float c1, float c2,
                 hipStream_t st)
{
    hipLaunchKernelGGL(k_mlp_adam, dim3((NPARAM + 63) / 64), dim3(64), 0, st, m->theta.as<float>(),
                       m->part.as<float>(), nparts, m->m1.as<float>(), m->m2.as<float>(),
                       m->wtsw.as<unsigned short>(), m->wisw.as<unsigned short>(), lr, b1, b2, eps, c1, c2);
}

// the gradient of the loss over n points (of a batch of weight 1 / inv_batch),
// one row of m->part per workgroup; returns the number of rows
uint32_t launch_train(snch_mlp* m, const float* pts, const float* dist, uint32_t n, float inv_batch, hipStream_t st)
{
    const uint32_t tiles = (n + TP - 1) / TP, wgs = std::min(train_workgroups(m), tiles);
    hipLaunchKernelGGL(k_mlp_train, dim3(wgs), dim3(TW * 128), 0, st, m->wisw.as<v4u>(), m->wtsw.as<v4u>(),
                       m->theta.as<float>(), m->fourier.as<float>(), m->fr, pts, dist, n, inv_batch,
                       m->part.as<float>(), m->loss.as<float>());
    return wgs;
}

int upload_params(snch_mlp* m, const float* params, hipStream_t st)
{
    hipError_t e = hipMemcpyAsync(m->theta.p, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice, st);
    if (e != hipSuccess)
        return hip_fail(e, "snch_mlp: upload");
    launch_adam(m, 0, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, st);
    e = hipStreamSynchronize(st);
    return e == hipSuccess ? SNCH_OK : hip_fail(e, "snch_mlp: refresh");
}

} // namespace

extern "C" {

uint32_t snch_mlp_num_params(void) { return NPARAM; }

int snch_mlp_create(snch_context* ctx, const float* lo, const float* hi, float sigma, uint64_t seed, snch_mlp** out)
{
    if (!ctx || !lo || !hi || !out) {
        set_error("snch_mlp_create: null argument");
        return SNCH_ERR_INVALID;
    }
    hipError_t e = hipSetDevice(ctx->device);
    if (e != hipSuccess)
        return hip_fail(e, "hipSetDevice");
    auto* m = new snch_mlp();
    m->ctx = ctx;
    double d2 = 0.0;
    float c[3], ih[3];
    for (int k = 0; k < 3; ++k) {
        c[k] = 0.5f * (lo[k] + hi[k]);
        const float h = 0.5f * (hi[k] - lo[k]);
        ih[k] = h > 0.0f ? 1.0f / h : 1.0f;
        d2 += (double)(hi[k] - lo[k]) * (hi[k] - lo[k]);
    }
    m->D = (float)std::sqrt(d2);
    m->fr = Frame{c[0], c[1], c[2], ih[0], ih[1], ih[2], 1.0f / m->D, 0.5f};
    // Fourier matrix B ~ N(0, sigma^2) (Box-Muller), and He-uniform weights
    uint64_t s = seed * 0x2545F4914F6CDD1Dull + 1;
    m->h_fourier.resize(3 * NFREQ);
    for (auto& v : m->h_fourier) {
        const double g = std::sqrt(-2.0 * std::log(u01(s))) * std::cos(2.0 * M_PI * u01(s));
        v = (float)(sigma * g);
    }
    std::vector<float> p(NPARAM, 0.0f);
    for (int l = 0; l < 4; ++l) {
        const double a = std::sqrt(6.0 / KIN[l]);
        for (int i = 0; i < H * KIN[l]; ++i)
            p[OFF_W[l] + i] = (float)((2.0 * u01(s) - 1.0) * a);
    }
    for (int i = 0; i < H; ++i)
        p[OFF_W5 + i] = (float)((2.0 * u01(s) - 1.0) * std::sqrt(3.0 / H));
    p[OFF_B5] = -2.0f;
    if ((e = m->theta.ensure(sizeof(float) * NPARAM)) != hipSuccess || (e = m->grad.ensure(sizeof(float) * NPARAM)) ||
        (e = m->m1.ensure(sizeof(float) * NPARAM)) || (e = m->m2.ensure(sizeof(float) * NPARAM)) ||
        (e = m->wtsw.ensure(sizeof(unsigned short) * NSW)) ||
        (e = m->wisw.ensure(sizeof(unsigned short) * NSW)) ||
        (e = m->fourier.ensure(sizeof(float) * 3 * NFREQ)) || (e = m->loss.ensure(sizeof(float) * 4)) ||
        (e = hipMemcpy(m->fourier.p, m->h_fourier.data(), sizeof(float) * 3 * NFREQ, hipMemcpyHostToDevice))) {
        delete m;
        return hip_fail(e, "snch_mlp_create");
    }
    for (DeviceBuffer* b : {&m->grad, &m->m1, &m->m2, &m->loss})
        hipLaunchKernelGGL(k_fill0, dim3((b->bytes / 4 + 255) / 256), dim3(256), 0, 0, b->as<float>(),
                           (int)(b->bytes / 4));
    int rc = upload_params(m, p.data(), 0);
    if (rc != SNCH_OK) {
        delete m;
        return rc;
    }
    *out = m;
    return SNCH_OK;
}

int snch_mlp_destroy(snch_mlp* m)
{
    delete m;
    return SNCH_OK;
}

int snch_mlp_params(snch_mlp* m, float* params_out, const float* params_in, float* fourier_out, float* frame_out)
{
    if (!m) {
        set_error("snch_mlp_params: null model");
        return SNCH_ERR_INVALID;
    }
    if (params_in) {
        int rc = upload_params(m, params_in, 0);
        if (rc != SNCH_OK)
            return rc;
    }
    if (params_out) {
        hipError_t e = hipMemcpy(params_out, m->theta.p, sizeof(float) * NPARAM, hipMemcpyDeviceToHost);
        if (e != hipSuccess)
            return hip_fail(e, "snch_mlp_params");
    }
    if (fourier_out)
        std::memcpy(fourier_out, m->h_fourier.data(), sizeof(float) * 3 * NFREQ);
    if (frame_out) {
        const float f[8] = {m->fr.cx, m->fr.cy, m->fr.cz, m->fr.ihx, m->fr.ihy, m->fr.ihz, m->fr.invD, m->D};
        std::memcpy(frame_out, f, sizeof(f));
    }
    return SNCH_OK;
}

int snch_mlp_set_loss(snch_mlp* m, float tau)
{
    if (!m || !(tau > 0.0f && tau < 1.0f)) {
        set_error("snch_mlp_set_loss: tau must lie in (0, 1)");
        return SNCH_ERR_INVALID;
    }
    m->fr.tau = tau;
    return SNCH_OK;
}

int snch_mlp_gradient(snch_mlp* m, const float* pts, const float* dist, uint32_t n, float* grad_out, float* loss_out,
                      void* stream)
{
    if (!m || !pts || !dist || n == 0) {
        set_error("snch_mlp_gradient: null argument or empty batch");
        return SNCH_ERR_INVALID;
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (const hipError_t a = m->part.ensure(sizeof(float) * NPARAM * train_workgroups(m)))
        return hip_fail(a, "snch_mlp_gradient: allocation");
    hipLaunchKernelGGL(k_fill0, dim3(1), dim3(256), 0, st, m->loss.as<float>(), 4);
    const uint32_t rows = launch_train(m, pts, dist, n, 1.0f / (float)n, st);
    hipLaunchKernelGGL(k_mlp_reduce, dim3((NPARAM + 63) / 64), dim3(64), 0, st, m->part.as<float>(), rows,
                       m->grad.as<float>());
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && grad_out)
        e = hipMemcpyAsync(grad_out, m->grad.p, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, st);
    float l = 0.0f;
    if (e == hipSuccess)
        e = hipMemcpyAsync(&l, m->loss.p, sizeof(float), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess)
        e = hipStreamSynchronize(st);
    if (e != hipSuccess)
        return hip_fail(e, "snch_mlp_gradient");
    if (loss_out)
        *loss_out = l / (float)n;
    return SNCH_OK;
}

int snch_mlp_train(snch_mlp* m, const float* pts, const float* dist, uint32_t n, uint32_t batch, uint32_t epochs,
                   float lr, float* epoch_loss, void* stream)
{
    if (!m || !pts || !dist || n == 0 || batch == 0 || batch % TP != 0) {
        set_error("snch_mlp_train: null argument, empty data or batch not a multiple of 64");
        return SNCH_ERR_INVALID;
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (const hipError_t a = m->part.ensure(sizeof(float) * NPARAM * train_workgroups(m)))
        return hip_fail(a, "snch_mlp_train: allocation");
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (uint32_t ep = 0; ep < epochs; ++ep) {
        hipLaunchKernelGGL(k_fill0, dim3(1), dim3(256), 0, st, m->loss.as<float>(), 4);
        for (uint32_t off = 0; off < n; off += batch) {
            const uint32_t nb = n - off < batch ? n - off : batch;
            const uint32_t rows = launch_train(m, pts + 3 * (size_t)off, dist + off, nb, 1.0f / (float)nb, st);
            ++m->step;
            const float c1 = 1.0f / (1.0f - std::pow(b1, (float)m->step));
            const float c2 = 1.0f / (1.0f - std::pow(b2, (float)m->step));
            launch_adam(m, rows, lr, b1, b2, eps, c1, c2, st);
        }
        float l = 0.0f;
        hipError_t e = hipGetLastError();
        if (e == hipSuccess)
            e = hipMemcpyAsync(&l, m->loss.p, sizeof(float), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess)
            e = hipStreamSynchronize(st);
        if (e != hipSuccess)
            return hip_fail(e, "snch_mlp_train");
        if (epoch_loss)
            epoch_loss[ep] = l / (float)n;
    }
    return SNCH_OK;
}

int snch_mlp_predict(snch_mlp* m, const float* pts, uint32_t n, int mode, float rel, float absm, float* out,
                     void* stream)
{
    if (!m || (n && (!pts || !out))) {
        set_error("snch_mlp_predict: null argument");
        return SNCH_ERR_INVALID;
    }
    if (n == 0)
        return SNCH_OK;
    constexpr int NW = MLP_INFER_WAVES, P = MLP_INFER_TILES;
    const uint32_t groups = (n + 16 * NW * P - 1) / (16 * NW * P);
    const uint32_t grid = groups < 2048 ? groups : 2048;
    hipLaunchKernelGGL((k_mlp_infer<NW, P>), dim3(grid), dim3(NW * 64), 0, static_cast<hipStream_t>(stream),
                       m->wisw.as<v4u>(), m->theta.as<float>(), m->fourier.as<float>(), m->fr, pts, n, mode, rel, absm,
                       m->D, out);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? SNCH_OK : hip_fail(e, "snch_mlp_predict");
}

} // extern "C"
