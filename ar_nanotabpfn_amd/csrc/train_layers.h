// The transformer layers of a training step around the row attention, forward and backward (gfx950;
// float32 parameters and residual stream, bfloat16 products with float32 sums: what autocast computes).
//
// A step of the reference's training configuration touches 38912 rows of width 128 twelve times over; every
// layer is five small products per row.  As library calls that is 1300 launches with a cast, a bias, a norm
// or a copy of 20 MB between any two products, and weight gradients whose 128 x 128 outputs leave most of
// the chip idle.  Here a layer is: forward one kernel and the attention call, backward one kernel and the
// attention's backward call, one split product for all weight gradients, one reduction.  They are bound by
// memory: each reads and writes the residual stream and what the weight gradients need once.
//
//   forward    behind the attention   r2 = x1 + attn W_o^T; x2 = LN2(r2); u = x2 W_1^T + b_1; r3 = x2 + gelu(u) W_2^T + b_2
//              in front of the next   x = LN3(r3); r1 = x + x W_fo^T; x1 = LN1(r1); qkv = x1 W_qkv^T
//   backward   d(qkv) -> dr1, d(x) | d(x) of the layer before -> dr3, du (u is recomputed), dr2, d(attn)
// with W_fo = out_proj v_proj of the single-column feature attention (one key per query: the softmax weight
// is 1); dW_out = dW_fo W_v^T and dW_v = W_out^T dW_fo follow from its gradient.  Of every LayerNorm the sum
// in front of it and (mean, 1/std) are kept; its output is recomputed where it is read.
//
// Tiles.  A workgroup of four wavefronts owns 32 rows and all columns; products are transposed as in
// fused_layer.h (C^T[n, m] = sum_k W[n, k] A[m, k], v_mfma_f32_16x16x32): a lane holds, for two token rows
// (lane % 16 and + 16), four consecutive features 4 (lane / 16) + r of every 16-feature block.  Small
// workgroups, so that the loads of one run under the products of others: four to a compute unit forward, three backward
// at d_model 128; three and two at 256.
//
// 38912 rows of 128: forward 45 us a layer (its bytes at the rate of a copy 25), backward 72 us (50).  The rest is the
// weights, 295 and 360 KB a tile from L2 (with one cached fragment for all of them 32 and 59 us), and that the few tiles
// of a compute unit (4.75) load, multiply and store nearly in step; with neither stores nor memory behind the loads 19 and
// 34.  Measured and not kept (forward): five workgroups to a compute unit (spills).
#pragma once

#include "common.h"
#include "fused_layer.h"
#include "mfma_flash.h"

namespace artab {

constexpr int kTrainWaves = 4, kTrainRows = 32;
constexpr int kTrainPackLayers = 16;   // layers per launch of the weight kernels
constexpr int kTrainMaxJobs = 32;      // 128 x 128 pieces of a layer's weight gradients

// packed bf16 matrices of a layer, in this order; T: the transposed matrix
enum TrainMatrix : int { kTmFo, kTmFoT, kTmQkv, kTmQkvT, kTmO, kTmOT, kTm1, kTm1T, kTm2, kTm2T, kTmCount };
template <int D, int F>
__host__ __device__ constexpr long train_matrix_at(int m) {  // element offset inside a layer's packed weights
    constexpr long size[kTmCount] = {D * D, D * D, 3 * D * D, 3 * D * D, D * D, D * D, D * F, D * F, D * F, D * F};
    long at = 0;
    for (int i = 0; i < m; ++i) at += size[i];
    return at;
}
template <int D, int F>
constexpr long train_packed_elems() { return train_matrix_at<D, F>(kTmCount); }

struct TrainWeights {  // float32 masters of up to kTrainPackLayers layers, row-major
    const float *v[kTrainPackLayers], *out[kTrainPackLayers];              // feature attention [D, D]
    const float *q[kTrainPackLayers], *k[kTrainPackLayers], *vr[kTrainPackLayers], *o[kTrainPackLayers];
    const float *w1[kTrainPackLayers], *w2[kTrainPackLayers];              // [F, D], [D, F]
};

// fo[layer] = out v: 16 rows of one layer per workgroup
template <int D>
__global__ __launch_bounds__(D) void train_fold_kernel(TrainWeights W, float *fo) {
    __shared__ float out_s[16][D];
    const int layer = blockIdx.y, n0 = 16 * blockIdx.x, k = threadIdx.x;
    const float *out = W.out[layer], *v = W.v[layer];
#pragma unroll
    for (int n = 0; n < 16; ++n) out_s[n][k] = out[(n0 + n) * D + k];
    __syncthreads();
    float acc[16];
#pragma unroll
    for (int n = 0; n < 16; ++n) acc[n] = 0.f;
#pragma unroll 16  // (as many loads on their way: few wavefronts, one after the other)
    for (int j = 0; j < D; ++j) {
        const float x = v[j * D + k];
#pragma unroll
        for (int n = 0; n < 16; ++n) acc[n] = fmaf(out_s[n][j], x, acc[n]);
    }
#pragma unroll
    for (int n = 0; n < 16; ++n) fo[(static_cast<long>(layer) * D + n0 + n) * D + k] = acc[n];
}

// dout[n][j] = sum_k dfo[n][k] v[j][k];  dv[j][k] = sum_n out[n][j] dfo[n][k].  16 rows per workgroup.
template <int D>
__global__ __launch_bounds__(D) void train_unfold_kernel(TrainWeights W, float *grads, long layer_stride, long at_fo, long at_out,
                                                         long at_v) {
    __shared__ float a_s[16][D + 1];
    const int layer = blockIdx.y, r0 = 16 * (blockIdx.x % (D / 16)), c = threadIdx.x;
    const bool for_v = blockIdx.x >= D / 16;
    float *g = grads + layer * layer_stride;
    const float *dfo = g + at_fo;
    float acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    if (!for_v) {
#pragma unroll
        for (int i = 0; i < 16; ++i) a_s[i][c] = dfo[(r0 + i) * D + c];
        __syncthreads();
        const f32x4 *row = reinterpret_cast<const f32x4 *>(W.v[layer] + static_cast<long>(c) * D);
#pragma unroll 8
        for (int k = 0; k < D / 4; ++k) {
            const f32x4 x = row[k];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = fmaf(a_s[i][4 * k + e], x[e], acc[i]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) a_s[i][c] = W.out[layer][static_cast<long>(c) * D + r0 + i];
        __syncthreads();
#pragma unroll 16
        for (int n = 0; n < D; ++n) {
            const float x = dfo[n * D + c];
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] = fmaf(a_s[i][n], x, acc[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) g[(for_v ? at_v : at_out) + (r0 + i) * D + c] = acc[i];
}

// Every matrix of a layer as bf16 operand fragments: fragment (nb, ks) of W [N, K] is 1 KiB, lane l holds
// W[16 nb + l % 16][32 ks + 8 (l / 16) ..].  One 16-byte piece per thread.
template <int D, int F>
__global__ __launch_bounds__(256) void train_pack_kernel(TrainWeights W, const float *fo, bf16_t *packed) {
    const int layer = blockIdx.y;
    const long piece = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (piece * 8 >= train_packed_elems<D, F>()) return;
    int m = 0;
    while (m + 1 < kTmCount && piece * 8 >= train_matrix_at<D, F>(m + 1)) ++m;
    const long in = piece - train_matrix_at<D, F>(m) / 8;
    const bool t = m & 1;
    int N, K;  // of the matrix as it is packed
    switch (m & ~1) {
        case kTmQkv: N = 3 * D; K = D; break;
        case kTm1: N = F; K = D; break;
        case kTm2: N = D; K = F; break;
        default: N = K = D; break;
    }
    if (t) { const int x = N; N = K; K = x; }
    const int lane = static_cast<int>(in & 63), frag = static_cast<int>(in >> 6), ks = frag % (K / 32), nb = frag / (K / 32);
    const int n = 16 * nb + (lane & 15), k0 = 32 * ks + 8 * (lane >> 4);
    const float *src;
    switch (m & ~1) {
        case kTmFo: src = fo + static_cast<long>(layer) * D * D; break;
        case kTmQkv: src = nullptr; break;
        case kTmO: src = W.o[layer]; break;
        case kTm1: src = W.w1[layer]; break;
        default: src = W.w2[layer]; break;
    }
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int row = t ? k0 + e : n, col = t ? n : k0 + e, width = t ? N : K;  // element [row][col] of the master
        if ((m & ~1) == kTmQkv) {
            const float *part = row < D ? W.q[layer] : row < 2 * D ? W.k[layer] : W.vr[layer];
            f[e] = part[static_cast<long>(row % D) * D + col];
        } else {
            f[e] = src[static_cast<long>(row) * width + col];
        }
    }
    const u32x4 v = {pack2<bf16_t>(f[0], f[1]), pack2<bf16_t>(f[2], f[3]), pack2<bf16_t>(f[4], f[5]), pack2<bf16_t>(f[6], f[7])};
    reinterpret_cast<u32x4 *>(packed + static_cast<long>(layer) * train_packed_elems<D, F>())[piece] = v;
}

// ---- tiles

template <int NB>
using TrainAcc = f32x4[NB][2];  // [16-feature block][token half]

// A pointer again, as one the compiler cannot trace: in a loop over tiles it would otherwise take the weights,
// which are the same for every tile, as something to keep in registers.
__device__ __forceinline__ const bf16_t *train_opaque(const bf16_t *p) {
    asm volatile("" : "+s"(p));
    return p;
}

// Global memory at a wavefront-uniform address and a lane's 32-bit byte offset, in global memory's own address space: a
// pointer the compiler cannot trace would be a generic one, whose loads count as LDS accesses too, and every wait for an
// activation in LDS would wait for the weights behind it; and the addition is the load's own, not two vector instructions
// in front of it.
template <typename V>
__device__ __forceinline__ V train_get(const void *base, unsigned byte) {
    typedef const __attribute__((address_space(1))) char *Global;
    return *(const __attribute__((address_space(1))) V *)((Global)base + byte);
}
template <typename V>
__device__ __forceinline__ void train_put(void *base, unsigned byte, const V &v) {
    typedef __attribute__((address_space(1))) char *Global;
    *(__attribute__((address_space(1))) V *)((Global)base + byte) = v;
}

typedef float TrainStat __attribute__((ext_vector_type(2)));  // (mean, 1/std) of a row

struct TrainLane {
    int wave, lane, tok, quad;
    long row0;
    int last;  // of the tile's rows
    __device__ __forceinline__ TrainLane(long tile, long M) {
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        lane = opaque(threadIdx.x & 63);
        tok = lane & 15;
        quad = lane >> 4;
        row0 = tile * kTrainRows;
        last = static_cast<int>(min(static_cast<long>(kTrainRows), M - row0)) - 1;
    }
    // of token half tb: its row in the tile (past the end the last one again) and whether it is one
    __device__ __forceinline__ int in(int tb) const { return min(16 * tb + tok, last); }
    __device__ __forceinline__ bool live(int tb) const { return 16 * tb + tok <= last; }
    __device__ __forceinline__ int col(int b) const { return 16 * (wave + kTrainWaves * b) + 4 * quad; }
};

template <int D, int NB>
__device__ __forceinline__ void train_load(f32x4 (&v)[NB][2], const float *src, const TrainLane &L) {
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int b = 0; b < NB; ++b) v[b][tb] = train_get<f32x4>(src + L.row0 * D, 4u * (L.in(tb) * D + L.col(b)));
}
template <int D, int NB>
__device__ __forceinline__ void train_store(float *dst, const f32x4 (&v)[NB][2], const TrainLane &L) {
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
        if (L.live(tb)) {
#pragma unroll
            for (int b = 0; b < NB; ++b) train_put(dst + L.row0 * D, 4u * (L.in(tb) * D + L.col(b)), v[b][tb]);
        }
}
// Values rounded for a store later on.
template <int NB>
struct TrainPacked {
    u32x2 v[NB][2];
    __device__ __forceinline__ explicit TrainPacked(const f32x4 (&x)[NB][2]) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) v[b][tb] = u32x2{pack2<bf16_t>(x[b][tb][0], x[b][tb][1]), pack2<bf16_t>(x[b][tb][2], x[b][tb][3])};
    }
    // (row stride LDG)
    template <int LDG>
    __device__ __forceinline__ void store(bf16_t *dst, int col0, const TrainLane &L) const {
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
            if (L.live(tb)) {
#pragma unroll
                for (int b = 0; b < NB; ++b) train_put(dst + L.row0 * LDG + col0, 2u * (L.in(tb) * LDG + L.col(b)), v[b][tb]);
            }
    }
};
template <int NB>
__device__ __forceinline__ void train_to_lds(bf16_t *tile, int ld, const f32x4 (&v)[NB][2], const TrainLane &L) {
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int b = 0; b < NB; ++b)
            store4f<bf16_t>(tile + (16 * tb + L.tok) * ld + L.col(b), v[b][tb][0], v[b][tb][1], v[b][tb][2], v[b][tb][3]);
}
// [32, W] bf16 between global memory (row stride W) and an LDS tile (row stride lds_ld), 16 bytes a lane
template <int W>
__device__ __forceinline__ void train_stage(bf16_t *tile, int lds_ld, const bf16_t *src, const TrainLane &L) {
    constexpr int CPR = W / 8;
    static_assert(kTrainRows * CPR % (kTrainWaves * 64) == 0, "whole passes");
    const int tid = opaque(threadIdx.x);
#pragma unroll
    for (int x = 0; x < kTrainRows * CPR / (kTrainWaves * 64); ++x) {
        const int i = tid + kTrainWaves * 64 * x, r = i / CPR, c = i % CPR;
        *reinterpret_cast<u32x4 *>(tile + r * lds_ld + 8 * c) = train_get<u32x4>(src + L.row0 * W, 2u * (min(r, L.last) * W + 8 * c));
    }
}
template <int W>
__device__ __forceinline__ void train_unstage(bf16_t *dst, const bf16_t *tile, int lds_ld, const TrainLane &L) {
    constexpr int CPR = W / 8;
    static_assert(kTrainRows * CPR % (kTrainWaves * 64) == 0, "whole passes");
    const int tid = opaque(threadIdx.x);
#pragma unroll
    for (int x = 0; x < kTrainRows * CPR / (kTrainWaves * 64); ++x) {
        const int i = tid + kTrainWaves * 64 * x, r = i / CPR, c = i % CPR;
        if (r <= L.last) train_put(dst + L.row0 * W, 2u * (r * W + 8 * c), *reinterpret_cast<const u32x4 *>(tile + r * lds_ld + 8 * c));
    }
}

// acc[b][tb] = sum_k W[16 (nb0 + wave + 4 b) ..][k] A[16 tb + tok][k].  A ring of eight weight fragments is on its way ahead of
// the one being multiplied; begin() requests the first.
//
// Order of requests.  A wavefront's loads and stores are counted together and in order: a wait for a load is a wait for
// every store in front of it, and their way to memory is longer than a product.  So the next product's first fragments, and
// the tensors it needs, are asked for before the results of the one behind are stored, and the parameter vectors lie in
// LDS.  38912 rows of 128, stores in front of the requests / behind them: forward 50.8 / 44.8 us, the last layer's
// backward 50.7 / 47.2, the others' 73.2 / 71.8 (without any stores 35.1, 32.4 and 50.8).
struct TrainRing {
    u32x4 f[8];
    template <int NB, int KS>
    static constexpr int ahead() { return 8 / NB < KS ? 8 / NB : KS; }  // contraction steps in the ring
    static __device__ __forceinline__ u32x4 get(const bf16_t *w, int nb0, int b, int ks, int steps, const TrainLane &L) {
        return train_get<u32x4>(reinterpret_cast<const char *>(w) + ((nb0 + L.wave + kTrainWaves * b) * static_cast<long>(steps) + ks) * 1024,
                                16u * L.lane);
    }
    template <int NB, int KS>
    __device__ __forceinline__ void begin(const bf16_t *w, int nb0, const TrainLane &L) {
#pragma unroll
        for (int p = 0; p < ahead<NB, KS>(); ++p)
#pragma unroll
            for (int b = 0; b < NB; ++b) f[p * NB + b] = get(w, nb0, b, p, KS, L);
    }
    template <int NB, int KS>
    __device__ __forceinline__ void run(f32x4 (&acc)[NB][2], const bf16_t *tile, int ld, const bf16_t *w, int nb0, const TrainLane &L) {
        typedef MfmaOps<bf16_t> Ops;
        constexpr int PF = ahead<NB, KS>();
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) acc[b][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
        const bf16_t *const a = tile + L.tok * ld + 8 * L.quad;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const bf16x8 a0 = *reinterpret_cast<const bf16x8 *>(a + 32 * ks), a1 = *reinterpret_cast<const bf16x8 *>(a + 16 * ld + 32 * ks);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                u32x4 &slot = f[ks % PF * NB + b];
                const bf16x8 wv = __builtin_bit_cast(bf16x8, slot);
                acc[b][0] = Ops::mma16(wv, a0, acc[b][0]);
                acc[b][1] = Ops::mma16(wv, a1, acc[b][1]);
                if (ks + PF < KS) slot = get(w, nb0, b, ks + PF, KS, L);
            }
        }
    }
};
template <int NB, int KS>
__device__ __forceinline__ void train_product(f32x4 (&acc)[NB][2], const bf16_t *tile, int ld, const bf16_t *w, int nb0, const TrainLane &L) {
    TrainRing ring;
    ring.begin<NB, KS>(w, nb0, L);
    ring.run<NB, KS>(acc, tile, ld, w, nb0, L);
}

// A parameter vector: in LDS where a kernel keeps it there, else in memory.  N floats by the lanes of one wavefront.
template <bool LDS>
struct TrainVector {
    const float *p;
    __device__ __forceinline__ f32x4 at(int col) const {
        if constexpr (LDS) return *reinterpret_cast<const f32x4 *>(p + col);
        else return train_get<f32x4>(p, 4u * col);
    }
};
template <int N>
__device__ __forceinline__ void train_keep(float *lds, const float *src, int wave) {
    static_assert(N <= 256 && N % 4 == 0, "one request of a wavefront");
    const int i = 4 * static_cast<int>(threadIdx.x & 63);
    if (static_cast<int>(threadIdx.x >> 6) == wave && i < N) *reinterpret_cast<f32x4 *>(lds + i) = train_get<f32x4>(src, 4u * i);
}

// Sums of two per-row values over all features: lanes, then wavefronts.  red: [4][32] float2.
struct TrainPair {
    float a, b;
};
__device__ __forceinline__ void train_row_sums(TrainPair (&s)[2], float2 *red, const TrainLane &L) {
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
        s[tb].a = row_sum(s[tb].a);
        s[tb].b = row_sum(s[tb].b);
        if (L.quad == 0) red[L.wave * kTrainRows + 16 * tb + L.tok] = make_float2(s[tb].a, s[tb].b);
    }
    __syncthreads();
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
        float2 p[kTrainWaves];
#pragma unroll
        for (int w = 0; w < kTrainWaves; ++w) p[w] = red[w * kTrainRows + 16 * tb + L.tok];
        s[tb].a = (p[0].x + p[1].x) + (p[2].x + p[3].x);
        s[tb].b = (p[0].y + p[1].y) + (p[2].y + p[3].y);
    }
}

// (mean, 1/std) of the rows of v, kept in `stats`; one barrier inside.  The wavefronts' means and squared
// deviations are combined pairwise (Chan et al.).
template <int D, int NB>
__device__ __forceinline__ void train_stats(const f32x4 (&v)[NB][2], float2 *red, float eps, float2 *stats, float2 (&st)[2], const TrainLane &L) {
    constexpr float kLocal = NB * 16;
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
        float s = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b) s += (v[b][tb][0] + v[b][tb][1]) + (v[b][tb][2] + v[b][tb][3]);
        const float mean = row_sum(s) * (1.f / kLocal);
        float q = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float d = v[b][tb][e] - mean;
                q = fmaf(d, d, q);
            }
        q = row_sum(q);
        if (L.quad == 0) red[L.wave * kTrainRows + 16 * tb + L.tok] = make_float2(mean, q);
    }
    __syncthreads();
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
        float2 p[kTrainWaves];
#pragma unroll
        for (int w = 0; w < kTrainWaves; ++w) p[w] = red[w * kTrainRows + 16 * tb + L.tok];
        const float mean = ((p[0].x + p[1].x) + (p[2].x + p[3].x)) * (1.f / kTrainWaves);
        float m2 = 0.f;
#pragma unroll
        for (int w = 0; w < kTrainWaves; ++w) {
            const float d = p[w].x - mean;
            m2 += fmaf(kLocal * d, d, p[w].y);
        }
        st[tb] = make_float2(mean, rsqrtf(m2 / D + eps));
        if (L.wave == 0 && L.quad == 0 && L.live(tb)) train_put(stats + L.row0, 8u * L.in(tb), TrainStat{st[tb].x, st[tb].y});
    }
}
__device__ __forceinline__ void train_get_stats(float2 (&st)[2], const float2 *stats, const TrainLane &L) {
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
        const TrainStat v = train_get<TrainStat>(stats + L.row0, 8u * L.in(tb));
        st[tb] = make_float2(v[0], v[1]);
    }
}
// x = (r - mean) / std * g + b
template <int NB, bool LDS>
__device__ __forceinline__ void train_norm(f32x4 (&x)[NB][2], const f32x4 (&r)[NB][2], const float2 (&st)[2], const TrainVector<LDS> &g, const TrainVector<LDS> &be,
                                           const TrainLane &L) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const f32x4 gv = g.at(L.col(b)), bv = be.at(L.col(b));
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[b][tb][e] = fmaf((r[b][tb][e] - st[tb].x) * st[tb].y, gv[e], bv[e]);
    }
}

// h = gelu(u) and its derivative, in float32: erf by the rational form 7.1.26 of Abramowitz and Stegun, which shares
// its exponential with the derivative.  Its absolute error is below 1.5e-7; both results are rounded to bf16, of
// whose unit in the last place that is a hundredth for u above -3 and a quarter at -4.5, where h is 1.5e-5.  On
// normal u the rounded results are as far from float64 as with erff (1.66620e-3 and 1.91314e-3 of their norms).  With
// normal_tail() instead a training step of 38912 rows and 12 layers takes 4.23 ms, 4.19 with this.
__device__ __forceinline__ void train_gelu(float u, float &h, float &dh) {
    const float z = fabsf(u) * 0.70710678118654752f, e = fast_exp2(-z * z * kLog2e);
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, z, 1.f));
    const float poly = t * fmaf(t, fmaf(t, fmaf(t, fmaf(t, 1.061405429f, -1.453152027f), 1.421413741f), -0.284496736f), 0.254829592f);
    const float cdf = fmaf(0.5f, copysignf(fmaf(-poly, e, 1.f), u), 0.5f);
    h = u * cdf;
    dh = fmaf(u * 0.39894228040143268f, e, cdf);
}

// What follows the attention of a layer, and what leads to the attention of the next: the stream between the two
// stays in registers.
struct TrainForward {
    // behind the attention (BACK)
    const bf16_t *attn;        // [M, D]
    const float *r1; const float2 *stats1;
    const float *g1, *b1;
    const float *g2, *b2, *bias1, *bias2;
    float eps2, eps3;
    float *r2; float2 *stats2;
    float *r3; float2 *stats3;
    const bf16_t *packed;
    // in front of the next (FRONT)
    const float *x;            // without BACK: its input
    const float *g3, *b3;      // with BACK: the norm between the two
    const float *next_g1, *next_b1;
    float next_eps1;
    float *next_r1; float2 *next_stats1;
    bf16_t *next_qkv;          // [M, 3 D]
    const bf16_t *next_packed;
    long M;
};

template <int D, int F, bool BACK, bool FRONT>
__global__ __launch_bounds__(kTrainWaves * 64, D == 128 ? 4 : 3) void train_forward_kernel(TrainForward P) {
    constexpr int NB = D / 64, NF = F / 64, LD = D + 8, LF = F + 8;
    __shared__ __attribute__((aligned(16))) bf16_t as[kTrainRows * (LD > LF || !BACK ? LD : LF)], ys[kTrainRows * LD];
    __shared__ float2 red[kTrainWaves * kTrainRows];
    __shared__ __attribute__((aligned(16))) float vecs[(BACK ? 5 * D + F : 0) + (FRONT ? 2 * D : 0)];
    float *const vec1 = vecs + (BACK ? 5 * D + F : 0);  // of the next layer's norm
    typedef TrainVector<true> Kept;
    const TrainLane L(blockIdx.x, P.M);
    TrainRing ring;
    f32x4 x[NB][2], acc[NB][2];
    float2 st[2];
    const bf16_t *const w_o = P.packed + train_matrix_at<D, F>(kTmO), *const w_1 = P.packed + train_matrix_at<D, F>(kTm1),
                 *const w_2 = P.packed + train_matrix_at<D, F>(kTm2), *const w_fo = P.next_packed + train_matrix_at<D, F>(kTmFo),
                 *const w_qkv = P.next_packed + train_matrix_at<D, F>(kTmQkv);
    if constexpr (BACK) {
        ring.begin<NB, D / 32>(w_o, 0, L);
        train_stage<D>(as, LD, P.attn, L);
        train_load<D>(x, P.r1, L);
        train_get_stats(st, P.stats1, L);
        train_keep<D>(vecs, P.g2, 0);
        train_keep<D>(vecs + D, P.b2, 1);
        train_keep<D>(vecs + 2 * D, P.bias2, 2);
        train_keep<F>(vecs + 5 * D, P.bias1, 3);
        if constexpr (FRONT) {
            train_keep<D>(vecs + 3 * D, P.g3, 0);
            train_keep<D>(vecs + 4 * D, P.b3, 1);
            train_keep<D>(vec1, P.next_g1, 2);
            train_keep<D>(vec1 + D, P.next_b1, 3);
        }
        train_norm(x, x, st, TrainVector<false>{P.g1}, TrainVector<false>{P.b1}, L);
        __syncthreads();
        ring.run<NB, D / 32>(acc, as, LD, w_o, 0, L);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) x[b][tb] += acc[b][tb];
        ring.begin<NF, D / 32>(w_1, 0, L);
        train_store<D>(P.r2, x, L);
        train_stats<D>(x, red, P.eps2, P.stats2, st, L);
        train_norm(x, x, st, Kept{vecs}, Kept{vecs + D}, L);
        train_to_lds(ys, LD, x, L);
        __syncthreads();
        {
            f32x4 u[NF][2];
            ring.run<NF, D / 32>(u, ys, LD, w_1, 0, L);
            ring.begin<NB, F / 32>(w_2, 0, L);
#pragma unroll
            for (int b = 0; b < NF; ++b) {
                const f32x4 bias = Kept{vecs + 5 * D}.at(L.col(b));
#pragma unroll
                for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float h, dh;
                        train_gelu(u[b][tb][e] + bias[e], h, dh);
                        u[b][tb][e] = h;
                    }
            }
            train_to_lds(as, LF, u, L);
        }
        __syncthreads();
        ring.run<NB, F / 32>(acc, as, LF, w_2, 0, L);
        if constexpr (FRONT) ring.begin<NB, D / 32>(w_fo, 0, L);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const f32x4 bias = Kept{vecs + 2 * D}.at(L.col(b));
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) x[b][tb] += acc[b][tb] + bias;
        }
        train_store<D>(P.r3, x, L);
        train_stats<D>(x, red, P.eps3, P.stats3, st, L);  // (its barrier: nobody reads the tiles any more)
        if constexpr (FRONT) train_norm(x, x, st, Kept{vecs + 3 * D}, Kept{vecs + 4 * D}, L);
    } else {
        ring.begin<NB, D / 32>(w_fo, 0, L);
        train_load<D>(x, P.x, L);
        train_keep<D>(vec1, P.next_g1, 2);
        train_keep<D>(vec1 + D, P.next_b1, 3);
    }
    if constexpr (FRONT) {
        const TrainLane L(blockIdx.x, P.M);
        train_to_lds(as, LD, x, L);
        __syncthreads();
        ring.run<NB, D / 32>(acc, as, LD, w_fo, 0, L);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) acc[b][tb] += x[b][tb];
        ring.begin<NB, D / 32>(w_qkv, 0, L);
        train_store<D>(P.next_r1, acc, L);
        train_stats<D>(acc, red, P.next_eps1, P.next_stats1, st, L);
        train_norm(acc, acc, st, Kept{vec1}, Kept{vec1 + D}, L);
        train_to_lds(ys, LD, acc, L);
        __syncthreads();
#pragma unroll
        for (int part = 0; part < 3; ++part) {
            ring.run<NB, D / 32>(acc, ys, LD, w_qkv, part * (D / 16), L);
            if (part < 2) ring.begin<NB, D / 32>(w_qkv, (part + 1) * (D / 16), L);
            TrainPacked<NB>(acc).template store<3 * D>(P.next_qkv, part * D, L);
        }
    }
}

// ---- backward

// Column sums over the token rows of this workgroup's tiles, in LDS: every column belongs to one lane group.
__device__ __forceinline__ void train_col_add(float *sums, const f32x4 &s, int col, const TrainLane &L) {
    f32x4 t = s;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float x = t[e];
        x += row_rotate<8>(x);
        x += row_rotate<4>(x);
        x += row_rotate<2>(x);
        x += row_rotate<1>(x);
        t[e] = x;
    }
    if (L.tok == 0) *reinterpret_cast<f32x4 *>(sums + col) += t;
}

// d(sum in front of a norm) from d(its output); column sums of the parameters' gradients.  Rows past the end
// contribute nothing.  One barrier inside.
template <int D, int NB, bool LDS>
__device__ __forceinline__ void train_norm_backward(f32x4 (&d)[NB][2], const f32x4 (&r)[NB][2], const float2 (&st)[2], const TrainVector<LDS> &g,
                                                    float *sum_g, float *sum_b, float2 *red, const TrainLane &L) {
    TrainPair s[2] = {{0.f, 0.f}, {0.f, 0.f}};
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const f32x4 gv = g.at(L.col(b));
        f32x4 cg = {0.f, 0.f, 0.f, 0.f}, cb = cg;
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            if (!L.live(tb)) d[b][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float xh = (r[b][tb][e] - st[tb].x) * st[tb].y, dy = d[b][tb][e];
                cg[e] = fmaf(dy, xh, cg[e]);
                cb[e] += dy;
                const float gy = dy * gv[e];
                s[tb].a += gy;
                s[tb].b = fmaf(gy, xh, s[tb].b);
                d[b][tb][e] = gy;
            }
        }
        train_col_add(sum_g, cg, L.col(b), L);
        train_col_add(sum_b, cb, L.col(b), L);
    }
    train_row_sums(s, red, L);
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
        const float m1 = s[tb].a * (1.f / D), m2 = s[tb].b * (1.f / D);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float xh = (r[b][tb][e] - st[tb].x) * st[tb].y;
                d[b][tb][e] = st[tb].y * (d[b][tb][e] - m1 - xh * m2);
            }
    }
}

// The front of a layer backward (FRONT), then the back of the layer before it (BACK): the gradient between the two
// stays in registers, and the sum in front of the norm between them is read once.
struct TrainBackward {
    // the layer whose d(qkv) is known
    const bf16_t *dqkv;        // [M, 3 D]
    const float *r1; const float2 *stats1; const float *g1, *b1;
    const bf16_t *packed;
    bf16_t *x1, *d1, *x;       // [M, D] each
    // between the two: the sum in front of the norm of the layer before (its output is this layer's input), or,
    // without BACK, the input itself
    const float *r3; const float2 *stats3; const float *g3, *b3;
    float *dx;                 // [M, D]: without FRONT the gradient of the layer's output, without BACK that of the input
    // the layer before
    const float *r2; const float2 *stats2; const float *g2, *b2;
    const float *bias1;
    const bf16_t *back_packed;
    bf16_t *d3, *x2, *h, *du, *d2, *dattn;  // [M, D], [M, D], [M, F], [M, F], [M, D], [M, D]
    float *dr2;                // [M, D]: gradient of x1 along the residual: of the later layer, then of the one before
    float *part;               // [gridDim.x][7 D + F]: column sums g3, b3, bias2, g2, b2 (D each), bias1 (F); g1, b1
    long M;
};

// (d_model 128: held to 168 registers, three workgroups to a compute unit.  For that the feed-forward goes in two halves
// and lane indices are taken anew in each part, or some 40 addresses would be kept over the loop: two workgroups
// of 256 registers took 90 us, three of them 83, every resident one started 74.)
template <int D, int F, bool FRONT, bool BACK>
__global__ __launch_bounds__(kTrainWaves * 64, D == 128 ? 3 : 2) void train_backward_kernel(TrainBackward P) {
    constexpr int NB = D / 64, LD = D + 8, LQ = 3 * D + 8, LF = F + 8, NS = 7 * D + F;
    constexpr int kWide = FRONT && LQ > LD + LF ? LQ : LD + LF;  // d(qkv) lies where x2 and d(u) do later
    constexpr bool kKept = D == 128;  // the parameter vectors in LDS (256: two workgroups to a compute unit leave no room)
    __shared__ __attribute__((aligned(16))) bf16_t ds[kTrainRows * LD], wide[kTrainRows * kWide];
    __shared__ float2 red[kTrainWaves * kTrainRows];
    __shared__ __attribute__((aligned(16))) float sums[NS], vecs[kKept ? 6 * D + F : 4];
    bf16_t *const qs = wide, *const xs = wide, *const us = wide + kTrainRows * LD;
    typedef TrainVector<kKept> Vector;
    const Vector g1{kKept ? vecs : P.g1}, b1{kKept ? vecs + D : P.b1}, g2{kKept ? vecs + 2 * D : P.g2}, b2{kKept ? vecs + 3 * D : P.b2},
        g3{kKept ? vecs + 4 * D : P.g3}, b3{kKept ? vecs + 5 * D : P.b3}, bias1{kKept ? vecs + 6 * D : P.bias1};
    const bool normed = BACK || P.stats3;  // (the input of the first layer stands for itself)
    if constexpr (kKept) {
        if constexpr (FRONT) {
            train_keep<D>(vecs, P.g1, 0);
            train_keep<D>(vecs + D, P.b1, 1);
        }
        if constexpr (BACK) {
            train_keep<D>(vecs + 2 * D, P.g2, 2);
            train_keep<D>(vecs + 3 * D, P.b2, 3);
            train_keep<F>(vecs + 6 * D, P.bias1, 0);
        }
        if (normed) {
            train_keep<D>(vecs + 4 * D, P.g3, 1);
            train_keep<D>(vecs + 5 * D, P.b3, 2);
        }
    }
    for (int i = threadIdx.x; i < NS; i += kTrainWaves * 64) sums[i] = 0.f;
    __syncthreads();
    const long tiles = (P.M + kTrainRows - 1) / kTrainRows;
    for (long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const TrainLane L(tile, P.M);
        const bf16_t *const packed = train_opaque(P.packed), *const back_packed = train_opaque(P.back_packed);
        const bf16_t *const w_qkv_t = packed + train_matrix_at<D, F>(kTmQkvT), *const w_fo_t = packed + train_matrix_at<D, F>(kTmFoT),
                     *const w_1 = back_packed + train_matrix_at<D, F>(kTm1), *const w_1_t = back_packed + train_matrix_at<D, F>(kTm1T),
                     *const w_2_t = back_packed + train_matrix_at<D, F>(kTm2T), *const w_o_t = back_packed + train_matrix_at<D, F>(kTmOT);
        constexpr int HF = F / 2, NH = HF / 64;  // the feed-forward in two halves of its width
        TrainRing ring;
        f32x4 d[NB][2], r[NB][2], acc[NB][2];
        float2 st[2];
        if constexpr (FRONT) {
            ring.begin<NB, 3 * D / 32>(w_qkv_t, 0, L);
            train_stage<3 * D>(qs, LQ, P.dqkv, L);
            train_load<D>(d, P.dr2, L);
            train_load<D>(r, P.r1, L);
            train_get_stats(st, P.stats1, L);
            __syncthreads();
            ring.run<NB, 3 * D / 32>(acc, qs, LQ, w_qkv_t, 0, L);
            ring.begin<NB, D / 32>(w_fo_t, 0, L);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) d[b][tb] += acc[b][tb];
            train_norm(acc, r, st, g1, b1, L);
            const TrainPacked<NB> x1(acc);
            f32x4 r3[NB][2];
            train_load<D>(r3, P.r3, L);
            float2 st3[2] = {};
            if (normed) train_get_stats(st3, P.stats3, L);
            x1.template store<D>(P.x1, 0, L);
            train_norm_backward<D>(d, r, st, g1, sums + 5 * D + F, sums + 6 * D + F, red, L);
            train_to_lds(ds, LD, d, L);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) r[b][tb] = r3[b][tb];
            st[0] = st3[0];
            st[1] = st3[1];
            __syncthreads();
            ring.run<NB, D / 32>(acc, ds, LD, w_fo_t, 0, L);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) d[b][tb] += acc[b][tb];
        } else {
            train_load<D>(d, P.dx, L);
            train_load<D>(r, P.r3, L);
            train_get_stats(st, P.stats3, L);
        }
        if constexpr (!BACK) {
            if (normed) train_norm(r, r, st, g3, b3, L);
            TrainPacked<NB>(r).template store<D>(P.x, 0, L);
            train_unstage<D>(P.d1, ds, LD, L);
            train_store<D>(P.dx, d, L);
        } else {
            const TrainLane L(tile, P.M);
            ring.begin<NH, D / 32>(w_1, 0, L);
            f32x4 r2[NB][2];
            float2 st2[2];
            train_load<D>(r2, P.r2, L);
            train_get_stats(st2, P.stats2, L);
            if constexpr (FRONT) {
                train_norm(acc, r, st, g3, b3, L);
                TrainPacked<NB>(acc).template store<D>(P.x, 0, L);
                train_unstage<D>(P.d1, ds, LD, L);
            }
            train_norm_backward<D>(d, r, st, g3, sums, sums + D, red, L);  // (its barrier: nobody reads ds or the wide tile any more)
#pragma unroll
            for (int b = 0; b < NB; ++b) train_col_add(sums + 2 * D, d[b][0] + d[b][1], L.col(b), L);  // (rows past the end are zero)
            train_to_lds(ds, LD, d, L);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) r[b][tb] = r2[b][tb];
            st[0] = st2[0];
            st[1] = st2[1];
            train_norm(acc, r, st, g2, b2, L);
            train_to_lds(xs, LD, acc, L);
            __syncthreads();
#pragma unroll 1
            for (int half = 0; half < 2; ++half) {
                const int f0 = half * HF;
                const TrainLane L(tile, P.M);
                f32x4 u[NH][2], dh[NH][2];
                ring.run<NH, D / 32>(u, xs, LD, w_1, f0 / 16, L);
                ring.begin<NH, D / 32>(w_2_t, f0 / 16, L);
#pragma unroll
                for (int b = 0; b < NH; ++b) {
                    const f32x4 bias = bias1.at(f0 + L.col(b));
#pragma unroll
                    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            float hv, dv;
                            train_gelu(u[b][tb][e] + bias[e], hv, dv);
                            dh[b][tb][e] = hv;
                            u[b][tb][e] = dv;
                        }
                }
                const TrainPacked<NH> h(dh);
                ring.run<NH, D / 32>(dh, ds, LD, w_2_t, f0 / 16, L);
                if (half == 0) ring.begin<NH, D / 32>(w_1, HF / 16, L);
                else ring.begin<NB, F / 32>(w_1_t, 0, L);
                h.template store<F>(P.h, f0, L);
                if (half == 0) {
                    train_unstage<D>(P.d3, ds, LD, L);
                    train_unstage<D>(P.x2, xs, LD, L);
                }
#pragma unroll
                for (int b = 0; b < NH; ++b) {
#pragma unroll
                    for (int tb = 0; tb < 2; ++tb) u[b][tb] *= dh[b][tb];
                    train_col_add(sums + 5 * D + f0, u[b][0] + u[b][1], L.col(b), L);
                }
                train_to_lds(us + f0, LF, u, L);
            }
            __syncthreads();
            ring.run<NB, F / 32>(acc, us, LF, w_1_t, 0, L);
            ring.begin<NB, D / 32>(w_o_t, 0, L);
            train_unstage<F>(P.du, us, LF, L);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) d[b][tb] += acc[b][tb];
            train_norm_backward<D>(d, r, st, g2, sums + 3 * D, sums + 4 * D, red, L);
            train_to_lds(ds, LD, d, L);  // (its readers are behind the barrier inside the norm)
            __syncthreads();
            ring.run<NB, D / 32>(acc, ds, LD, w_o_t, 0, L);
            train_store<D>(P.dr2, d, L);
            train_unstage<D>(P.d2, ds, LD, L);
            TrainPacked<NB>(acc).template store<D>(P.dattn, 0, L);
        }
        __syncthreads();
    }
    // (without the other half its columns are zero and belong to nobody)
    for (int i = threadIdx.x; i < NS; i += kTrainWaves * 64) P.part[static_cast<long>(blockIdx.x) * NS + i] = sums[i];
}

// ---- the norm behind the stack, on the rows the head reads (rows first .. R - 1 of every batch entry)

struct TrainFinal {
    const float *r3; const float2 *stats3; const float *g3, *b3;  // of the last layer
    const float *g, *b; float eps;                                 // backbone.norm
    float *z;                  // [B, R - first, D]
    const float *dz;
    float *dx;                 // [M, D] gradient of the last layer's output: zero where the head does not read
    float *part;               // [gridDim.x][2 D]
    int B, R, first;
};

// Sum over the wavefront without the LDS: a row's four sums one after the other, 19 rows to a wavefront, were most of the
// backward kernel's time (38912 rows of 128: 24.3 us, 16.8 with this).
__device__ __forceinline__ float train_wave_sum(float x) {
    x += row_rotate<8>(x);
    x += row_rotate<4>(x);
    x += row_rotate<2>(x);
    x += row_rotate<1>(x);
    return row_sum(x);
}

// one wavefront per row; lane l holds elements l D/64 ..
template <int D, bool BACKWARD>
__global__ __launch_bounds__(256) void train_final_kernel(TrainFinal P) {
    constexpr int E = D / 64;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __shared__ float sums[4][2 * D];
    float cg[E], cb[E], g3[E], b3[E], g[E], be[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        cg[e] = cb[e] = 0.f;
        g3[e] = P.g3[lane * E + e];
        b3[e] = P.b3[lane * E + e];
        g[e] = P.g[lane * E + e];
        be[e] = P.b[lane * E + e];
    }
    const int per = BACKWARD ? P.R : P.R - P.first;
    const long rows = static_cast<long>(P.B) * per;
    for (long i = static_cast<long>(blockIdx.x) * 4 + wave; i < rows; i += static_cast<long>(gridDim.x) * 4) {
        const long b = i / per;
        const int in = static_cast<int>(i % per), at = BACKWARD ? in : in + P.first;
        const long m = b * P.R + at;
        if (BACKWARD && at < P.first) {
#pragma unroll
            for (int e = 0; e < E; ++e) P.dx[m * D + lane * E + e] = 0.f;
            continue;
        }
        const float2 st = P.stats3[m];
        float x[E], s = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            x[e] = fmaf((P.r3[m * D + lane * E + e] - st.x) * st.y, g3[e], b3[e]);
            s += x[e];
        }
        const float mean = train_wave_sum(s) * (1.f / D);
        float q = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) q = fmaf(x[e] - mean, x[e] - mean, q);
        const float rstd = rsqrtf(train_wave_sum(q) * (1.f / D) + P.eps);
        const long zi = (b * (P.R - P.first) + (at - P.first)) * D + lane * E;
        if (!BACKWARD) {
#pragma unroll
            for (int e = 0; e < E; ++e) P.z[zi + e] = fmaf((x[e] - mean) * rstd, g[e], be[e]);
        } else {
            float xh[E], gy[E], s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const float dy = P.dz[zi + e];
                xh[e] = (x[e] - mean) * rstd;
                cg[e] = fmaf(dy, xh[e], cg[e]);
                cb[e] += dy;
                gy[e] = dy * g[e];
                s1 += gy[e];
                s2 = fmaf(gy[e], xh[e], s2);
            }
            const float m1 = train_wave_sum(s1) * (1.f / D), m2 = train_wave_sum(s2) * (1.f / D);
#pragma unroll
            for (int e = 0; e < E; ++e) P.dx[m * D + lane * E + e] = rstd * (gy[e] - m1 - xh[e] * m2);
        }
    }
    if (BACKWARD) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            sums[wave][lane * E + e] = cg[e];
            sums[wave][D + lane * E + e] = cb[e];
        }
        __syncthreads();
        for (int i = threadIdx.x; i < 2 * D; i += 256)
            P.part[static_cast<long>(blockIdx.x) * 2 * D + i] = (sums[0][i] + sums[1][i]) + (sums[2][i] + sums[3][i]);
    }
}

// ---- weight gradients: C[n][k] = sum_m P[m][n] Q[m][k] in pieces of 128 x 128, each over `slices` runs of
// rows.  Both operands want the contraction (rows) consecutive in a lane: transposing reads of row-major LDS
// tiles.  Eight wavefronts: two groups take half of a tile's 64 rows each, a group's four hold 64 x 64.
//
// Bound: the trip to memory; a workgroup waits for one tile while it has multiplied the one before.  38912 rows of 128, nine
// pieces (140 MB): 40 us.  Two tiles on their way, or tiles of 128 rows on sixteen wavefronts, took 29, and both were in the
// tree when a run of the device tests faulted; neither is to come back before the cause of that is known.
struct TrainGradJobs {
    const bf16_t *p[kTrainMaxJobs], *q[kTrainMaxJobs];
    int ldp[kTrainMaxJobs], ldq[kTrainMaxJobs];
    float *part;               // [slices][jobs][128 * 128]
    long M, rows_per_slice;    // a multiple of 64
    int jobs;
};

static __global__ __launch_bounds__(512) void train_weight_grad_kernel(TrainGradJobs J) {
    typedef MfmaOps<bf16_t> Ops;
    constexpr int TR = 64, LD = 128 + 16;  // 288 bytes: 32 mod 128, what the transposing reads want
    __shared__ __attribute__((aligned(16))) bf16_t lds[2][2][TR * LD];
    const int job = blockIdx.x, slice = blockIdx.y;
    const bf16_t *const p = J.p[job], *const q = J.q[job];
    const int ldp = J.ldp[job], ldq = J.ldq[job];
    const long m0 = slice * J.rows_per_slice, m1 = min(J.M, m0 + J.rows_per_slice);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int half = wave >> 2, wn = wave & 1, wk = (wave >> 1) & 1;
    f32x16 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][c][v] = 0.f;
    u32x4 rp[2], rq[2];
    auto fetch = [&](long m) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int i = tid + 512 * x, r = i / 16, c = i % 16;
            const long row = min(m + r, J.M - 1);
            rp[x] = *reinterpret_cast<const u32x4 *>(p + row * ldp + 8 * c);
            rq[x] = *reinterpret_cast<const u32x4 *>(q + row * ldq + 8 * c);
        }
    };
    auto put = [&](int buf, long m) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int i = tid + 512 * x, r = i / 16, c = i % 16;
            const u32x4 zero = {0u, 0u, 0u, 0u};
            *reinterpret_cast<u32x4 *>(&lds[buf][0][r * LD + 8 * c]) = m + r < m1 ? rp[x] : zero;  // rows past the end: no product
            *reinterpret_cast<u32x4 *>(&lds[buf][1][r * LD + 8 * c]) = rq[x];
        }
    };
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    // rows m .. m + 15, columns n .. n + 31 as an operand: lane column n + lane % 32, rows m + 8 (lane / 32) + e
    auto operand = [&](const bf16_t *t, int m, int n) {
        const bf16_t *a = t + (m + 8 * (lane >> 5) + ((lane & 15) >> 2)) * LD + n + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(a));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(a + 4 * LD));
        const s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        return __builtin_bit_cast(bf16x8, both);
    };
    if (m0 < m1) {
        fetch(m0);
        put(0, m0);
        int buf = 0;
        for (long m = m0; m < m1; m += TR, buf ^= 1) {
            const bool more = m + TR < m1;
            if (more) fetch(m + TR);
            __syncthreads();
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                bf16x8 a[2], c[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    a[i] = operand(lds[buf][0], 32 * half + 16 * ks, 64 * wn + 32 * i);
                    c[i] = operand(lds[buf][1], 32 * half + 16 * ks, 64 * wk + 32 * i);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = Ops::mma(a[i], c[j], acc[i][j]);
            }
            if (more) put(buf ^ 1, m + TR);  // the other buffer's readers passed the barrier above
        }
    }
    // the second group's sums through LDS (64 x 64 floats per wavefront pair would fill it: one quarter at a time)
    float *const x = reinterpret_cast<float *>(lds);
    float *const out = J.part + (static_cast<long>(slice) * J.jobs + job) * (128 * 128);
    const int c32 = lane & 31, hb = lane >> 5;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            __syncthreads();
            if (half == 1) {
#pragma unroll
                for (int v = 0; v < 16; ++v) x[(wave & 3) * 1024 + v * 64 + lane] = acc[i][j][v];
            }
            __syncthreads();
            if (half == 0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int n = 64 * wn + 32 * i + 8 * (v >> 2) + 4 * hb + (v & 3), k = 64 * wk + 32 * j + c32;
                    out[n * 128 + k] = acc[i][j][v] + x[(wave & 3) * 1024 + v * 64 + lane];
                }
            }
        }
}

// Adds up the slices of the weight gradients (where each piece goes: `out`, row stride `ld`) and the workgroups'
// column sums.  Bound: trips to memory one after the other, so a thread has all it adds up on its way at once, up to 32
// slices; a column's rows (some 700) are dealt over 16 threads, the columns over as many workgroups.  A step's reduction of
// 28 slices of nine pieces: 7.7 us with 64 columns to a workgroup and 16 slices on their way, 6.2 with these.
constexpr int kTrainReduceCols = 16;
struct TrainReduce {
    const float *part; int jobs, slices;
    float *out[kTrainMaxJobs]; int ld[kTrainMaxJobs];
    struct Cols {
        const float *part;     // [groups][ld], n columns of it
        float *out;
        int groups, ld, n;     // n: a multiple of kTrainReduceCols
    } cols[2];
    int n_cols;
};
static __global__ __launch_bounds__(256) void train_reduce_kernel(TrainReduce P) {
    const int tid = threadIdx.x;
    const int piece_groups = P.jobs * 16;  // 16 workgroups of 1024 elements per piece
    if (static_cast<int>(blockIdx.x) < piece_groups) {
        const int job = blockIdx.x / 16, e = (blockIdx.x % 16) * 1024 + 4 * tid;
        const long step = static_cast<long>(P.jobs) * 16384;
        const float *const from = P.part + static_cast<long>(job) * 16384 + e;
        constexpr int AHEAD = 32;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        for (int i = 0; i < P.slices; i += AHEAD) {
            f32x4 v[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) v[u] = *reinterpret_cast<const f32x4 *>(from + min(i + u, P.slices - 1) * step);
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) s += i + u < P.slices ? v[u] : f32x4{0.f, 0.f, 0.f, 0.f};
        }
        *reinterpret_cast<f32x4 *>(P.out[job] + static_cast<long>(e / 128) * P.ld[job] + e % 128) = s;
        return;
    }
    __shared__ float acc[256];
    int at = (static_cast<int>(blockIdx.x) - piece_groups) * kTrainReduceCols;
    int which = 0;
    while (which + 1 < P.n_cols && at >= P.cols[which].n) {
        at -= P.cols[which].n;
        ++which;
    }
    const TrainReduce::Cols C = P.cols[which];
    constexpr int SIDE = 256 / kTrainReduceCols, AHEAD = 32;
    const int c = tid % kTrainReduceCols, side = tid / kTrainReduceCols;
    float part[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) part[u] = 0.f;
    const float *col = C.part + at + c;
    for (int i = side; i < C.groups; i += SIDE * AHEAD) {
        float v[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) v[u] = col[static_cast<long>(min(i + SIDE * u, C.groups - 1)) * C.ld];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) part[u] += i + SIDE * u < C.groups ? v[u] : 0.f;
    }
#pragma unroll
    for (int half = AHEAD / 2; half > 0; half /= 2)
#pragma unroll
        for (int u = 0; u < half; ++u) part[u] += part[u + half];
    acc[tid] = part[0];
    __syncthreads();
    if (tid < kTrainReduceCols) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < SIDE; ++i) s += acc[i * kTrainReduceCols + tid];
        C.out[at + tid] = s;
    }
}

// ---- row embeddings (model.py:23-76, :323-333): x = mean(features) w_x + b_x + marker, context and buffer rows
// with y w_y + b_y, buffer rows with their position token

struct TrainEmbed {
    const float *x[3], *y[2];  // context, buffer, target rows: [B, n, feat] and [B, n]
    int n[3], feat;
    const float *w_x, *b_x, *w_y, *b_y, *markers, *tokens;  // markers [3, D]: target, context, buffer; tokens [>= n[1], D]
    float *out;                // [B, R, D]
    float2 *xy;                // [B, R] (feature mean, y): what the backward pass needs of the data
    int B, R;
};
template <int D>
__global__ __launch_bounds__(256) void train_embed_kernel(TrainEmbed P) {
    constexpr int PER = D / 4;  // threads per row
    const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x, m = i / PER;
    const int d = 4 * static_cast<int>(i % PER);
    if (m >= static_cast<long>(P.B) * P.R) return;
    const long b = m / P.R;
    int r = static_cast<int>(m % P.R), kind = 0;
    while (kind < 2 && r >= P.n[kind]) r -= P.n[kind++];
    const long at = b * P.n[kind] + r;
    float mean = 0.f;
    for (int f = 0; f < P.feat; ++f) mean += P.x[kind][at * P.feat + f];
    mean /= P.feat;
    const float y = kind < 2 ? P.y[kind][at] : 0.f;
    f32x4 v = *reinterpret_cast<const f32x4 *>(P.w_x + d) * mean + *reinterpret_cast<const f32x4 *>(P.b_x + d) +
              *reinterpret_cast<const f32x4 *>(P.markers + (kind == 2 ? 0 : kind + 1) * D + d);
    if (kind < 2) v += *reinterpret_cast<const f32x4 *>(P.w_y + d) * y + *reinterpret_cast<const f32x4 *>(P.b_y + d);
    if (kind == 1) v += *reinterpret_cast<const f32x4 *>(P.tokens + static_cast<long>(r) * D + d);
    *reinterpret_cast<f32x4 *>(P.out + m * D + d) = v;
    if (d == 0) P.xy[m] = make_float2(mean, y);
}

// Column sums of dx [B, R, D]: over context rows, buffer rows, target rows, weighted by the feature mean, by y.
// blockIdx.y < slices: a share of one batch entry's rows -> part[block][5][D];
// blockIdx.y == slices: the gradient of token blockIdx.x, summed over the batch (blockIdx.x < n_tokens).
struct TrainEmbedBackward {
    const float *dx;
    const float2 *xy;
    int B, R, n_ctx, n_buf, slices;
    float *part, *d_tokens;
};
// Four columns to a thread, as many rows side by side as a workgroup has threads for (38912 rows of 128: 33 us with one
// column to a thread and one row to a workgroup, under 10).
template <int D>
__global__ __launch_bounds__(256) void train_embed_backward_kernel(TrainEmbedBackward P) {
    constexpr int PER = D / 4, SIDE = 256 / PER;
    __shared__ __attribute__((aligned(16))) f32x4 acc[5][256];
    const int tid = threadIdx.x, d = 4 * (tid % PER), side = tid / PER;
    f32x4 s[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bool tokens = static_cast<int>(blockIdx.y) == P.slices;
    if (tokens ? static_cast<int>(blockIdx.x) >= P.n_buf : static_cast<int>(blockIdx.x) >= P.B) return;
    if (tokens) {
        const float *const src = P.dx + (P.n_ctx + blockIdx.x) * static_cast<long>(D) + d;
#pragma unroll 4
        for (int b = side; b < P.B; b += SIDE) s[0] += *reinterpret_cast<const f32x4 *>(src + static_cast<long>(b) * P.R * D);
    } else {
        const long b = blockIdx.x;
#pragma unroll 4
        for (int r = blockIdx.y * SIDE + side; r < P.R; r += P.slices * SIDE) {
            const f32x4 v = *reinterpret_cast<const f32x4 *>(P.dx + (b * P.R + r) * D + d);
            const float2 xy = P.xy[b * P.R + r];
            const int kind = r < P.n_ctx ? 0 : r < P.n_ctx + P.n_buf ? 1 : 2;
#pragma unroll
            for (int k = 0; k < 3; ++k) s[k] += k == kind ? v : f32x4{0.f, 0.f, 0.f, 0.f};
            s[3] += v * xy.x;
            s[4] += v * xy.y;
        }
    }
    const int sums = tokens ? 1 : 5;
#pragma unroll
    for (int k = 0; k < 5; ++k) acc[k][tid] = s[k];
    __syncthreads();
    for (int i = tid; i < sums * PER; i += 256) {
        const int k = i / PER, c = i % PER;
        f32x4 t = acc[k][c];
#pragma unroll
        for (int x = 1; x < SIDE; ++x) t += acc[k][x * PER + c];
        float *const out = tokens ? P.d_tokens + static_cast<long>(blockIdx.x) * D : P.part + ((blockIdx.x * static_cast<long>(P.slices) + blockIdx.y) * 5 + k) * D;
        *reinterpret_cast<f32x4 *>(out + 4 * c) = t;
    }
}
// sums [5][D] -> d(w_x), d(b_x), d(w_y), d(b_y) [D] each, d(markers) [3, D]
static __global__ void train_embed_finish_kernel(const float *sums, float *grads, int D) {
    const int d = threadIdx.x;
    const float ctx = sums[d], buf = sums[D + d], tgt = sums[2 * D + d];
    grads[d] = sums[3 * D + d];
    grads[D + d] = ctx + buf + tgt;
    grads[2 * D + d] = sums[4 * D + d];
    grads[3 * D + d] = ctx + buf;
    grads[4 * D + d] = tgt;
    grads[5 * D + d] = ctx;
    grads[6 * D + d] = buf;
}

}  // namespace artab
