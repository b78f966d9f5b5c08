// The layer kernels of fused_layer.h for many token rows (gfx950, bf16/f16): prefill and teacher-forced passes over
// thousands of rows, where what counts is rows per second and not the latency of one tile.
//
// Bound: the row-wise vector work (three norms, the activation, packing) and the matrix cores, about 12 us each for
// 32768 rows of 256 at best; tensors in and out once are 20 us.  fused_layer.h keeps whole matrices in flight in
// registers, one workgroup of 32 rows per compute unit, so that nothing else runs on it while a norm exchanges its row
// sums.  Here a wavefront has 128 registers: a ring of kRing weight fragments that runs on from product to product, and
// 32 RB rows per workgroup, each fragment multiplied with RB row blocks.  Two workgroups share a compute unit and
// are in different phases.  q, k and v leave through the wavefront's own columns of the tile that is free by then,
// without a barrier.  At 32768 rows of 256 (52 us; before 71) the vector units are 37 % busy, the matrix cores 25 %, the
// address unit 48 % and the LDS 29 %: what is left is four wavefronts per SIMD that wait for each other.
//
// Sums: a workgroup starts its contractions at its own step (as WeightStream::begin, and for the same reason), so the
// order of a product's sums depends on the tile of the row.  The activation is x Phi(x) from normal_tail(), 0.51 units
// in the last place of f16 after rounding (erff 1.7).
#pragma once

#include "fused_layer.h"

namespace artab {

// Row blocks of 32 per workgroup for `rows` token rows; 0: the tiles of fused_layer.h, which are faster while a
// compute unit has one of them, the more so where some have none: those fetch the weights into the L2 (5001 rows of
// 256 between two attention calls: 17.6, here 20.5, though on weights that are in the L2 17.7 and 17.1).  One layer boundary in bf16, us, 16-row tiles / 32-row tiles of fused_layer.h / one block / two:
// d_model 128, 8192 rows 13.0 / 13.9 / 12.5, 16384 22.5 / 17.9 / 16.5, 32768 41.1 / 32.6 / 26.0, 65536 82 / 62 / 46.5;
// d_model 256, 4096 rows 14.7 / 17.4 / 16.8 / 25.1, 9000 36.1 / 31.9 / 25.3 / 26.5, 16384 49.0 / 34.9 / 29.5 / 31.9,
// 24000 77.9 / 53.7 / 44.5 / 44.8, 32768 100 / 71.3 / 57.1 / 51.7, 65536 197 / 139 / 115 / 101;
// d_model 512, 4096 rows 39.9 / 49.1 / 44.2, 9000 98.6 / 95.3 / 72.4, 32768 274 / 209 / 172.
constexpr int wide_blocks(int D, long rows) { return rows <= 8192 ? 0 : D == 256 && rows > 24576 ? 2 : 1; }
constexpr int kWideRing = 8;
constexpr int kWideFeedForward = 256;  // the feed-forward width these are built for (others: fused_layer.h)

// Where the projected keys and values go instead of the q/k/v matrix: row r of the launch is row r % N of batch entry
// r / N, head h starts h * sh elements into its entry.
struct KeyValueRows {
    void *k, *v;  // null: the matrix
    long sb, sh;  // elements
    int N, Dh;    // head_dim: 32, 64 or 128, rows of a head contiguous
};

__device__ __forceinline__ float wide_over_token(float x) {  // the lanes that hold the same token: l and l ^ 32
    const unsigned a = __builtin_bit_cast(unsigned, x);
    auto s = __builtin_amdgcn_permlane32_swap(a, a, false, false);
    const unsigned lo = s[0], hi = s[1];
    return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
__device__ __forceinline__ float wide_gelu(float x) {
    const float tail = normal_tail(x);
    return x * (x > 0.f ? 1.f - tail : tail);
}

// One workgroup's products on tiles of 32 RB rows in LDS (row strides LDD and LDF).
template <typename T, int D, int F, int RB>
struct WideTile {
    static constexpr int TR = 32 * RB, NW = fused_waves(D), NT = NW * 64;
    static constexpr int LDD = D + 8, LDF = F + 8, LDM = LDD > LDF ? LDD : LDF, VW = D > F ? D : F;
    static constexpr int NBD = D / 32 / NW, NBF = F / 32 / NW;
    static_assert(D % (32 * NW) == 0 && F % (32 * NW) == 0, "whole blocks per wavefront");
    typedef typename MfmaOps<T>::vec vec;
    static constexpr size_t kLds = sizeof(T) * (TR * LDM + TR * LDD + kVecSlots * VW) + sizeof(float) * 2 * NW * TR;

    T *a0, *a1, *vecs;
    float *red_a, *red_b;
    int wave, lane, c, hb, rot;
    vec ring[kWideRing];

    __device__ __forceinline__ WideTile(unsigned char *lds) {
        a0 = reinterpret_cast<T *>(lds);
        a1 = a0 + TR * LDM;
        vecs = a1 + TR * LDD;
        red_a = reinterpret_cast<float *>(vecs + kVecSlots * VW);
        red_b = red_a + NW * TR;
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        lane = threadIdx.x & 63;
        c = lane & 31;
        hb = lane >> 5;
        rot = static_cast<int>(blockIdx.x) >> 3;
    }

    // Fragment i (contraction step i / NB, block i % NB of this wavefront) of the product with packed weight w [.., K].
    template <int K, int NB>
    __device__ __forceinline__ vec fragment(const T *w, int i) const {
        const int ks = (i / NB + rot) & (K / 16 - 1), blk = wave + NW * (i % NB);
        const T *p = w + (static_cast<long>(blk) * (K / 16) + ks) * 512;
        return *reinterpret_cast<const vec *>(p + 8 * lane);
    }
    template <int K, int NB>
    __device__ __forceinline__ void start(const T *w) {
#pragma unroll
        for (int i = 0; i < kWideRing; ++i) ring[i] = fragment<K, NB>(w, i);
    }
    // acc[b][r] = (W A^T) for block b of the wavefront and row block r; the ring goes on with the next product's fragments.
    template <int K, int NB, int KN, int NBN>
    __device__ __forceinline__ void product(f32x16 (&acc)[NB][RB], const T *w, const T *act, int ld, const T *w_next) {
        constexpr int KS = K / 16, N = KS * NB;
        static_assert(N % kWideRing == 0 && (KN / 16) * NBN % kWideRing == 0, "a product is whole turns of the ring");
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < RB; ++r)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[b][r][v] = 0.f;
        const T *a = act + c * ld + 8 * hb;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            vec af[RB];
#pragma unroll
            for (int r = 0; r < RB; ++r) af[r] = *reinterpret_cast<const vec *>(a + 32 * r * ld + 16 * ((ks + rot) & (KS - 1)));
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int i = ks * NB + b;
#pragma unroll
                for (int r = 0; r < RB; ++r) acc[b][r] = MfmaOps<T>::mma(ring[i % kWideRing], af[r], acc[b][r]);
                if (i + kWideRing < N) ring[i % kWideRing] = fragment<K, NB>(w, i + kWideRing);
                else if (w_next) ring[i % kWideRing] = fragment<KN, NBN>(w_next, i + kWideRing - N);
            }
        }
    }
    // acc = LayerNorm(acc + res [+ bias]) into dst (row stride LDD); one barrier inside, after which nobody reads what
    // the products and the residual read.
    __device__ __forceinline__ void norm(f32x16 (&acc)[NBD][RB], const T *res, const T *bias, const T *gam, const T *bet, T *dst, float eps) {
        constexpr float kLocal = NBD * 32;
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            float s = 0.f, q = 0.f;
#pragma unroll
            for (int b = 0; b < NBD; ++b)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int col = 32 * (wave + NW * b) + 8 * g + 4 * hb;
                    float x[4];
                    load4f<T>(res + (32 * r + c) * LDD + col, x);
                    if (bias) {
                        float y[4];
                        load4f<T>(bias + col, y);
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[e] += y[e];
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        acc[b][r][4 * g + e] += x[e];
                        s += acc[b][r][4 * g + e];
                    }
                }
            s = wide_over_token(s);
            const float mean = s * (1.f / kLocal);
#pragma unroll
            for (int b = 0; b < NBD; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const float d = acc[b][r][v] - mean;
                    q = fmaf(d, d, q);
                }
            q = wide_over_token(q);
            if (hb == 0) {
                red_a[wave * TR + 32 * r + c] = mean;
                red_b[wave * TR + 32 * r + c] = q;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            float lm[NW], tot = 0.f, m2 = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                lm[w] = red_a[w * TR + 32 * r + c];
                tot += lm[w];
            }
            const float mean = tot * (1.f / NW);
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const float d = lm[w] - mean;
                m2 += red_b[w * TR + 32 * r + c] + kLocal * d * d;
            }
            const float rstd = rsqrtf(m2 * (1.f / D) + eps);
#pragma unroll
            for (int b = 0; b < NBD; ++b)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int col = 32 * (wave + NW * b) + 8 * g + 4 * hb;
                    float ga[4], be[4], o[4];
                    load4f<T>(gam + col, ga);
                    load4f<T>(bet + col, be);
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = (acc[b][r][4 * g + e] - mean) * rstd * ga[e] + be[e];
                    store4f<T>(dst + (32 * r + c) * LDD + col, o[0], o[1], o[2], o[3]);
                }
        }
        __syncthreads();
    }
    __device__ __forceinline__ void activation(f32x16 (&acc)[NBF][RB], const T *bias) {
#pragma unroll
        for (int b = 0; b < NBF; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int col = 32 * (wave + NW * b) + 8 * g + 4 * hb;
                float y[4];
                load4f<T>(bias + col, y);
#pragma unroll
                for (int r = 0; r < RB; ++r) {
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = wide_gelu(acc[b][r][4 * g + e] + y[e]);
                    store4f<T>(a0 + (32 * r + c) * LDF + col, o[0], o[1], o[2], o[3]);
                }
            }
        __syncthreads();
    }
    // The wavefront's columns of a tile in registers to memory, through its own columns of `tile` (row stride LDD):
    // `at(row)` is where the tile's row begins, `head(col0)` how much further 32 columns from col0 on do.
    template <typename Row, typename Head>
    __device__ __forceinline__ void store_columns(const f32x16 (&acc)[NBD][RB], T *tile, int valid, Row at, Head head) {
#pragma unroll
        for (int b = 0; b < NBD; ++b) {
            const int col0 = 32 * (wave + NW * b);
#pragma unroll
            for (int r = 0; r < RB; ++r)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    store4f<T>(tile + (32 * r + c) * LDD + col0 + 8 * g + 4 * hb, acc[b][r][4 * g], acc[b][r][4 * g + 1], acc[b][r][4 * g + 2],
                               acc[b][r][4 * g + 3]);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < TR / 16; ++i) {  // 16 rows of 64 bytes at a time
                const int row = 16 * i + (lane >> 2), col = col0 + 8 * (lane & 3);
                const u32x4 v = *reinterpret_cast<const u32x4 *>(tile + row * LDD + col);
                if (row < valid) *reinterpret_cast<u32x4 *>(at(row) + head(col0) + 8 * (lane & 3)) = v;
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    __device__ __forceinline__ void store_tile(const T *tile, T *dst, int valid) {
        unstage_tile<T, D, NT, TR>(dst, D, tile, LDD, valid, threadIdx.x);
    }

    // x1 = LN2(y + attn W_o^T), out = LN3(x1 + gelu(x1 W_1^T + b_1) W_2^T + b_2), left in a0.  The ring holds W_o's first
    // fragments and, at the end, those of `w_next` [D, D].
    __device__ __forceinline__ void post(const FusedPostParams &P, const T *w_next) {
        const T *w_o = static_cast<const T *>(P.w_o), *w_1 = static_cast<const T *>(P.w_1), *w_2 = static_cast<const T *>(P.w_2);
        f32x16 acc[NBD][RB];
        product<D, NBD, D, NBF>(acc, w_o, a0, LDD, w_1);
        norm(acc, a1, nullptr, vecs + kVecG2 * VW, vecs + kVecB2 * VW, a1, P.eps2);
        {
            f32x16 h[NBF][RB];
            product<D, NBF, F, NBD>(h, w_1, a1, LDD, w_2);
            activation(h, vecs + kVecBias1 * VW);
        }
        product<F, NBD, D, NBD>(acc, w_2, a0, LDF, w_next);
        norm(acc, a1, vecs + kVecBias2 * VW, vecs + kVecG3 * VW, vecs + kVecB3 * VW, a0, P.eps3);
    }
    // y = LN1(x + x W_fo^T) and q, k, v = y W^T from the tile in a0.  The ring holds W_fo's first fragments.
    __device__ __forceinline__ void pre(const FusedPreParams &P, const KeyValueRows &kv, long row0, int valid) {
        const T *w_fo = static_cast<const T *>(P.w_fo), *w_qkv = static_cast<const T *>(P.w_qkv);
        f32x16 acc[NBD][RB];
        product<D, NBD, D, NBD>(acc, w_fo, a0, LDD, w_qkv);
        norm(acc, a0, nullptr, vecs + kVecG1 * VW, vecs + kVecB1 * VW, a1, P.eps);
        store_tile(a1, static_cast<T *>(P.y) + row0 * D, valid);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const T *w = w_qkv + static_cast<long>(p) * D * D;
            product<D, NBD, D, NBD>(acc, w, a1, LDD, p < 2 ? w + static_cast<long>(D) * D : nullptr);
            if (p == 0 || !kv.k) {
                T *const dst = static_cast<T *>(P.qkv) + row0 * (3 * D) + p * D;
                store_columns(acc, a0, valid, [&](int row) { return dst + row * (3L * D); }, [](int col0) { return col0; });
            } else {
                T *const dst = static_cast<T *>(p == 1 ? kv.k : kv.v);
                const unsigned first = static_cast<unsigned>(row0), n_rows = static_cast<unsigned>(kv.N);
                store_columns(
                    acc, a0, valid,
                    [&](int row) {
                        const unsigned r = first + row, entry = r / n_rows;
                        return dst + entry * kv.sb + static_cast<long>(r - entry * n_rows) * kv.Dh;
                    },
                    [&](int col0) { return col0 / kv.Dh * kv.sh + col0 % kv.Dh; });
            }
        }
    }
};

template <typename T, int D, int F, int RB>
__device__ __forceinline__ void wide_stage_post(WideTile<T, D, F, RB> &tile, const FusedPostParams &P, long row0, int valid) {
    typedef WideTile<T, D, F, RB> W;
    const int tid = threadIdx.x;
    dma_tile<T, D, W::NT, W::TR>(tile.a0, W::LDD, static_cast<const T *>(P.attn) + row0 * P.lda, P.lda, valid, tid);
    dma_tile<T, D, W::NT, W::TR>(tile.a1, W::LDD, static_cast<const T *>(P.y) + row0 * P.ldy, P.ldy, valid, tid);
    dma_vector<T, D, W::NT>(tile.vecs + kVecG2 * W::VW, P.g2, tid, 0);
    dma_vector<T, D, W::NT>(tile.vecs + kVecB2 * W::VW, P.b2, tid, 1);
    dma_vector<T, F, W::NT>(tile.vecs + kVecBias1 * W::VW, P.bias_1, tid, 2);
    dma_vector<T, D, W::NT>(tile.vecs + kVecG3 * W::VW, P.g3, tid, 3);
    dma_vector<T, D, W::NT>(tile.vecs + kVecB3 * W::VW, P.b3, tid, 4);
    dma_vector<T, D, W::NT>(tile.vecs + kVecBias2 * W::VW, P.bias_2, tid, 5);
}

template <typename T, int D, int F, int RB>
__global__ __launch_bounds__(fused_waves(D) * 64, 4) void wide_pre_kernel(FusedPreParams P, KeyValueRows kv) {
    typedef WideTile<T, D, F, RB> W;
    __shared__ __attribute__((aligned(16))) unsigned char lds[W::kLds];
    W tile(lds);
    const long row0 = static_cast<long>(blockIdx.x) * W::TR;
    const int valid = static_cast<int>(min(static_cast<long>(W::TR), P.rows - row0));
    tile.template start<D, W::NBD>(static_cast<const T *>(P.w_fo));
    dma_tile<T, D, W::NT, W::TR>(tile.a0, W::LDD, static_cast<const T *>(P.x) + row0 * P.ldx, P.ldx, valid, threadIdx.x);
    stage_pre_vectors<T, D, W::NT>(P, tile.vecs, W::VW, threadIdx.x);
    wait_all_loads();
    __syncthreads();
    tile.pre(P, kv, row0, valid);
}

template <typename T, int D, int F, int RB>
__global__ __launch_bounds__(fused_waves(D) * 64, 4) void wide_post_kernel(FusedPostParams P) {
    typedef WideTile<T, D, F, RB> W;
    __shared__ __attribute__((aligned(16))) unsigned char lds[W::kLds];
    W tile(lds);
    const long row0 = static_cast<long>(blockIdx.x) * W::TR;
    const int valid = static_cast<int>(min(static_cast<long>(W::TR), P.rows - row0));
    tile.template start<D, W::NBD>(static_cast<const T *>(P.w_o));
    wide_stage_post<T, D, F, RB>(tile, P, row0, valid);
    wait_all_loads();
    __syncthreads();
    tile.post(P, nullptr);
    tile.store_tile(tile.a0, static_cast<T *>(P.out) + row0 * D, valid);
}

template <typename T, int D, int F, int RB>
__global__ __launch_bounds__(fused_waves(D) * 64, 4) void wide_post_pre_kernel(FusedPostParams P, FusedPreParams N, KeyValueRows kv) {
    typedef WideTile<T, D, F, RB> W;
    __shared__ __attribute__((aligned(16))) unsigned char lds[W::kLds];
    W tile(lds);
    const long row0 = static_cast<long>(blockIdx.x) * W::TR;
    const int valid = static_cast<int>(min(static_cast<long>(W::TR), P.rows - row0));
    tile.template start<D, W::NBD>(static_cast<const T *>(P.w_o));
    wide_stage_post<T, D, F, RB>(tile, P, row0, valid);
    stage_pre_vectors<T, D, W::NT>(N, tile.vecs, W::VW, threadIdx.x);
    wait_all_loads();
    __syncthreads();
    tile.post(P, static_cast<const T *>(N.w_fo));
    tile.pre(N, kv, row0, valid);
}

}  // namespace artab
