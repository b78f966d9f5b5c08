// The layer around the row attention in float32 (gfx950, v_mfma_f32_16x16x4_f32), one launch between two
// attention calls: the tail of a layer (out projection, norm2, feed-forward, norm3) and the head of the next
// (feature stage, norm1, q/k/v projections), or either part alone.
//
// A workgroup takes TR rows through all products with the activations in LDS; only attention output, y and
// q/k/v touch memory.  Bound: the float32 matrix rate of its compute unit, 256 FLOP per clock: 16 rows of
// d_model 256 are 14.7 MFLOP, 24 us; a launch of up to 4096 rows takes 38 to 41 us, where seven library products
// and the norms and activation between them took 60 (1440 rows) and, from Python, 200 us of host time.
//
// Few rows leave most compute units idle in tiles of 16, so there are tiles of 8 and 4, which have to do without the
// 16x16 form: v_mfma_f32_4x4x1_16b_f32 takes four tokens to 64 weights at the same rate, the sixteen blocks of a
// fragment being four groups of outputs times four of contraction elements, whose sums are added at the end.  Four rows
// are 6 us of products at d_model 256, under the 12 us that 1.8 MB of weights take through the compute unit.  A layer of
// 333 rows of 256 with its attention 46 -> 30 us, of 1773 (density of 16 x 45 targets) 71 -> 59.  Layouts:
//   * D = W X^T: a weight row is a row of the first operand, a token a column, so that a lane holds four
//     neighbouring outputs of one token; contraction step 4t + e takes the elements {16t + 4g + e} (g = lane / 16),
//     so fragments of both operands are 16-byte pieces;
//   * weights are packed once per fragment ([N / 16][K / 16][64 lanes][4], 1 KiB each), read from the L2 straight
//     into registers, 4 to 8 fragments ahead: 1 KiB feeds 4 products of 32 clocks, 32 bytes per clock and CU,
//     half of what its L2 port delivers.  Tiles of 32 rows, half the weight traffic, were no faster at any size:
//     4096 rows 406 -> 502 us for 4 layers with their attention, 12288 rows 849 -> 932, 16896 rows 1310 -> 1379.
#pragma once

#include "common.h"

namespace artab {

struct F32LayerParams {
    // tail of a layer; post == 0: x is read instead
    const float *attn, *y, *w_o, *gamma2, *beta2, *w_1, *b_1, *w_2, *b_2, *gamma3, *beta3;
    const float *x;
    float *out;  // the layer's output where no head follows
    // head of the next; pre == 0: out is written instead
    const float *w_fo, *gamma1, *beta1, *w_qkv;
    float *y_next, *qkv;
    long rows;
    int post, pre;
    float eps1, eps2, eps3;
};

constexpr int f32_layer_waves(int D) { return D == 128 ? 8 : 16; }

// The results of a product over a tile of TR rows, and where in a wavefront they are: a lane that `holds` has outputs
// 4 sub .. 4 sub + 3 of token tok.
template <int TR>
struct F32Tile {
    static_assert(TR == 4 || TR == 8 || TR == 16, "whole sets of four rows");
    static constexpr bool kNarrow = TR < 16;  // products of 4x4 blocks
    static constexpr int kSets = kNarrow ? TR / 4 : 1;
    int tok, sub;
    bool holds;
    __device__ __forceinline__ explicit F32Tile(int lane) {
        if constexpr (kNarrow) {  // every row of 16 lanes has all sums: the first kSets rows hold a set of four tokens each
            tok = 4 * (lane >> 4) + (lane & 3);
            sub = (lane >> 2) & 3;
            holds = lane < 16 * kSets;
        } else {
            tok = lane & 15;
            sub = lane >> 4;
            holds = true;
        }
    }
    // the row of the tile that the lane reads as the second operand, of set i
    static __device__ __forceinline__ int row(int lane, int i) { return kNarrow ? 4 * i + (lane & 3) : lane & 15; }
    static __device__ __forceinline__ f32x4 mma(float w, float x, const f32x4 &acc) {
        if constexpr (kNarrow) return __builtin_amdgcn_mfma_f32_4x4x1f32(w, x, acc, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f32_16x16x4f32(w, x, acc, 0, 0, 0);
    }
    // 4x4 blocks: lanes 16 g .. have summed the contraction elements {16 t + 4 g + e} only
    static __device__ __forceinline__ f32x4 finish(const f32x4 (&acc)[kSets], int lane) {
        if constexpr (kNarrow) {
            f32x4 r;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x[kSets];
#pragma unroll
                for (int i = 0; i < kSets; ++i) x[i] = row_sum(acc[i][e]);
                r[e] = kSets > 1 && (lane & 16) ? x[kSets - 1] : x[0];
            }
            return r;
        }
        return acc[0];
    }
};

// Products of one wavefront: its blocks of 16 outputs against the tile.  Fragments arrive in chunks of C, one
// chunk ahead across block boundaries; begin() requests the first, to be called in front of the barrier or
// the norm that the product has to wait for.
template <int K, int NB, int NW, int TR>
struct F32Product {
    typedef F32Tile<TR> Tile;
    static constexpr int C = K > 256 ? 4 : 8, T = K / 16,  // (8 would spill at K 512)
                        N = NB * T / C;
    static_assert(T % C == 0 && N >= 1, "whole chunks");
    f32x4 ring[2][C];

    static __device__ __forceinline__ const f32x4 *at(const float *w, int i, int wave, int lane) {
        const int nb = wave + NW * (i / (T / C)), t0 = i % (T / C) * C;
        return reinterpret_cast<const f32x4 *>(w) + (static_cast<long>(nb) * T + t0) * 64 + lane;
    }
    __device__ __forceinline__ void begin(const float *w, int wave, int lane) {
        const f32x4 *p = at(w, 0, wave, lane);
#pragma unroll
        for (int j = 0; j < C; ++j) ring[0][j] = p[64 * j];
    }
    // done(block of 16 outputs, acc): acc as F32Tile says
    template <typename Done>
    __device__ __forceinline__ void run(const float *w, const float *tile, int ld, int wave, int lane, Done done) {
        constexpr int S = Tile::kSets;
        const float *src[S];
#pragma unroll
        for (int s = 0; s < S; ++s) src[s] = tile + Tile::row(lane, s) * ld + 4 * (lane >> 4);
        f32x4 acc[S];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (i % (T / C) == 0) {
#pragma unroll
                for (int s = 0; s < S; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            if (i + 1 < N) {
                const f32x4 *p = at(w, i + 1, wave, lane);
#pragma unroll
                for (int j = 0; j < C; ++j) ring[(i + 1) & 1][j] = p[64 * j];
            }
#pragma unroll
            for (int j = 0; j < C; ++j) {
                f32x4 v[S];
#pragma unroll
                for (int s = 0; s < S; ++s) v[s] = *reinterpret_cast<const f32x4 *>(src[s] + 16 * (i % (T / C) * C + j));
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int s = 0; s < S; ++s) acc[s] = Tile::mma(ring[i & 1][j][e], v[s][e], acc[s]);
            }
            __builtin_amdgcn_sched_barrier(0);  // requests further ahead than the ring would be parked in scratch memory
            if (i % (T / C) == T / C - 1) done(wave + NW * (i / (T / C)), Tile::finish(acc, lane));
        }
    }
};

// Rows of `tile` normalised in place, a wavefront per row; `store` (or null): rows of D written there too.
template <int D, int NW, int TR>
__device__ __forceinline__ void f32_norm_rows(float *tile, int ld, const float *gamma, const float *beta, float eps, int wave, int lane,
                                              float *store, long row0, int valid) {
    constexpr int E = D / 64;
    float g[E], b[E];
#pragma unroll
    for (int e = 0; e < E; ++e) g[e] = gamma[64 * e + lane], b[e] = beta[64 * e + lane];
#pragma unroll
    for (int r = wave; r < TR; r += NW) {
        float *row = tile + r * ld;
        float v[E], sum = 0.f, sq = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) sum += v[e] = row[64 * e + lane];
        const float mean = wave_sum(sum) / D;
#pragma unroll
        for (int e = 0; e < E; ++e) sq += (v[e] - mean) * (v[e] - mean);
        const float rstd = rsqrtf(wave_sum(sq) / D + eps);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float n = (v[e] - mean) * rstd * g[e] + b[e];
            row[64 * e + lane] = n;
            if (store && r < valid) store[(row0 + r) * D + 64 * e + lane] = n;
        }
    }
}

template <int D, int F, int TR>
__global__ __launch_bounds__(f32_layer_waves(D) * 64) void f32_layer_kernel(F32LayerParams P) {
    constexpr int NW = f32_layer_waves(D), NT = NW * 64;
    constexpr int LD = D + 4, LF = F + 4, LM = LD > LF ? LD : LF;
    constexpr int NBD = D / 16 / NW, NBF = F / 16 / NW;
    static_assert(NBD * NW * 16 == D && NBF * NW * 16 == F, "whole blocks per wavefront");
    __shared__ __attribute__((aligned(16))) float a[TR * LM];  // attention output, hidden layer, then the layer output
    __shared__ __attribute__((aligned(16))) float s[TR * LD];  // the row sums that are normalised
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const F32Tile<TR> at(lane);
    const int c = at.tok, g = at.sub;
    const long row0 = static_cast<long>(blockIdx.x) * TR;
    const int valid = static_cast<int>(min(static_cast<long>(TR), P.rows - row0));
    // rows past the end read the last one: valid addresses, and nothing of them is stored
    const auto load_rows = [&](float *tile, int ld, const float *src) {
        for (int i = tid; i < TR * (D / 4); i += NT) {
            const int r = i / (D / 4), d = i % (D / 4) * 4;
            *reinterpret_cast<f32x4 *>(tile + r * ld + d) =
                *reinterpret_cast<const f32x4 *>(src + (row0 + (r < valid ? r : valid - 1)) * D + d);
        }
    };
    const auto add_to = [&](float *tile, const float *bias) {  // residual rows in `tile` += outputs (+ bias)
        return [=](int nb, const f32x4 &acc) {
            if (!at.holds) return;
            f32x4 *p = reinterpret_cast<f32x4 *>(tile + c * LD + 16 * nb + 4 * g);
            f32x4 v = *p;
            if (bias) {
                const f32x4 t = *reinterpret_cast<const f32x4 *>(bias + 16 * nb + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += acc[e] + t[e];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += acc[e];
            }
            *p = v;
        };
    };

    F32Product<D, NBD, NW, TR> fo;
    if (P.post) {
        F32Product<D, NBD, NW, TR> o;
        o.begin(P.w_o, wave, lane);
        load_rows(a, LD, P.attn);
        load_rows(s, LD, P.y);
        __syncthreads();
        o.run(P.w_o, a, LD, wave, lane, add_to(s, nullptr));
        F32Product<D, NBF, NW, TR> up;
        up.begin(P.w_1, wave, lane);
        __syncthreads();
        f32_norm_rows<D, NW, TR>(s, LD, P.gamma2, P.beta2, P.eps2, wave, lane, nullptr, 0, 0);
        __syncthreads();
        up.run(P.w_1, s, LD, wave, lane, [&](int nb, const f32x4 &acc) {
            const f32x4 t = *reinterpret_cast<const f32x4 *>(P.b_1 + 16 * nb + 4 * g);
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float h = acc[e] + t[e];
                v[e] = 0.5f * h * (1.f + erff(h * 0.70710678118654752f));
            }
            if (at.holds) *reinterpret_cast<f32x4 *>(a + c * LF + 16 * nb + 4 * g) = v;
        });
        F32Product<F, NBD, NW, TR> down;
        down.begin(P.w_2, wave, lane);
        __syncthreads();
        down.run(P.w_2, a, LF, wave, lane, add_to(s, P.b_2));
        if (P.pre) fo.begin(P.w_fo, wave, lane);
        __syncthreads();
        f32_norm_rows<D, NW, TR>(s, LD, P.gamma3, P.beta3, P.eps3, wave, lane, P.pre ? nullptr : P.out, row0, valid);
        if (!P.pre) return;
    } else {
        fo.begin(P.w_fo, wave, lane);
        load_rows(s, LD, P.x);
    }
    __syncthreads();
    // y = norm1(x + x W_fo^T): every wavefront reads all of s, so the sums go to the other tile
    fo.run(P.w_fo, s, LD, wave, lane, [&](int nb, const f32x4 &acc) {
        if (!at.holds) return;
        const int to = c * LD + 16 * nb + 4 * g;
        f32x4 v = *reinterpret_cast<const f32x4 *>(s + to);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += acc[e];
        *reinterpret_cast<f32x4 *>(a + to) = v;
    });
    F32Product<D, 3 * NBD, NW, TR> qkv;
    qkv.begin(P.w_qkv, wave, lane);
    __syncthreads();
    f32_norm_rows<D, NW, TR>(a, LD, P.gamma1, P.beta1, P.eps1, wave, lane, P.y_next, row0, valid);
    __syncthreads();
    qkv.run(P.w_qkv, a, LD, wave, lane, [&](int nb, const f32x4 &acc) {
        if (at.holds && c < valid) *reinterpret_cast<f32x4 *>(P.qkv + (row0 + c) * (3 * D) + 16 * nb + 4 * g) = acc;
    });
}

}  // namespace artab
