// The layer around the row attention in float32 (gfx950, v_mfma_f32_16x16x4_f32), one launch between two
// attention calls: the tail of a layer (out projection, norm2, feed-forward, norm3) and the head of the next
// (feature stage, norm1, q/k/v projections), or either part alone.
//
// A workgroup takes 16 rows through all products with the activations in LDS; only attention output, y and
// q/k/v touch memory.  Bound: the float32 matrix rate of its compute unit, 256 FLOP per clock: 16 rows of
// d_model 256 are 14.7 MFLOP, 24 us; a launch of up to 4096 rows takes 38 to 40 us, where seven library products
// and the norms and activation between them took 60 (1440 rows) and, from Python, 200 us of host time.  Layouts:
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

constexpr int kF32Rows = 16;

constexpr int f32_layer_waves(int D) { return D == 128 ? 8 : 16; }

// Products of one wavefront: its blocks of 16 outputs against the tile.  Fragments arrive in chunks of C, one
// chunk ahead across block boundaries; begin() requests the first, to be called in front of the barrier or
// the norm that the product has to wait for.
template <int K, int NB, int NW>
struct F32Product {
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
    // done(block of 16 outputs, acc): acc holds outputs 4 g .. 4 g + 3 of token lane % 16
    template <typename Done>
    __device__ __forceinline__ void run(const float *w, const float *tile, int ld, int wave, int lane, Done done) {
        const float *src = tile + (lane & 15) * ld + 4 * (lane >> 4);
        f32x4 acc;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (i % (T / C) == 0) acc = f32x4{0.f, 0.f, 0.f, 0.f};
            if (i + 1 < N) {
                const f32x4 *p = at(w, i + 1, wave, lane);
#pragma unroll
                for (int j = 0; j < C; ++j) ring[(i + 1) & 1][j] = p[64 * j];
            }
#pragma unroll
            for (int j = 0; j < C; ++j) {
                const f32x4 v = *reinterpret_cast<const f32x4 *>(src + 16 * (i % (T / C) * C + j));
#pragma unroll
                for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ring[i & 1][j][e], v[e], acc, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);  // requests further ahead than the ring would be parked in scratch memory
            if (i % (T / C) == T / C - 1) done(wave + NW * (i / (T / C)), acc);
        }
    }
};

// Rows of `tile` normalised in place, a wavefront per row; `store` (or null): rows of D written there too.
template <int D, int NW>
__device__ __forceinline__ void f32_norm_rows(float *tile, int ld, const float *gamma, const float *beta, float eps, int wave, int lane,
                                              float *store, long row0, int valid) {
    constexpr int E = D / 64;
    float g[E], b[E];
#pragma unroll
    for (int e = 0; e < E; ++e) g[e] = gamma[64 * e + lane], b[e] = beta[64 * e + lane];
#pragma unroll
    for (int r = wave; r < kF32Rows; r += NW) {
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

template <int D, int F>
__global__ __launch_bounds__(f32_layer_waves(D) * 64) void f32_layer_kernel(F32LayerParams P) {
    constexpr int NW = f32_layer_waves(D), NT = NW * 64, TR = kF32Rows;
    constexpr int LD = D + 4, LF = F + 4, LM = LD > LF ? LD : LF;
    constexpr int NBD = D / 16 / NW, NBF = F / 16 / NW;
    static_assert(NBD * NW * 16 == D && NBF * NW * 16 == F, "whole blocks per wavefront");
    __shared__ __attribute__((aligned(16))) float a[TR * LM];  // attention output, hidden layer, then the layer output
    __shared__ __attribute__((aligned(16))) float s[TR * LD];  // the row sums that are normalised
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
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

    F32Product<D, NBD, NW> fo;
    if (P.post) {
        F32Product<D, NBD, NW> o;
        o.begin(P.w_o, wave, lane);
        load_rows(a, LD, P.attn);
        load_rows(s, LD, P.y);
        __syncthreads();
        o.run(P.w_o, a, LD, wave, lane, add_to(s, nullptr));
        F32Product<D, NBF, NW> up;
        up.begin(P.w_1, wave, lane);
        __syncthreads();
        f32_norm_rows<D, NW>(s, LD, P.gamma2, P.beta2, P.eps2, wave, lane, nullptr, 0, 0);
        __syncthreads();
        up.run(P.w_1, s, LD, wave, lane, [&](int nb, const f32x4 &acc) {
            const f32x4 t = *reinterpret_cast<const f32x4 *>(P.b_1 + 16 * nb + 4 * g);
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float h = acc[e] + t[e];
                v[e] = 0.5f * h * (1.f + erff(h * 0.70710678118654752f));
            }
            *reinterpret_cast<f32x4 *>(a + c * LF + 16 * nb + 4 * g) = v;
        });
        F32Product<F, NBD, NW> down;
        down.begin(P.w_2, wave, lane);
        __syncthreads();
        down.run(P.w_2, a, LF, wave, lane, add_to(s, P.b_2));
        if (P.pre) fo.begin(P.w_fo, wave, lane);
        __syncthreads();
        f32_norm_rows<D, NW>(s, LD, P.gamma3, P.beta3, P.eps3, wave, lane, P.pre ? nullptr : P.out, row0, valid);
        if (!P.pre) return;
    } else {
        fo.begin(P.w_fo, wave, lane);
        load_rows(s, LD, P.x);
    }
    __syncthreads();
    // y = norm1(x + x W_fo^T): every wavefront reads all of s, so the sums go to the other tile
    fo.run(P.w_fo, s, LD, wave, lane, [&](int nb, const f32x4 &acc) {
        const int at = c * LD + 16 * nb + 4 * g;
        f32x4 v = *reinterpret_cast<const f32x4 *>(s + at);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += acc[e];
        *reinterpret_cast<f32x4 *>(a + at) = v;
    });
    F32Product<D, 3 * NBD, NW> qkv;
    qkv.begin(P.w_qkv, wave, lane);
    __syncthreads();
    f32_norm_rows<D, NW>(a, LD, P.gamma1, P.beta1, P.eps1, wave, lane, P.y_next, row0, valid);
    __syncthreads();
    qkv.run(P.w_qkv, a, LD, wave, lane, [&](int nb, const f32x4 &acc) {
        if (c < valid) *reinterpret_cast<f32x4 *>(P.qkv + (row0 + c) * (3 * D) + 16 * nb + 4 * g) = acc;
    });
}

}  // namespace artab
