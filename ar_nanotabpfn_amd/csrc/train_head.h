// The mixture head of a training step and its loss, forward and backward (gfx950): z -> gelu(z W_1^T + b_1) W_2^T + b_2
// -> means, deviations and log-weights of K normals (model.py:150-246) -> the mean negative log-likelihood of y.
// Float32 parameters, bf16 products with float32 sums; the mixture is float32 throughout.
//
// As modules under autocast this is some 60 launches over [rows, K] tensors, and two weight gradients whose small outputs
// (256 x 128 and 3 K x 256, contracted over 32768 rows) a library runs on seven workgroups.  Here a pass is one kernel
// (the backward one computes the forward again) and the split product of the layers' weight gradients.  Bound by memory;
// tiles as in train_layers.h, the mixture of a row on eight lanes.  32768 rows of 128, K = 20: some 500 us of
// modules -> 23 forward, 41 + 15 backward (their bytes at the rate of a copy: 4 and 17 + 14; the rest is the mixture's
// exponentials and logarithms, in float32, and few tiles to a compute unit as in train_layers.h).
#pragma once

#include "train_layers.h"

namespace artab {

constexpr int kHeadCols = 128;  // width of the raw outputs' gradient: a piece of the weight gradients

struct TrainHead {
    const float *z, *y;        // [M, D], [M] (y: forward)
    float *kept_y;             // [M]: written forward, read backward
    const float *w1, *b1, *w2, *b2;                    // [F, D], [F], [3 K, F], [3 K]
    const float *mean_bias, *std_bias, *weight_bias;   // [K]
    float std_min;
    int K;
    long M;
    bf16_t *packed;            // W_1, W_1^T, W_2, W_2^T
    float *part_loss;          // [gridDim.x] sums of the log-likelihood (forward)
    const float *dloss;        // scalar (backward)
    float *dz;                 // [M, D]
    bf16_t *zb, *h, *du, *draw;  // [M, D], [M, F], [M, F], [M, kHeadCols]
    float *part;               // [gridDim.x][F + kHeadCols]: column sums of d(u), d(raw)
};

template <int D, int F, int NP>
constexpr long train_head_packed_elems() { return 2L * F * (D + NP); }

// the four matrices as operand fragments (train_pack_kernel's layout); rows and columns past 3 K are zero
template <int D, int F, int NP>
__global__ __launch_bounds__(256) void train_head_pack_kernel(TrainHead P) {
    const long piece = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (piece * 8 >= train_head_packed_elems<D, F, NP>()) return;
    constexpr long at[4] = {0, F * D / 8, 2 * F * D / 8, 2 * F * D / 8 + F * NP / 8};
    const int m = piece < at[1] ? 0 : piece < at[2] ? 1 : piece < at[3] ? 2 : 3;
    const long in = piece - at[m];
    const int K = m == 0 ? D : m == 3 ? NP : F;  // contraction of the matrix as it is packed
    const int lane = static_cast<int>(in & 63), frag = static_cast<int>(in >> 6), ks = frag % (K / 32), nb = frag / (K / 32);
    const int n = 16 * nb + (lane & 15), k0 = 32 * ks + 8 * (lane >> 4);
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int row = m & 1 ? k0 + e : n, col = m & 1 ? n : k0 + e;  // element of the master
        f[e] = m < 2 ? P.w1[static_cast<long>(row) * D + col] : row < 3 * P.K ? P.w2[static_cast<long>(row) * F + col] : 0.f;
    }
    const u32x4 v = {pack2<bf16_t>(f[0], f[1]), pack2<bf16_t>(f[2], f[3]), pack2<bf16_t>(f[4], f[5]), pack2<bf16_t>(f[6], f[7])};
    reinterpret_cast<u32x4 *>(P.packed)[piece] = v;
}

// over eight lanes side by side: within fours, then the two fours
template <typename Op>
__device__ __forceinline__ float over_eight(float x, Op op) {
    float o = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1, 0xf, 0xf, true));
    x = op(x, o);
    o = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x4E, 0xf, 0xf, true));
    x = op(x, o);
    o = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x141, 0xf, 0xf, true));
    return op(x, o);
}

template <int D, int F, int NP, bool BACKWARD>
__global__ __launch_bounds__(kTrainWaves * 64, 3) void train_head_kernel(TrainHead P) {
    constexpr int NB = D / 64, NF = F / 64, NR = NP / 64, LD = D + 8, LF = F + 8, LR = NP + 4, LG = kHeadCols + 8, NS = F + kHeadCols;
    __shared__ __attribute__((aligned(16))) bf16_t zs[kTrainRows * LD], hs[kTrainRows * LF];
    __shared__ __attribute__((aligned(16))) float raw_s[kTrainRows * LR];
    __shared__ __attribute__((aligned(16))) bf16_t gs[BACKWARD ? kTrainRows * LG : 8];
    __shared__ __attribute__((aligned(16))) float sums[BACKWARD ? NS : 4];
    const int K3 = 3 * P.K;
    if constexpr (BACKWARD) {
        for (int i = threadIdx.x; i < NS; i += kTrainWaves * 64) sums[i] = 0.f;
        for (int i = threadIdx.x; i < kTrainRows * LG / 8; i += kTrainWaves * 64) reinterpret_cast<u32x4 *>(gs)[i] = u32x4{0u, 0u, 0u, 0u};
    }
    const float grad = BACKWARD ? -*P.dloss / static_cast<float>(P.M) : 0.f;  // of a row's log-likelihood
    float sum_ll = 0.f;
    const long tiles = (P.M + kTrainRows - 1) / kTrainRows;
    for (long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const TrainLane L(tile, P.M);
        const bf16_t *const packed = train_opaque(P.packed);
        const bf16_t *const w1 = packed, *const w1t = w1 + F * D, *const w2 = w1t + F * D, *const w2t = w2 + F * NP;
        {
            f32x4 z[NB][2];
            train_load<D>(z, P.z, L);
            train_to_lds(zs, LD, z, L);
        }
        __syncthreads();
        f32x4 u[NF][2];  // gelu'(u), backward
        {
            f32x4 h[NF][2];
            train_product<NF, D / 32>(h, zs, LD, w1, 0, L);
#pragma unroll
            for (int b = 0; b < NF; ++b) {
                const f32x4 bias = *reinterpret_cast<const f32x4 *>(P.b1 + L.col(b));
#pragma unroll
                for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float hv, dv;
                        train_gelu(h[b][tb][e] + bias[e], hv, dv);
                        h[b][tb][e] = hv;
                        u[b][tb][e] = dv;
                    }
            }
            train_to_lds(hs, LF, h, L);
        }
        __syncthreads();
        if constexpr (BACKWARD) {
            train_unstage<D>(P.zb, zs, LD, L);
            train_unstage<F>(P.h, hs, LF, L);
        }
        {
            f32x4 raw[NR][2];
            train_product<NR, F / 32>(raw, hs, LF, w2, 0, L);
#pragma unroll
            for (int b = 0; b < NR; ++b) {
                f32x4 bias;
#pragma unroll
                for (int e = 0; e < 4; ++e) bias[e] = L.col(b) + e < K3 ? P.b2[L.col(b) + e] : 0.f;
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) *reinterpret_cast<f32x4 *>(raw_s + (16 * tb + L.tok) * LR + L.col(b)) = raw[b][tb] + bias;
            }
        }
        __syncthreads();
        {   // the mixture of a row: eight lanes, component k on lane k % 8
            const int tid = opaque(threadIdx.x), row = tid >> 3, j = tid & 7;
            const bool live = L.row0 + row < P.M;
            const float y = (BACKWARD ? P.kept_y : P.y)[min(L.row0 + row, P.M - 1)];
            if (!BACKWARD && live && j == 0) P.kept_y[L.row0 + row] = y;
            float *const r = raw_s + row * LR;
            const auto add = [](float a, float b) { return a + b; };
            const auto larger = [](float a, float b) { return a > b || a != a ? a : b; };  // (a NaN stays)
            struct Component {
                float t, s, logit, slope;
            };
            auto component = [&](int k) {
                Component c;
                const float x = r[3 * k + 1] + P.std_bias[k], e = expf(x), soft = x > 20.f ? x : log1pf(e);
                c.slope = soft > 2.f ? 0.f : x > 20.f ? 1.f : e / (1.f + e);  // of the deviation: softplus, not above 2
                c.s = (soft > 2.f ? 2.f : soft) + P.std_min;
                c.t = (y - (r[3 * k] + P.mean_bias[k])) / c.s;
                c.logit = r[3 * k + 2] + P.weight_bias[k];
                return c;
            };
            float top_w = -INFINITY;
            for (int k = j; k < P.K; k += 8) top_w = larger(r[3 * k + 2] + P.weight_bias[k], top_w);
            top_w = over_eight(top_w, larger);
            float sum_w = 0.f, top_c = -INFINITY;
            for (int k = j; k < P.K; k += 8) {
                const Component c = component(k);
                sum_w += expf(c.logit - top_w);
                top_c = larger(-0.5f * c.t * c.t - logf(c.s) + (c.logit - top_w), top_c);
            }
            sum_w = over_eight(sum_w, add);
            top_c = over_eight(top_c, larger);
            if (fabsf(top_c) == INFINITY) top_c = 0.f;
            float sum_c = 0.f;
            for (int k = j; k < P.K; k += 8) {
                const Component c = component(k);
                sum_c += expf(-0.5f * c.t * c.t - logf(c.s) + (c.logit - top_w) - top_c);
            }
            sum_c = over_eight(sum_c, add);
            if constexpr (!BACKWARD) {
                constexpr float kHalfLog2Pi = 0.91893853320467274f;
                if (live && j == 0) sum_ll += top_c + logf(sum_c) - logf(sum_w) - kHalfLog2Pi;
            } else {
                bf16_t *const g = gs + row * LG;
                const float gr = live ? grad : 0.f, inv_c = 1.f / sum_c, inv_w = 1.f / sum_w;
                for (int k = j; k < P.K; k += 8) {  // (only this lane reads component k of the row)
                    const Component c = component(k);
                    const float weight = expf(c.logit - top_w);
                    const float mine = expf(-0.5f * c.t * c.t - logf(c.s) + (c.logit - top_w) - top_c) * inv_c;
                    const float d[3] = {gr * mine * (c.t / c.s), gr * mine * ((c.t * c.t - 1.f) / c.s) * c.slope, gr * (mine - weight * inv_w)};
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        const float v = live ? d[i] : 0.f;
                        r[3 * k + i] = v;
                        g[3 * k + i] = from_f32<bf16_t>(v);
                    }
                }
            }
        }
        if constexpr (BACKWARD) {
            __syncthreads();
            if (static_cast<int>(threadIdx.x) < K3) {  // (K3 <= kHeadCols < threads)
                float s = 0.f;
#pragma unroll 8
                for (int row = 0; row < kTrainRows; ++row) s += raw_s[row * LR + threadIdx.x];
                sums[F + threadIdx.x] += s;
            }
            train_unstage<kHeadCols>(P.draw, gs, LG, L);
            f32x4 d[NF][2];
            train_product<NF, NP / 32>(d, gs, LG, w2t, 0, L);
#pragma unroll
            for (int b = 0; b < NF; ++b) {
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) d[b][tb] *= u[b][tb];
                train_col_add(sums, d[b][0] + d[b][1], L.col(b), L);
            }
            train_to_lds(hs, LF, d, L);
            __syncthreads();
            train_unstage<F>(P.du, hs, LF, L);
            f32x4 dz[NB][2];
            train_product<NB, F / 32>(dz, hs, LF, w1t, 0, L);
            train_store<D>(P.dz, dz, L);
        }
        __syncthreads();
    }
    if constexpr (BACKWARD) {
        for (int i = threadIdx.x; i < NS; i += kTrainWaves * 64) P.part[static_cast<long>(blockIdx.x) * NS + i] = sums[i];
    } else {
        sum_ll = wave_sum(sum_ll);
        if ((threadIdx.x & 63) == 0) raw_s[threadIdx.x >> 6] = sum_ll;
        __syncthreads();
        if (threadIdx.x == 0) P.part_loss[blockIdx.x] = (raw_s[0] + raw_s[1]) + (raw_s[2] + raw_s[3]);
    }
}

// loss = -(sum of the workgroups' sums) / rows, in one order
static __global__ __launch_bounds__(256) void train_head_loss_kernel(const float *part, int groups, long M, float *loss) {
    __shared__ float acc[4];
    float s = 0.f;
    for (int i = threadIdx.x; i < groups; i += 256) s += part[i];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) acc[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) *loss = -((acc[0] + acc[1]) + (acc[2] + acc[3])) / static_cast<float>(M);
}

}  // namespace artab
