// Both ends of a prefill or a density in one launch each (gfx950; bf16, f16, float32): the rows' embedding, and the
// final norm, the mixture head and the log-density of the target rows.
//
// As library calls the ends are 8 launches for a context's embedding, 20 for the targets' and 25 for the densities, over
// tensors that are small or have a column count the library has no good product for (features to D: contraction length 1;
// 3 K outputs): 250 us of host time for any call, and 110 us of a density of 64 x (512 + 2 x 128) rows of 256 against 14 + 9 + 15 of
// these.  Bound: writing the rows; the launch and the chain norm, product, activation, product, mixture.
//
// Everything is float32 between the inputs and the results, but for the operands of the two products, which are of the
// model's type, and the sum of a row's float32 features (64 bits).
#pragma once

#include "common.h"
#include "mfma_flash.h"

namespace artab {

struct EmbedRowsParams {
    const void *x, *y;        // features [B, N, C], values [B, N], any strides (elements)
    long xb, xn, xc, yb, yn;
    int B, N, C, D;
    double one_over_c;
    int pairs;                // 0: context rows [B, N, D]; 1: buffer rows, then target rows [B, 2 N, D]
    const void *w_x, *b_x, *w_y, *b_y;  // [D]
    const void *markers;      // [3, D]: target, context, buffer
    const void *tokens;       // [bs, D]: position token of buffer row n: n % bs
    int bs;
    void *out;
};

// 16 bytes of a row per thread.
template <typename T>
__global__ __launch_bounds__(256) void embed_rows_kernel(EmbedRowsParams P) {
    constexpr int PER = 16 / sizeof(T);
    // (fewer than 2^31 threads: 32-bit divisions)
    const unsigned per_row = P.D / PER, per_batch = P.pairs ? 2 * P.N : P.N, i = blockIdx.x * 256u + threadIdx.x, row = i / per_row;
    if (row >= P.B * per_batch) return;
    const int d = PER * static_cast<int>(i % per_row);
    const long m = row, b = row / per_batch;
    int n = static_cast<int>(row % per_batch);
    const bool target = P.pairs && n >= P.N;
    if (target) n -= P.N;
    const T *const x = static_cast<const T *>(P.x) + b * P.xb + n * P.xn;
    // Eight sums, so that eight loads are on their way at a time; of float32 features in 64 bits.  In 32 bits the rows were further off
    // than the library's reduction leaves them (21 features of mean 3 and deviation 1: 5.9e-8 against 5.1e-8 to 5.9e-8, by its
    // order; 4.6e-8 now, modelled on the CPU).
    typedef std::conditional_t<sizeof(T) == 4, double, float> Sum;
    constexpr int SUMS = 8;
    Sum part[SUMS] = {};
    for (int c0 = 0; c0 < P.C; c0 += SUMS) {
        float t[SUMS];
#pragma unroll
        for (int u = 0; u < SUMS; ++u) t[u] = to_f32(x[min(c0 + u, P.C - 1) * P.xc]);
#pragma unroll
        for (int u = 0; u < SUMS; ++u) part[u] += c0 + u < P.C ? t[u] : 0.f;
    }
    const Sum sum = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
    float mean;
    if constexpr (sizeof(T) == 4) mean = static_cast<float>(sum * P.one_over_c);
    else mean = sum / P.C;
    auto vector = [&](float (&to)[PER], const void *p, long at, auto use) {
        const u32x4 raw = *reinterpret_cast<const u32x4 *>(static_cast<const T *>(p) + at + d);
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            if constexpr (sizeof(T) == 2) {
                const unsigned word = raw[e / 2];
                use(to[e], e & 1 ? unpack_hi<T>(word) : unpack_lo<T>(word));
            } else {
                const unsigned word = raw[e];
                use(to[e], __builtin_bit_cast(float, word));
            }
        }
    };
    const auto take = [](float &a, float t) { a = t; };
    const auto add = [](float &a, float t) { a += t; };
    const auto line = [&](float (&to)[PER], float at, const void *slope, const void *start) {
        float w[PER];
        vector(w, slope, 0, take);
        vector(to, start, 0, take);
#pragma unroll
        for (int e = 0; e < PER; ++e) to[e] = fmaf(at, w[e], to[e]);
    };
    // in the modules' order: (mean w_x + b_x) + (y w_y + b_y) + marker + token
    float v[PER];
    line(v, mean, P.w_x, P.b_x);
    if (!target) {
        float u[PER];
        line(u, to_f32(static_cast<const T *>(P.y)[b * P.yb + n * P.yn]), P.w_y, P.b_y);
#pragma unroll
        for (int e = 0; e < PER; ++e) v[e] += u[e];
    }
    vector(v, P.markers, (target ? 0 : P.pairs ? 2 : 1) * static_cast<long>(P.D), add);
    if (P.pairs && !target) vector(v, P.tokens, static_cast<long>(n % P.bs) * P.D, add);
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (sizeof(T) == 2) o[e] = pack2<T>(v[2 * e], v[2 * e + 1]);
        else o[e] = __builtin_bit_cast(unsigned, v[e]);
    }
    *reinterpret_cast<u32x4 *>(static_cast<T *>(P.out) + m * P.D + d) = o;
}

struct DensityParams {
    const void *x;            // [B, ., D]: target row t of batch entry b at x + b * xb + t * D elements
    long xb;
    const void *norm_g, *norm_b;
    float eps;
    const void *w1, *b1, *w2, *b2;               // [F, D], [F], [3 K, F], [3 K], as the modules have them
    const void *mean_bias, *std_bias, *weight_bias;  // [K]
    int K;
    float std_min;
    const void *y;            // [B, Nt], any strides
    long yb, yn;
    void *out;                // [B, Nt]
    int B, Nt;
};

constexpr int kDensityRows = 16, kDensityWaves = 4, kDensityMaxOut = 128;

// Operands of a product with 16-row and 16-column fragments of 1 KiB: row lane % 16, kPer consecutive elements at kPer (lane / 16).
// A float32 step is four products: step 4 t + e takes the elements {16 t + 4 (lane / 16) + e} of both operands.
template <typename T>
struct DensityOps {
    static constexpr int kStep = 32, kPer = 8;
    static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
        typedef typename MfmaOps<T>::vec vec;
        return MfmaOps<T>::mma16(__builtin_bit_cast(vec, a), __builtin_bit_cast(vec, b), c);
    }
    static __device__ __forceinline__ float gelu(float x) {
        const float tail = normal_tail(x);
        return x * (x > 0.f ? 1.f - tail : tail);
    }
};
template <>
struct DensityOps<float> {
    static constexpr int kStep = 16, kPer = 4;
    static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
        const f32x4 fa = __builtin_bit_cast(f32x4, a), fb = __builtin_bit_cast(f32x4, b);
#pragma unroll
        for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[j], fb[j], c, 0, 0, 0);
        return c;
    }
    static __device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }
};

// 16 target rows per workgroup; the weights are read as the modules have them, 64 bytes of 16 rows per fragment.
template <typename T, int D, int F>
__global__ __launch_bounds__(kDensityWaves * 64) void density_kernel(DensityParams P) {
    typedef DensityOps<T> Ops;
    constexpr int NW = kDensityWaves, TR = kDensityRows, PAD = 16 / sizeof(T), LD = D + PAD, LF = F + PAD, LR = kDensityMaxOut + 4, E = D / 64;
    __shared__ __attribute__((aligned(16))) T zs[TR * LD], hs[TR * LF];
    __shared__ __attribute__((aligned(16))) float raw_s[TR * LR];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, tok = lane & 15, quad = lane >> 4;
    const int rows = P.B * P.Nt, row0 = static_cast<int>(blockIdx.x) * TR;
    // rows past the end are the last one again: valid addresses, and nothing of them is stored
    auto place = [&](int r, long &b, int &t) {
        const unsigned m = min(row0 + r, rows - 1), n = P.Nt;
        b = m / n;
        t = static_cast<int>(m % n);
    };
    {   // the final norm, a wavefront per row
        float x[TR / NW][E], g[E], be[E];
#pragma unroll
        for (int i = 0; i < TR / NW; ++i) {
            long b;
            int t;
            place(wave + NW * i, b, t);
            const T *const src = static_cast<const T *>(P.x) + b * P.xb + static_cast<long>(t) * D;
#pragma unroll
            for (int e = 0; e < E; ++e) x[i][e] = to_f32(src[64 * e + lane]);
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            g[e] = to_f32(static_cast<const T *>(P.norm_g)[64 * e + lane]);
            be[e] = to_f32(static_cast<const T *>(P.norm_b)[64 * e + lane]);
        }
#pragma unroll
        for (int i = 0; i < TR / NW; ++i) {
            float s = 0.f, q = 0.f;
#pragma unroll
            for (int e = 0; e < E; ++e) s += x[i][e];
            const float mean = wave_sum(s) * (1.f / D);
#pragma unroll
            for (int e = 0; e < E; ++e) q = fmaf(x[i][e] - mean, x[i][e] - mean, q);
            const float rstd = rsqrtf(wave_sum(q) * (1.f / D) + P.eps);
#pragma unroll
            for (int e = 0; e < E; ++e) zs[(wave + NW * i) * LD + 64 * e + lane] = from_f32<T>(fmaf((x[i][e] - mean) * rstd, g[e], be[e]));
        }
    }
    __syncthreads();
    // acc[i] = W rows 16 (wave + 4 i) .. of the tile's rows; weight rows past `last` are that one again
    auto product = [&](auto &acc, const T *w, int last, auto k_, const T *tile, int ld) {
        constexpr int K = decltype(k_)::value, KS = K / Ops::kStep, NB = sizeof(acc) / sizeof(acc[0]), AHEAD = 4;
        static_assert(KS % AHEAD == 0, "whole groups of steps");
        const T *row[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            row[i] = w + static_cast<long>(min(16 * (wave + NW * i) + tok, last)) * K + Ops::kPer * quad;
            acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const T *const act = tile + tok * ld + Ops::kPer * quad;
#pragma unroll 2
        for (int k0 = 0; k0 < KS; k0 += AHEAD) {
            u32x4 a[AHEAD][NB];
#pragma unroll
            for (int k = 0; k < AHEAD; ++k)
#pragma unroll
                for (int i = 0; i < NB; ++i) a[k][i] = *reinterpret_cast<const u32x4 *>(row[i] + Ops::kStep * (k0 + k));
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) {
                const u32x4 b = *reinterpret_cast<const u32x4 *>(act + Ops::kStep * (k0 + k));
#pragma unroll
                for (int i = 0; i < NB; ++i) acc[i] = Ops::mma(a[k][i], b, acc[i]);
            }
        }
    };
    {   // h = gelu(z W_1^T + b_1): features 16 nb + 4 quad + e of row tok
        constexpr int NB = F / 16 / NW;
        f32x4 acc[NB];
        product(acc, static_cast<const T *>(P.w1), F - 1, std::integral_constant<int, D>{}, zs, LD);
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int col = 16 * (wave + NW * i) + 4 * quad + e;
                hs[tok * LF + col] = from_f32<T>(Ops::gelu(acc[i][e] + to_f32(static_cast<const T *>(P.b1)[col])));
            }
    }
    __syncthreads();
    // h W_2^T + b_2
    auto outputs = [&](auto nb_) {
        constexpr int NB = decltype(nb_)::value;
        f32x4 acc[NB];
        const int last = 3 * P.K - 1;
        product(acc, static_cast<const T *>(P.w2), last, std::integral_constant<int, F>{}, hs, LF);
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int col = 16 * (wave + NW * i) + 4 * quad + e;
                raw_s[tok * LR + col] = acc[i][e] + to_f32(static_cast<const T *>(P.b2)[min(col, last)]);
            }
    };
    if (3 * P.K <= 16 * NW) outputs(std::integral_constant<int, 1>{});
    else outputs(std::integral_constant<int, kDensityMaxOut / 16 / NW>{});
    __syncthreads();
    // the mixture of a row: 16 lanes, component k on lane k % 16
    const int r = tid >> 4, j = tid & 15;
    long b;
    int t;
    place(r, b, t);
    const float y = to_f32(static_cast<const T *>(P.y)[b * P.yb + t * P.yn]);
    const float *const raw = raw_s + r * LR;
    const auto larger = [](float a, float c) { return a > c || a != a ? a : c; };  // (a NaN stays)
    const auto largest = [&](float x) {
        x = larger(x, row_rotate<8>(x));
        x = larger(x, row_rotate<4>(x));
        x = larger(x, row_rotate<2>(x));
        return larger(x, row_rotate<1>(x));
    };
    const auto total = [](float x) {
        x += row_rotate<8>(x);
        x += row_rotate<4>(x);
        x += row_rotate<2>(x);
        return x + row_rotate<1>(x);
    };
    auto at = [](const void *p, int i) { return to_f32(static_cast<const T *>(p)[i]); };
    // of the component's density without 1 / sqrt(2 pi), weighted as softmax's numerators are: its logarithm
    auto component = [&](int k, float logit, float top_w) {
        const float s_raw = raw[3 * k + 1] + at(P.std_bias, k), soft = s_raw > 20.f ? s_raw : log1pf(expf(s_raw));
        const float s = (soft > 2.f ? 2.f : soft) + P.std_min, z = (y - (raw[3 * k] + at(P.mean_bias, k))) / s;
        return -0.5f * z * z - logf(s) + (logit - top_w);
    };
    float top_w = -INFINITY;
    for (int k = j; k < P.K; k += 16) top_w = larger(raw[3 * k + 2] + at(P.weight_bias, k), top_w);
    top_w = largest(top_w);
    constexpr int kMost = (kDensityMaxOut / 3 + 15) / 16;  // components of a lane
    float sum_w = 0.f, top_c = -INFINITY, c[kMost];
#pragma unroll
    for (int i = 0; i < kMost; ++i) {
        const int k = j + 16 * i;
        c[i] = -INFINITY;
        if (k < P.K) {
            const float logit = raw[3 * k + 2] + at(P.weight_bias, k);
            sum_w += expf(logit - top_w);
            c[i] = component(k, logit, top_w);
        }
        top_c = larger(c[i], top_c);
    }
    sum_w = total(sum_w);
    top_c = largest(top_c);
    if (fabsf(top_c) == INFINITY) top_c = 0.f;
    float sum_c = 0.f;
#pragma unroll
    for (int i = 0; i < kMost; ++i) sum_c += expf(c[i] - top_c);
    sum_c = total(sum_c);
    constexpr float kHalfLog2Pi = 0.91893853320467274f;
    if (j == 0 && row0 + r < rows) static_cast<T *>(P.out)[row0 + r] = from_f32<T>(top_c + logf(sum_c) - logf(sum_w) - kHalfLog2Pi);
}

}  // namespace artab
