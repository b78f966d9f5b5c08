// A whole autoregressive sampling run in one launch: every workgroup takes a few trajectories through
// all steps and all layers (gfx950; bf16 / f16 / float32; head_dim 32).
//
// Given the cached context, trajectories do not depend on each other: the only thing a decode step
// of one trajectory needs from the rest of the chip is the weights and the context's keys and values,
// both constant.  A step that is cut into launches (context pass, buffer pass, layer boundary, tail)
// pays 30-40 us per layer for them whatever the size of the problem; here a layer costs what one
// compute unit needs to stream its weights and keys through (64 B per clock from the L2) plus nine
// workgroup barriers.  What bounds it: that stream.  Measured per layer at d_model 128 / 256 / 512
// (short contexts): see trajectory_decode_applies() in trajectory_launch.hip, which holds the rule
// for when the launches of the other route, which spread one layer over the whole chip, are faster.
//
// Rows.  A workgroup owns G <= 8 trajectories; token row 2 g is trajectory g's buffer row of the step
// (the value drawn last), row 2 g + 1 its target row: 16 rows = one MFMA column block.  Products are
// transposed as in fused_layer.h (C^T[n, m] = sum_k W[n, k] A[m, k] on 16x16 tiles): weights are the
// A operand, the 16-row activation tile in LDS is the B operand; lane l holds token l % 16 and four
// consecutive features 4 (l / 16) + r of every 16-feature block.
//
// Weights.  Each wavefront has a tape: the 1 KiB operand fragments it will consume, in the order it
// consumes them, layer after layer, then the head's; the first kRing of them are repeated behind the
// end.  A ring of kRing fragments in registers is always kRing ahead, across products, barriers,
// layers and steps: after a fragment has been multiplied its registers receive the one kRing further
// on.  All ring positions are compile-time constants (the fragments of a layer are a multiple of
// kRing).
//
// Attention.  One wavefront owns a head (or half of a head's keys at 4 heads, two heads in turn at
// 16); the columns of S^T = K Q^T are the 16 token rows.  Keys come in blocks: the shared context
// serves every column, a trajectory's own rows only its two columns (the others are masked, their
// state does not change), so no merge of partial results is needed.  The rows of this step that
// have just been projected are keys too: one last block straight from LDS, masked to (row 2 g,
// columns 2 g and 2 g + 1).  Softmax is online in float32 with scale * log2(e) folded into the
// queries and rounded to the model's type, probabilities are rounded to the model's type: the
// rounding model of the other kernels.
#pragma once

#include "common.h"
#include "mfma_flash.h"

namespace artab {

constexpr int kTrajRows = 16;   // token rows of a workgroup
constexpr int kTrajMax = 8;     // trajectories of a workgroup
constexpr int kTrajWaves = 8;
constexpr int kTrajMaxMix = 21; // 3 K outputs of the head fit 64 columns
constexpr int kTrajHeadOut = 64;

struct TrajectoryParams {
    const char *tape;        // kTrajWaves tapes of `tape_stride` bytes
    long tape_stride;
    const void *vecs;        // [n_layers][8][max(D, F)]: g1, b1, g2, b2, bias_1, g3, b3, bias_2
    const unsigned long long *kv;  // [n_layers][4] addresses: context K, V; trajectory K, V
    int n_layers;
    // shared context: rows [0, n_ctx) of [H, ctx_rows, 32]; own_base = 0.  Per-trajectory context:
    // n_ctx = 0 and the trajectory's cache holds its context in rows [0, own_base).
    int n_ctx, ctx_rows, own_base;
    int own_rows;            // rows of a trajectory's cache [B, H, own_rows, 32]
    int park_target;         // leave the last target row's K/V behind the committed rows
    float qscale;            // softmax scale * log2(e)
    float eps1, eps2, eps3;
    const void *norm_g, *norm_b; float eps_out;
    const void *b_h1;        // [F]
    const void *b_h2;        // [64], zeros behind 3 K
    const void *mix;         // [3][K]: mean, std, weight biases
    int K; float std_min, std_max;
    const float *rand_u;     // [Nt, B]
    const void *rand_n;      // [Nt, B] in float32 or the model's type
    int rand_n_f32;
    const void *x_mean;      // [B, Nt]
    const void *w_x, *b_x, *w_y, *b_y;  // [D]
    const void *markers;     // [3, D]: target, context, buffer
    const void *ar_tokens; int bs;      // [bs, D]
    void *preds;             // [B, Nt]
    int B, Nt, G;
};

// One 1 KiB fragment of each operand: 16-bit types one 16x16x32 product, float32 four 16x16x4 ones
// (element j of every lane's four makes the contraction indices 4 s + j of both operands).
template <typename T>
struct TrajOps {
    static constexpr int kStep = 32, kPer = 8;
    static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
        typedef typename MfmaOps<T>::vec vec;
        return MfmaOps<T>::mma16(__builtin_bit_cast(vec, a), __builtin_bit_cast(vec, b), c);
    }
};
template <>
struct TrajOps<float> {
    static constexpr int kStep = 16, kPer = 4;
    static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
        const f32x4 fa = __builtin_bit_cast(f32x4, a), fb = __builtin_bit_cast(f32x4, b);
#pragma unroll
        for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[j], fb[j], c, 0, 0, 0);
        return c;
    }
};

template <typename T>
__device__ __forceinline__ void traj_load4(const T *p, float (&f)[4]) {
    if constexpr (sizeof(T) == 2) {
        const u32x2 r = *reinterpret_cast<const u32x2 *>(p);
        f[0] = unpack_lo<T>(r[0]); f[1] = unpack_hi<T>(r[0]); f[2] = unpack_lo<T>(r[1]); f[3] = unpack_hi<T>(r[1]);
    } else {
        const f32x4 r = *reinterpret_cast<const f32x4 *>(p);
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = r[e];
    }
}
template <typename T>
__device__ __forceinline__ void traj_store4(T *p, const float (&f)[4]) {
    if constexpr (sizeof(T) == 2) {
        const u32x2 r = {pack2<T>(f[0], f[1]), pack2<T>(f[2], f[3])};
        *reinterpret_cast<u32x2 *>(p) = r;
    } else {
        const f32x4 r = {f[0], f[1], f[2], f[3]};
        *reinterpret_cast<f32x4 *>(p) = r;
    }
}

// A lane's entries of NB parameter vectors' 16-feature blocks, as they come from memory (converted where
// they are used, so that nothing waits for them where they are requested).
template <typename T, int NB>
struct TrajCols {
    typedef typename std::conditional<sizeof(T) == 2, u32x2, f32x4>::type raw_t;
    raw_t raw[NB];
    __device__ __forceinline__ void load(const T *vec, int wave, int s4) {
#pragma unroll
        for (int b = 0; b < NB; ++b) raw[b] = *reinterpret_cast<const raw_t *>(vec + 16 * (wave + kTrajWaves * b) + 4 * s4);
    }
    __device__ __forceinline__ void get(int b, float (&f)[4]) const {
        if constexpr (sizeof(T) == 2) {
            f[0] = unpack_lo<T>(raw[b][0]); f[1] = unpack_hi<T>(raw[b][0]);
            f[2] = unpack_lo<T>(raw[b][1]); f[3] = unpack_hi<T>(raw[b][1]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = raw[b][e];
        }
    }
};

// Sizes shared by the kernel and the host code that writes the tapes.
template <typename T, int D, int F>
struct TrajShape {
    static constexpr int NW = kTrajWaves;
    static constexpr int KD = D / TrajOps<T>::kStep, KF = F / TrajOps<T>::kStep;  // contraction steps
    static constexpr int ND = D / 16 / NW, NF = F / 16 / NW;                      // 16-feature blocks per wavefront
    static constexpr int kFo = ND * KD, kQkv = 3 * ND * KD, kO = ND * KD, k1 = NF * KD, k2 = ND * KF;
    static constexpr int kLayer = kFo + kQkv + kO + k1 + k2;
    static constexpr int ring() {
        for (int r = 16; r > 1; --r)
            if (kLayer % r == 0) return r;
        return 1;
    }
    static constexpr int kRing = ring();
    static constexpr int kH1 = NF * KD, kH2 = KF;  // the head's second layer: 64 outputs, wavefronts 0 .. 3
    static constexpr int kHead = (kH1 + kH2 + kRing - 1) / kRing * kRing;
    static_assert(ND >= 1 && NF >= 1 && D % (16 * NW) == 0 && F % (16 * NW) == 0, "whole blocks per wavefront");
};

// Copies one matrix W [N, K] into the tapes: wavefront w's blocks are w, w + 8, ... (n_blocks of them
// in all, zeros where N has none), fragment (step, block) at `first` + step * stride + offset + block.
template <typename T>
__global__ void trajectory_tape_kernel(const T *w, char *tape, long tape_stride, int N, int K, int per_wave, int first,
                                       int stride, int offset) {
    constexpr int kStep = TrajOps<T>::kStep, kPer = TrajOps<T>::kPer;
    const int steps = K / kStep;
    const long frag = static_cast<long>(blockIdx.x) * (blockDim.x / 64) + threadIdx.x / 64;
    const int lane = threadIdx.x & 63;
    if (frag >= static_cast<long>(kTrajWaves) * per_wave * steps) return;
    const int b = static_cast<int>(frag % per_wave), ks = static_cast<int>(frag / per_wave % steps),
              wave = static_cast<int>(frag / per_wave / steps);
    const int row = 16 * (wave + kTrajWaves * b) + (lane & 15);
    u32x4 v = {0u, 0u, 0u, 0u};
    if (row < N) v = *reinterpret_cast<const u32x4 *>(w + static_cast<long>(row) * K + kStep * ks + kPer * (lane >> 4));
    *reinterpret_cast<u32x4 *>(tape + wave * tape_stride + (static_cast<long>(first) + ks * stride + offset + b) * 1024 +
                               16 * lane) = v;
}
template <typename T, int D, int F>
__global__ __launch_bounds__(kTrajWaves * 64) void trajectory_decode_kernel(TrajectoryParams P) {
    typedef TrajOps<T> Ops;
    typedef TrajShape<T, D, F> S;
    constexpr int NW = kTrajWaves, NT = NW * 64, DH = 32, H = D / DH;
    constexpr bool k16 = sizeof(T) == 2;
    constexpr int LD = D + (k16 ? 8 : 4), LF = F + (k16 ? 8 : 4);  // row strides: 16 bytes off a multiple of 128
    constexpr int VW = D > F ? D : F;
    constexpr int BK = k16 ? 32 : 16;      // keys per block
    constexpr int NP = NW > H ? NW / H : 1;  // wavefronts per head
    constexpr int HPW = H > NW ? H / NW : 1; // heads per wavefront, in turn
    constexpr int VPAD = DH + 16;

    __shared__ __attribute__((aligned(16))) T xs[kTrajRows * LD];   // layer input; attention output
    __shared__ __attribute__((aligned(16))) T ys[kTrajRows * LD];   // normed feature stage, then x1; z of the head
    constexpr int QKV = 3 * kTrajRows * LD, HID = kTrajRows * LF;
    __shared__ __attribute__((aligned(16))) T qkv[QKV > HID ? QKV : HID];  // q, k, v of the step; hidden layer
    T *const qs = qkv, *const kn = qkv + kTrajRows * LD, *const vn = qkv + 2 * kTrajRows * LD, *const hs = qkv;
    __shared__ __attribute__((aligned(16))) T v_lds[k16 ? NW * BK * VPAD : 8];
    __shared__ float red_a[NW * kTrajRows], red_b[NW * kTrajRows];
    __shared__ float part_o[NP > 1 ? NW * kTrajRows * DH : 1];
    __shared__ float part_m[NP > 1 ? NW * kTrajRows : 1], part_l[NP > 1 ? NW * kTrajRows : 1];
    __shared__ float raw_s[kTrajRows][kTrajHeadOut + 1];
    __shared__ float y_s[kTrajMax], x_s[2 * kTrajMax];
    // what the end of every step needs: norm g and b, x and y embedding w and b, markers target and
    // buffer; the head's biases; the position token of the coming step
    __shared__ __attribute__((aligned(16))) T cst[8 * D + F + kTrajHeadOut + 3 * kTrajMaxMix + 1], tok_s[D];
    T *const c_ng = cst, *const c_nb = cst + D, *const c_wx = cst + 2 * D, *const c_bx = cst + 3 * D, *const c_wy = cst + 4 * D,
             *const c_by = cst + 5 * D, *const c_mt = cst + 6 * D, *const c_mb = cst + 7 * D, *const c_b1 = cst + 8 * D,
             *const c_b2 = c_b1 + F, *const c_mix = c_b2 + kTrajHeadOut;

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int tok = lane & 15, s4 = lane >> 4;
    const long b0 = static_cast<long>(blockIdx.x) * P.G;
    const int valid = static_cast<int>(min(static_cast<long>(P.G), P.B - b0));

    // ---- the weight tape
    u32x4 ring[S::kRing];
    const char *next = P.tape + wave * P.tape_stride + 16 * lane;
#pragma unroll
    for (int i = 0; i < S::kRing; ++i) {
        ring[i] = *reinterpret_cast<const u32x4 *>(next);
        next += 1024;
    }
    // acc[b] += W_b A^T over KS steps of NB blocks; fragments pos .. pos + KS * NB - 1 of the tape section
    auto product = [&](auto pos_, auto ks_, auto &acc, const T *act, int ld) {
        constexpr int POS = decltype(pos_)::value, KS = decltype(ks_)::value;
        constexpr int NB = sizeof(acc) / sizeof(acc[0]);
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const u32x4 bf = *reinterpret_cast<const u32x4 *>(act + tok * ld + Ops::kStep * ks + Ops::kPer * s4);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                constexpr int R = S::kRing;
                const int slot = (POS + ks * NB + b) % R;
                acc[b] = Ops::mma(ring[slot], bf, acc[b]);
                ring[slot] = *reinterpret_cast<const u32x4 *>(next);
                next += 1024;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // LayerNorm of v (this lane's features of its token row) into dst
    auto norm_store = [&](auto &v, const auto &gam, const auto &bet, float eps, T *dst) {
        constexpr int NB = sizeof(v) / sizeof(v[0]);
        constexpr float kLocal = NB * 16;
        float sum = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) sum += v[b][e];
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        const float lmean = sum * (1.f / kLocal);
        float q = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float d = v[b][e] - lmean;
                q += d * d;
            }
        q += __shfl_xor(q, 16, 64);
        q += __shfl_xor(q, 32, 64);
        if (s4 == 0) {
            red_a[wave * kTrajRows + tok] = lmean;
            red_b[wave * kTrajRows + tok] = q;
        }
        __syncthreads();
        float lm[NW], tot = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            lm[w] = red_a[w * kTrajRows + tok];
            tot += lm[w];
        }
        const float mean = tot * (1.f / NW);
        float m2 = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float d = lm[w] - mean;
            m2 += red_b[w * kTrajRows + tok] + kLocal * d * d;
        }
        const float rstd = rsqrtf(m2 / D + eps);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float o[4], g[4], be[4];
            gam.get(b, g);
            bet.get(b, be);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (v[b][e] - mean) * rstd * g[e] + be[e];
            traj_store4<T>(dst + tok * LD + 16 * (wave + NW * b) + 4 * s4, o);
        }
        __syncthreads();
    };
    auto gelu = [](float t) { return 0.5f * t * (1.f + erff(t * 0.70710678118654752f)); };

    // ---- attention of this wavefront's head(s): committed rows, then the rows of this step
    const int part = wave / H;  // (only with NP > 1)
    T *const vt = v_lds + (k16 ? wave * BK * VPAD : 0);
    auto attention = [&](const T *kc, const T *vc, const T *ko, const T *vo, int t) {
        const int n_own = P.own_base + (t > 0 ? t - 1 : 0);  // rows of a trajectory's cache
        const int nb_ctx = (P.n_ctx + BK - 1) / BK, nb_own = (n_own + BK - 1) / BK;
        const int n_blocks = nb_ctx + valid * nb_own;
        for (int hh = 0; hh < HPW; ++hh) {
            const int h = NP > 1 ? wave % H : wave + NW * hh;
            u32x4 qf[k16 ? 1 : 2];
#pragma unroll
            for (int x = 0; x < (k16 ? 1 : 2); ++x)
                qf[x] = *reinterpret_cast<const u32x4 *>(qs + tok * LD + DH * h + Ops::kStep * x + Ops::kPer * s4);
            f32x4 o_acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
            float m_run = -1e30f, l_run = 0.f;
            // one block of keys as it comes from memory: K in operand order; V as 16-byte pieces of the
            // row-major tile (16-bit) or as the operand of the second product (float32)
            struct Block {
                u32x4 k[2];
                u32x4 v[2];
            };
            // keys [row0, row0 + BK) of block i: where they start, how many there are, whose they are
            auto locate = [&](int i, const T *&kp, const T *&vp, int &row0, int &n, int &g) {
                if (i < nb_ctx) {
                    g = -1;
                    row0 = i * BK;
                    n = P.n_ctx;
                    const long at = static_cast<long>(h) * P.ctx_rows * DH;
                    kp = kc + at;
                    vp = vc + at;
                } else {
                    int j = i - nb_ctx;
                    g = 0;
                    while (j >= nb_own) {
                        j -= nb_own;
                        ++g;
                    }
                    row0 = j * BK;
                    n = n_own;
                    const long at = ((b0 + g) * H + h) * P.own_rows * DH;
                    kp = ko + at;
                    vp = vo + at;
                }
            };
            auto fetch = [&](int i, Block &r) {
                const T *kp, *vp;
                int row0, n, g;
                locate(i, kp, vp, row0, n, g);
                if constexpr (k16) {
#pragma unroll
                    for (int x = 0; x < 2; ++x)
                        r.k[x] = *reinterpret_cast<const u32x4 *>(kp + static_cast<long>(min(row0 + 16 * x + tok, n - 1)) * DH + 8 * s4);
#pragma unroll
                    for (int x = 0; x < 2; ++x) {
                        const int p = lane + 64 * x;
                        r.v[x] = *reinterpret_cast<const u32x4 *>(vp + static_cast<long>(min(row0 + p / 4, n - 1)) * DH + 8 * (p % 4));
                    }
                } else {
                    const T *kr = kp + static_cast<long>(min(row0 + tok, n - 1)) * DH + 4 * s4;
#pragma unroll
                    for (int x = 0; x < 2; ++x) r.k[x] = *reinterpret_cast<const u32x4 *>(kr + 16 * x);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const T *vr = vp + static_cast<long>(min(row0 + 4 * s4 + j, n - 1)) * DH + tok;
                        r.v[0][j] = __builtin_bit_cast(unsigned, vr[0]);
                        r.v[1][j] = __builtin_bit_cast(unsigned, vr[16]);
                    }
                }
            };
            // softmax bookkeeping of a block of scores (lane: keys 4 s + r of each 16-key half, its token)
            auto fold = [&](auto &sc, auto &pb) {
                constexpr int NX = sizeof(sc) / sizeof(sc[0]);
                float tmax = sc[0][0];
#pragma unroll
                for (int x = 0; x < NX; ++x)
#pragma unroll
                    for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, sc[x][r]);
                tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
                tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
                const float m_new = fmaxf(m_run, tmax);
                const float alpha = fast_exp2(m_run - m_new);
                if (__any(alpha != 1.f)) {
                    l_run *= alpha;
#pragma unroll
                    for (int db = 0; db < 2; ++db)
#pragma unroll
                        for (int r = 0; r < 4; ++r) o_acc[db][r] *= alpha;
                }
                m_run = m_new;
#pragma unroll
                for (int x = 0; x < NX; ++x)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float p = fast_exp2(sc[x][r] - m_new);
                        l_run += p;
                        pb[x][r] = p;
                    }
            };
            auto compute = [&](int i, const Block &r) {
                const T *kp, *vp;
                int row0, n, g;
                locate(i, kp, vp, row0, n, g);
                constexpr int NX = BK / 16;
                f32x4 sc[NX];
                if constexpr (k16) {
#pragma unroll
                    for (int x = 0; x < 2; ++x) {
                        const int p = lane + 64 * x;
                        *reinterpret_cast<u32x4 *>(vt + (p / 4) * VPAD + 8 * (p % 4)) = r.v[x];
                    }
#pragma unroll
                    for (int x = 0; x < 2; ++x) sc[x] = Ops::mma(r.k[x], qf[0], f32x4{0.f, 0.f, 0.f, 0.f});
                } else {
                    sc[0] = Ops::mma(r.k[0], qf[0], f32x4{0.f, 0.f, 0.f, 0.f});
                    sc[0] = Ops::mma(r.k[1], qf[1], sc[0]);
                }
                if (row0 + BK > n || g >= 0) {
                    const bool mine = g < 0 || (tok >> 1) == g;
#pragma unroll
                    for (int x = 0; x < NX; ++x)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (!mine || row0 + 16 * x + 4 * s4 + e >= n) sc[x][e] = -INFINITY;
                }
                float pb[NX][4];
                fold(sc, pb);
                if constexpr (k16) {
                    const u32x4 pv = {pack2<T>(pb[0][0], pb[0][1]), pack2<T>(pb[0][2], pb[0][3]),
                                      pack2<T>(pb[1][0], pb[1][1]), pack2<T>(pb[1][2], pb[1][3])};
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int db = 0; db < 2; ++db) {
                        const T *a = vt + (4 * s4 + (tok >> 2)) * VPAD + 16 * db + 4 * (tok & 3);
                        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(a));
                        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(a + 16 * VPAD));
                        typedef short s16x8 __attribute__((ext_vector_type(8)));
                        const s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                        o_acc[db] = Ops::mma(__builtin_bit_cast(u32x4, both), pv, o_acc[db]);
                    }
                    __builtin_amdgcn_wave_barrier();
                } else {
                    const u32x4 pv = {__builtin_bit_cast(unsigned, pb[0][0]), __builtin_bit_cast(unsigned, pb[0][1]),
                                      __builtin_bit_cast(unsigned, pb[0][2]), __builtin_bit_cast(unsigned, pb[0][3])};
#pragma unroll
                    for (int db = 0; db < 2; ++db) o_acc[db] = Ops::mma(r.v[db], pv, o_acc[db]);
                }
            };
            Block r0, r1, r2;
            const int first = NP > 1 ? part : 0;
            if (first < n_blocks) fetch(first, r0);
            if (first + NP < n_blocks) fetch(first + NP, r1);
            for (int i = first; i < n_blocks;) {
                if (i + 2 * NP < n_blocks) fetch(i + 2 * NP, r2);
                compute(i, r0);
                if ((i += NP) >= n_blocks) break;
                if (i + 2 * NP < n_blocks) fetch(i + 2 * NP, r0);
                compute(i, r1);
                if ((i += NP) >= n_blocks) break;
                if (i + 2 * NP < n_blocks) fetch(i + 2 * NP, r1);
                compute(i, r2);
                i += NP;
            }
            if (t > 0 && (NP == 1 || part == 0)) {  // the buffer rows of this step
                f32x4 sc[1];
                if constexpr (k16) {
                    const u32x4 kf = *reinterpret_cast<const u32x4 *>(kn + tok * LD + DH * h + 8 * s4);
                    sc[0] = Ops::mma(kf, qf[0], f32x4{0.f, 0.f, 0.f, 0.f});
                } else {
                    const T *kr = kn + tok * LD + DH * h + 4 * s4;
                    sc[0] = Ops::mma(*reinterpret_cast<const u32x4 *>(kr), qf[0], f32x4{0.f, 0.f, 0.f, 0.f});
                    sc[0] = Ops::mma(*reinterpret_cast<const u32x4 *>(kr + 16), qf[1], sc[0]);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (4 * s4 + e != (tok & ~1)) sc[0][e] = -INFINITY;
                float pb[1][4];
                fold(sc, pb);
                if constexpr (k16) {
                    const u32x4 pv = {pack2<T>(pb[0][0], pb[0][1]), pack2<T>(pb[0][2], pb[0][3]), 0u, 0u};
#pragma unroll
                    for (int db = 0; db < 2; ++db) {
                        const T *a = vn + (4 * s4 + (tok >> 2)) * LD + DH * h + 16 * db + 4 * (tok & 3);
                        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(a));
                        typedef short s16x8 __attribute__((ext_vector_type(8)));
                        const s16x8 both = {lo[0], lo[1], lo[2], lo[3], 0, 0, 0, 0};
                        o_acc[db] = Ops::mma(__builtin_bit_cast(u32x4, both), pv, o_acc[db]);
                    }
                } else {
#pragma unroll
                    for (int db = 0; db < 2; ++db) {
                        u32x4 vf, pv;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            vf[j] = __builtin_bit_cast(unsigned, vn[(4 * s4 + j) * LD + DH * h + 16 * db + tok]);
                            pv[j] = __builtin_bit_cast(unsigned, pb[0][j]);
                        }
                        o_acc[db] = Ops::mma(vf, pv, o_acc[db]);
                    }
                }
            }
            float l_tot = l_run + __shfl_xor(l_run, 16, 64);
            l_tot += __shfl_xor(l_tot, 32, 64);
            if constexpr (NP > 1) {  // the other wavefronts' keys of this head
                if (part > 0) {
                    if (s4 == 0) {
                        part_m[wave * kTrajRows + tok] = m_run;
                        part_l[wave * kTrajRows + tok] = l_tot;
                    }
#pragma unroll
                    for (int db = 0; db < 2; ++db)
                        *reinterpret_cast<f32x4 *>(part_o + (wave * kTrajRows + tok) * DH + 16 * db + 4 * s4) = o_acc[db];
                }
                __syncthreads();
                if (part == 0) {
#pragma unroll
                    for (int p = 1; p < NP; ++p) {
                        const int w = wave + p * H;
                        const float m2 = part_m[w * kTrajRows + tok], l2 = part_l[w * kTrajRows + tok];
                        const float m_new = fmaxf(m_run, m2);
                        const float a1 = fast_exp2(m_run - m_new), a2 = fast_exp2(m2 - m_new);
#pragma unroll
                        for (int db = 0; db < 2; ++db) {
                            const f32x4 o2 = *reinterpret_cast<const f32x4 *>(part_o + (w * kTrajRows + tok) * DH + 16 * db + 4 * s4);
#pragma unroll
                            for (int e = 0; e < 4; ++e) o_acc[db][e] = o_acc[db][e] * a1 + o2[e] * a2;
                        }
                        l_tot = l_tot * a1 + l2 * a2;
                        m_run = m_new;
                    }
                }
            }
            if (NP == 1 || part == 0) {
                const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
#pragma unroll
                for (int db = 0; db < 2; ++db) {
                    const float o[4] = {o_acc[db][0] * inv, o_acc[db][1] * inv, o_acc[db][2] * inv, o_acc[db][3] * inv};
                    traj_store4<T>(xs + tok * LD + DH * h + 16 * db + 4 * s4, o);
                }
            }
        }
    };

    // ---- embedding of step 0: target rows; every other row is zero
    const T *const xm = static_cast<const T *>(P.x_mean);
    for (int d = tid; d < D; d += NT) {
        c_ng[d] = static_cast<const T *>(P.norm_g)[d];
        c_nb[d] = static_cast<const T *>(P.norm_b)[d];
        c_wx[d] = static_cast<const T *>(P.w_x)[d];
        c_bx[d] = static_cast<const T *>(P.b_x)[d];
        c_wy[d] = static_cast<const T *>(P.w_y)[d];
        c_by[d] = static_cast<const T *>(P.b_y)[d];
        c_mt[d] = static_cast<const T *>(P.markers)[d];
        c_mb[d] = static_cast<const T *>(P.markers)[2 * D + d];
    }
    for (int d = tid; d < F; d += NT) c_b1[d] = static_cast<const T *>(P.b_h1)[d];
    if (tid < kTrajHeadOut) c_b2[tid] = static_cast<const T *>(P.b_h2)[tid];
    if (tid < 3 * P.K) c_mix[tid] = static_cast<const T *>(P.mix)[tid];
    __syncthreads();
    for (int i = tid; i < kTrajRows * D; i += NT) {
        const int r = i / D, d = i % D, g = r >> 1;
        float v = 0.f;
        if ((r & 1) && g < valid) v = to_f32(xm[(b0 + g) * P.Nt]) * to_f32(c_wx[d]) + to_f32(c_bx[d]) + to_f32(c_mt[d]);
        xs[r * LD + d] = from_f32<T>(v);
    }
    __syncthreads();

    using std::integral_constant;
    for (int t = 0; t < P.Nt; ++t) {
        const bool last_step = t + 1 == P.Nt;
        // the variates and feature means of the step's draw, long before they are needed
        float my_u = 0.f, my_n = 0.f;
        T my_x = from_f32<T>(0.f), my_tok = my_x;
        if (tid < valid) {
            const long at = static_cast<long>(t) * P.B + b0 + tid;
            my_u = P.rand_u[at];
            my_n = P.rand_n_f32 ? static_cast<const float *>(P.rand_n)[at] : to_f32(static_cast<const T *>(P.rand_n)[at]);
        }
        if (tid < 2 * valid && !last_step) my_x = xm[(b0 + (tid >> 1)) * P.Nt + t + (tid & 1)];
        if (tid < D) my_tok = static_cast<const T *>(P.ar_tokens)[static_cast<long>((t + 1) % P.bs) * D + tid];
        for (int l = 0; l < P.n_layers; ++l) {
            // the layer's parameter vectors and cache addresses are requested ahead of everything
            const T *vec = static_cast<const T *>(P.vecs) + static_cast<long>(l) * 8 * VW;
            TrajCols<T, S::ND> g1, be1, g2, be2, g3, be3, bias2;
            TrajCols<T, S::NF> bias1;
            g1.load(vec, wave, s4);
            be1.load(vec + VW, wave, s4);
            g2.load(vec + 2 * VW, wave, s4);
            be2.load(vec + 3 * VW, wave, s4);
            bias1.load(vec + 4 * VW, wave, s4);
            g3.load(vec + 5 * VW, wave, s4);
            be3.load(vec + 6 * VW, wave, s4);
            bias2.load(vec + 7 * VW, wave, s4);
            unsigned long long kv_raw[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) kv_raw[i] = P.kv[4 * l + i];
            {   // y = LN1(x + x W_fo^T)
                f32x4 acc[S::ND];
                product(integral_constant<int, 0>{}, integral_constant<int, S::KD>{}, acc, xs, LD);
                float v[S::ND][4];
#pragma unroll
                for (int b = 0; b < S::ND; ++b) {
                    float r[4];
                    traj_load4<T>(xs + tok * LD + 16 * (wave + NW * b) + 4 * s4, r);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[b][e] = acc[b][e] + r[e];
                }
                norm_store(v, g1, be1, P.eps1, ys);
            }
            {   // q, k, v
                f32x4 acc[3 * S::ND];
                product(integral_constant<int, S::kFo>{}, integral_constant<int, S::KD>{}, acc, ys, LD);
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int b = 0; b < S::ND; ++b) {
                        float o[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            o[e] = acc[p * S::ND + b][e];
                            if (p == 0) o[e] = to_f32(from_f32<T>(o[e])) * P.qscale;
                        }
                        traj_store4<T>(qkv + p * kTrajRows * LD + tok * LD + 16 * (wave + NW * b) + 4 * s4, o);
                    }
                __syncthreads();
            }
            T *kv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(kv_raw[i])),
                               hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(kv_raw[i] >> 32));
                kv[i] = reinterpret_cast<T *>(static_cast<unsigned long long>(hi) << 32 | lo);
            }
            // the caches: row 2 g is committed at slot t - 1 of trajectory g (its first read is a step away)
            {
                constexpr int CPR = DH * sizeof(T) / 16, PER = H * CPR;  // 16-byte pieces of a head's row, of a row
                const int rows = P.park_target && last_step ? 2 : 1;
                for (int i = tid; i < valid * rows * 2 * PER; i += NT) {
                    const int c = i % PER, which = i / PER & 1, rr = i / (2 * PER), g = rr / rows, target = rr % rows;
                    const int slot = P.own_base + t - 1 + target;
                    if (!target && t == 0) continue;
                    T *dst = (which ? kv[3] : kv[2]) + (((b0 + g) * H + c / CPR) * P.own_rows + slot) * DH + (c % CPR) * (16 / sizeof(T));
                    const T *src = (which ? vn : kn) + (2 * g + target) * LD + c * (16 / sizeof(T));
                    *reinterpret_cast<u32x4 *>(dst) = *reinterpret_cast<const u32x4 *>(src);
                }
            }
            attention(kv[0], kv[1], kv[2], kv[3], t);
            __syncthreads();
            {   // x1 = LN2(y + attn W_o^T)
                f32x4 acc[S::ND];
                product(integral_constant<int, S::kFo + S::kQkv>{}, integral_constant<int, S::KD>{}, acc, xs, LD);
                float v[S::ND][4];
#pragma unroll
                for (int b = 0; b < S::ND; ++b) {
                    float r[4];
                    traj_load4<T>(ys + tok * LD + 16 * (wave + NW * b) + 4 * s4, r);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[b][e] = acc[b][e] + r[e];
                }
                norm_store(v, g2, be2, P.eps2, ys);
            }
            {   // h = gelu(x1 W_1^T + b_1)
                f32x4 acc[S::NF];
                product(integral_constant<int, S::kFo + S::kQkv + S::kO>{}, integral_constant<int, S::KD>{}, acc, ys, LD);
#pragma unroll
                for (int b = 0; b < S::NF; ++b) {
                    float o[4], bias[4];
                    bias1.get(b, bias);
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = gelu(acc[b][e] + bias[e]);
                    traj_store4<T>(hs + tok * LF + 16 * (wave + NW * b) + 4 * s4, o);
                }
                __syncthreads();
            }
            {   // x = LN3(x1 + h W_2^T + b_2)
                f32x4 acc[S::ND];
                product(integral_constant<int, S::kFo + S::kQkv + S::kO + S::k1>{}, integral_constant<int, S::KF>{}, acc, hs, LF);
                float v[S::ND][4];
#pragma unroll
                for (int b = 0; b < S::ND; ++b) {
                    float r[4], bias[4];
                    bias2.get(b, bias);
                    traj_load4<T>(ys + tok * LD + 16 * (wave + NW * b) + 4 * s4, r);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[b][e] = acc[b][e] + r[e] + bias[e];
                }
                norm_store(v, g3, be3, P.eps3, xs);
            }
        }

        // ---- the head on the target rows, one draw per trajectory, the rows of the next step
        {
            constexpr int EPL = D / 64;
            float gam[EPL], bet[EPL];
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                gam[e] = to_f32(c_ng[lane * EPL + e]);
                bet[e] = to_f32(c_nb[lane * EPL + e]);
            }
            for (int r = wave; r < kTrajRows; r += NW) {
                const T *row = xs + r * LD + lane * EPL;
                float x[EPL], sum = 0.f;
#pragma unroll
                for (int e = 0; e < EPL; ++e) {
                    x[e] = to_f32(row[e]);
                    sum += x[e];
                }
                const float mean = wave_sum(sum) / D;
                float q = 0.f;
#pragma unroll
                for (int e = 0; e < EPL; ++e) q += (x[e] - mean) * (x[e] - mean);
                const float rstd = rsqrtf(wave_sum(q) / D + P.eps_out);
#pragma unroll
                for (int e = 0; e < EPL; ++e) ys[r * LD + lane * EPL + e] = from_f32<T>((x[e] - mean) * rstd * gam[e] + bet[e]);
            }
            __syncthreads();
        }
        {
            f32x4 acc[S::NF];
            product(integral_constant<int, 0>{}, integral_constant<int, S::KD>{}, acc, ys, LD);
#pragma unroll
            for (int b = 0; b < S::NF; ++b) {
                float o[4], bias[4];
                traj_load4<T>(c_b1 + 16 * (wave + NW * b) + 4 * s4, bias);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = gelu(acc[b][e] + bias[e]);
                traj_store4<T>(hs + tok * LF + 16 * (wave + NW * b) + 4 * s4, o);
            }
            __syncthreads();
        }
        {
            f32x4 acc[1];
            product(integral_constant<int, S::kH1>{}, integral_constant<int, S::KF>{}, acc, hs, LF);
            if (16 * wave < kTrajHeadOut) {
                float bias[4];
                traj_load4<T>(c_b2 + 16 * wave + 4 * s4, bias);
#pragma unroll
                for (int e = 0; e < 4; ++e) raw_s[tok][16 * wave + 4 * s4 + e] = acc[0][e] + bias[e];
            }
            // fragments that only fill the head's part of the tape up to a whole number of rings
#pragma unroll
            for (int i = S::kH1 + S::kH2; i < S::kHead; ++i) {
                ring[i % S::kRing] = *reinterpret_cast<const u32x4 *>(next);
                next += 1024;
            }
            if (tid < 2 * valid) x_s[tid] = to_f32(my_x);
            if (tid < D) tok_s[tid] = my_tok;
            next -= (static_cast<long>(P.n_layers) * S::kLayer + S::kHead) * 1024;
            __syncthreads();
        }
        if (tid < valid) {
            const float *raw = raw_s[2 * tid + 1];
            const T *const mix = c_mix;
            float mx = -INFINITY;
            for (int k = 0; k < P.K; ++k) mx = fmaxf(mx, raw[3 * k + 2] + to_f32(mix[2 * P.K + k]));
            float z = 0.f;
            for (int k = 0; k < P.K; ++k) z += expf(raw[3 * k + 2] + to_f32(mix[2 * P.K + k]) - mx);
            const float target = my_u * z;
            int comp = P.K - 1;
            float cum = 0.f;
            for (int k = 0; k < P.K; ++k) {
                cum += expf(raw[3 * k + 2] + to_f32(mix[2 * P.K + k]) - mx);
                if (cum > target) {
                    comp = k;
                    break;
                }
            }
            const float mean = raw[3 * comp] + to_f32(mix[comp]);
            const float sraw = raw[3 * comp + 1] + to_f32(mix[P.K + comp]);
            const float sp = sraw > 20.f ? sraw : log1pf(expf(sraw));
            const T y = from_f32<T>(mean + (fminf(sp, P.std_max) + P.std_min) * my_n);
            static_cast<T *>(P.preds)[(b0 + tid) * P.Nt + t] = y;
            y_s[tid] = to_f32(y);
        }
        __syncthreads();
        if (last_step) break;
        {
            for (int i = tid; i < 2 * valid * (D / 4); i += NT) {
                const int d = 4 * (i % (D / 4)), r = i / (D / 4);
                float wx[4], bx[4], m[4], o[4];
                traj_load4<T>(c_wx + d, wx);
                traj_load4<T>(c_bx + d, bx);
                traj_load4<T>((r & 1 ? c_mt : c_mb) + d, m);
                const float xv = x_s[r];
                if (r & 1) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = xv * wx[e] + bx[e] + m[e];
                } else {
                    float wy[4], by[4], tk[4];
                    traj_load4<T>(c_wy + d, wy);
                    traj_load4<T>(c_by + d, by);
                    traj_load4<T>(tok_s + d, tk);
                    const float yv = y_s[r >> 1];
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = xv * wx[e] + bx[e] + yv * wy[e] + by[e] + m[e] + tk[e];
                }
                traj_store4<T>(xs + r * LD + d, o);
            }
            __syncthreads();
        }
    }
}

}  // namespace artab
