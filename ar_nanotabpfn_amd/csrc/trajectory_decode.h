// A whole autoregressive sampling run in one launch: every workgroup takes a few trajectories through
// all steps and all layers (gfx950; bf16 / f16 / float32; head_dim 32).
//
// Given the cached context, trajectories do not depend on each other: the only thing a decode step
// of one trajectory needs from the rest of the chip is the weights and the context's keys and values,
// both constant.  A step that is cut into launches (context pass, buffer pass, layer boundary, tail)
// pays 30-40 us per layer for them whatever the size of the problem; here a layer costs what one
// compute unit needs to stream its weights and keys through (64 B per clock from the L2) plus ten
// workgroup barriers and the latency chains between them.  The rule for when the launches of the
// other route, which spread one layer over the whole chip, are faster is artab_trajectory_group_layers().  One
// trajectory per workgroup on a context that is not long: trajectory_crews.h.
//
// Rows.  A workgroup owns G trajectories; token row 2 g is trajectory g's buffer row of the step (the
// value drawn last), row 2 g + 1 its target row: at most 16 rows (16-bit types) or 4 (float32, whose
// matrix rate is an eighth: a 16-row tile with two rows in use would be bound by it).  Products are
// transposed as in fused_layer.h (C^T[n, m] = sum_k W[n, k] A[m, k]): weights are the A operand, the
// activation rows in LDS the B operand; a lane holds, for its token row, four consecutive features
// 4 sub + r of every 16-feature block (TrajOps).
//
// Weights.  Each wavefront has a tape: the 1 KiB operand fragments it will consume, in the order it
// consumes them, layer after layer, then the head's; the first kRing of them are repeated behind the
// end.  A ring of kRing fragments in registers is always kRing ahead, across products, barriers,
// layers and steps: after a fragment has been multiplied its registers receive the one kRing further
// on.  All ring positions are compile-time constants (the fragments of a layer are a multiple of
// kRing).  A layer's small vectors travel one layer ahead into the other of two LDS buffers.
//
// Attention.  One wavefront owns a head (or half of a head's keys at 4 heads, two heads in turn at
// 16); the columns of S^T = K Q^T are the token rows.  Keys come in blocks: the shared context serves
// every column, a trajectory's own rows only its two columns (the others are masked, their state does
// not change), so no merge of partial results is needed.  The first blocks are requested ahead of the
// q/k/v product.  The rows of this step that have just been projected are keys too: one last block
// straight from LDS, masked to (row 2 g, columns 2 g and 2 g + 1).  A value that is not finite stays with
// the columns that see it: products of keys that only some columns see reach those columns only.  Softmax in float32 with scale *
// log2(e) folded into the queries and rounded to the model's type, probabilities rounded to the
// model's type and summed as rounded: the rounding model of the context pass (mfma_flash.h).  The reference a column's probabilities are
// taken against follows its maximum only when that has risen by more than kSlack (base 2): the common
// block has no exchange between lanes and no rescaling.
#pragma once

#include <type_traits>

#include "common.h"
#include "mfma_flash.h"

namespace artab {

constexpr int kTrajWaves = 8;
constexpr int kTrajMaxMix = 21; // 3 K outputs of the head fit 64 columns
constexpr int kTrajHeadOut = 64;
constexpr int kTrajMaxLayers = 64;

struct TrajectoryParams {
    const char *tape;        // kTrajWaves tapes of `tape_stride` bytes
    long tape_stride;
    const void *vecs;        // [n_layers][8][max(D, F)]: g1, b1, g2, b2, bias_1, g3, b3, bias_2
    const unsigned long long *kv;  // [n_layers][4] addresses: context K, V; trajectory K, V
    int n_layers;            // <= kTrajMaxLayers
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
    // several workgroups to a trajectory (trajectory_crews.h): how often one of them looks for another's word, and what they
    // give each other, zero in front of the launch.  One workgroup to a trajectory: null, or the words of such a launch in
    // front of this one, which is then for the trajectories that it has given up.
    int most_polls;
    unsigned long long *exchange;
};
// A look for another workgroup's word takes about a microsecond: some 60 ms in all.  The others are on the chip, or will be
// when kernels of other streams make room; longer than that costs more than the run with one workgroup.
constexpr int kTrajMostPolls = 1 << 16;
constexpr unsigned kTrajGone = ~0u;  // in the place of an exchange's number: the workgroup has given its trajectory up
// Whether the two-crew kernel is built for `parts` workgroups to a trajectory: each has one head or more, a wavefront of one
// crew or more for each of them.
constexpr bool traj_parts_built(int D, int parts) {
    return (parts == 2 || parts == 4 || parts == 8) && D / 32 >= parts && D / 32 / parts <= kTrajWaves;
}
// Words of 8 bytes in one exchange between a trajectory's workgroups: two rows of D values, four bytes of them per word.
template <typename T>
constexpr int traj_exchange_words(int D) { return 2 * D * static_cast<int>(sizeof(T)) / 4; }
static __global__ __launch_bounds__(256) void trajectory_exchange_kernel(unsigned long long *words, long n) {
    const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) words[i] = 0;  // (the number of no exchange)
}
// Whether trajectory b has been given up by a launch of several workgroups to a trajectory.  For all NT threads of a workgroup.
template <typename T, int D, int NT>
__device__ __forceinline__ bool traj_given_up(const unsigned long long *exchange, long b, int tid) {
    __shared__ int found;
    if (tid == 0) found = 0;
    __syncthreads();
    for (int i = tid; i < 2 * traj_exchange_words<T>(D); i += NT)
        if (static_cast<unsigned>(exchange[b * 2 * traj_exchange_words<T>(D) + i] >> 32) == kTrajGone) found = 1;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(found) != 0;
}

// One 1 KiB fragment per operand and product.  Both types read the A operand as row lane % 16 of a
// 16-row block, kPer consecutive contraction elements at kPer (lane / 16).
//   16-bit: one 16x16x32 product; token lane % 16, features 4 sub + r with sub = lane / 16.
//   float32: four 4x4x1 products of 16 independent 4x4 blocks: block (lane / 16, lane / 4 % 4) holds
//   the partial sums of features 4 (lane / 4 % 4) + r over the contraction elements of lane / 16;
//   finish() adds the four of them, every row of 16 lanes then holds the same values.
template <typename T>
struct TrajOps {
    static constexpr int kRows = 16, kMax = 8, kStep = 32, kPer = 8;
    static constexpr float kSlack = std::is_same<T, f16_t>::value ? 8.f : 16.f;
    static __device__ __forceinline__ int tok(int lane) { return lane & 15; }
    static __device__ __forceinline__ int sub(int lane) { return lane >> 4; }
    static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
        typedef typename MfmaOps<T>::vec vec;
        return MfmaOps<T>::mma16(__builtin_bit_cast(vec, a), __builtin_bit_cast(vec, b), c);
    }
    static __device__ __forceinline__ void finish(f32x4 &) {}
    static __device__ __forceinline__ float sum(float x) { return row_sum(x); }  // over a token's four subs
    static __device__ __forceinline__ float max(float x) { return row_max(x); }
};
template <>
struct TrajOps<float> {
    static constexpr int kRows = 4, kMax = 2, kStep = 16, kPer = 4;
    static constexpr float kSlack = 16.f;
    static __device__ __forceinline__ int tok(int lane) { return lane & 3; }
    static __device__ __forceinline__ int sub(int lane) { return (lane >> 2) & 3; }
    static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
        const f32x4 fa = __builtin_bit_cast(f32x4, a), fb = __builtin_bit_cast(f32x4, b);
#pragma unroll
        for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_4x4x1f32(fa[j], fb[j], c, 0, 0, 0);
        return c;
    }
    static __device__ __forceinline__ void finish(f32x4 &c) {
#pragma unroll
        for (int r = 0; r < 4; ++r) c[r] = row_sum(c[r]);
    }
    static __device__ __forceinline__ float sum(float x) {
        x += row_rotate<8>(x);
        return x + row_rotate<4>(x);
    }
    static __device__ __forceinline__ float max(float x) {
        x = fmaxf(x, row_rotate<8>(x));
        return fmaxf(x, row_rotate<4>(x));
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

// gelu for results that are rounded to 16 bits (with erff, at two token rows in use, the activation of all 16 was a
// quarter of its product)
__device__ __forceinline__ float traj_gelu16(float x) {
    const float tail = normal_tail(x);
    return x * (x > 0.f ? 1.f - tail : tail);
}

// Sizes shared by the kernel and the host code that writes the tapes.
template <typename T, int D, int F>
struct TrajShape {
    static constexpr int NW = kTrajWaves;
    static constexpr int KD = D / TrajOps<T>::kStep, KF = F / TrajOps<T>::kStep;  // contraction steps
    static constexpr int ND = D / 16 / NW, NF = F / 16 / NW;                      // 16-feature blocks per wavefront
    static constexpr int kFo = ND * KD, kQkv = 3 * ND * KD, kO = ND * KD, k1 = NF * KD, k2 = ND * KF;
    static constexpr int pFo = 0, pQkv = kFo, pO = pQkv + kQkv, p1 = pO + kO, p2 = p1 + k1;  // in a layer's part of the tape
    static constexpr int kLayer = p2 + k2;
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
// ---- what the one-crew and the two-crew kernel (trajectory_crews.h) have in common at both ends of a step

// What the end of every step needs, in LDS: norm g and b, x and y embedding w and b, markers target and buffer; the
// head's biases.
template <typename T, int D, int F>
struct TrajConstants {
    static constexpr int kElems = 8 * D + F + kTrajHeadOut + 3 * kTrajMaxMix + 1;
    T *ng, *nb, *wx, *bx, *wy, *by, *mt, *mb, *b1, *b2, *mix;
    __device__ __forceinline__ explicit TrajConstants(T *at)
        : ng(at), nb(at + D), wx(at + 2 * D), bx(at + 3 * D), wy(at + 4 * D), by(at + 5 * D), mt(at + 6 * D), mb(at + 7 * D),
          b1(at + 8 * D), b2(b1 + F), mix(b2 + kTrajHeadOut) {}
    template <int NT>
    __device__ __forceinline__ void load(const TrajectoryParams &P, int tid) const {
        for (int d = tid; d < D; d += NT) {
            ng[d] = static_cast<const T *>(P.norm_g)[d];
            nb[d] = static_cast<const T *>(P.norm_b)[d];
            wx[d] = static_cast<const T *>(P.w_x)[d];
            bx[d] = static_cast<const T *>(P.b_x)[d];
            wy[d] = static_cast<const T *>(P.w_y)[d];
            by[d] = static_cast<const T *>(P.b_y)[d];
            mt[d] = static_cast<const T *>(P.markers)[d];
            mb[d] = static_cast<const T *>(P.markers)[2 * D + d];
        }
        for (int d = tid; d < F; d += NT) b1[d] = static_cast<const T *>(P.b_h1)[d];
        if (tid < kTrajHeadOut) b2[tid] = static_cast<const T *>(P.b_h2)[tid];
        if (tid < 3 * P.K) mix[tid] = static_cast<const T *>(P.mix)[tid];
    }
    // The rows of step 0, `rows` of them from trajectory b0 on: the target rows of `valid` trajectories, zero elsewhere.
    template <int NT>
    __device__ __forceinline__ void first_rows(const TrajectoryParams &P, long b0, int valid, int rows, T *xs, int ld, int tid) const {
        const T *const xm = static_cast<const T *>(P.x_mean);
        for (int i = tid; i < rows * D; i += NT) {
            const int r = i / D, d = i % D, g = r >> 1;
            float v = 0.f;
            if ((r & 1) && g < valid) v = to_f32(xm[(b0 + g) * P.Nt]) * to_f32(wx[d]) + to_f32(bx[d]) + to_f32(mt[d]);
            xs[r * ld + d] = from_f32<T>(v);
        }
    }
    // The rows of the next step: buffer row 2 g with the value just drawn and the position's token, target row 2 g + 1.
    template <int NT>
    __device__ __forceinline__ void next_rows(const float *x_s, const float *y_s, const T *tok_s, int valid, T *xs, int ld, int tid) const {
        for (int i = tid; i < 2 * valid * (D / 4); i += NT) {
            const int d = 4 * (i % (D / 4)), r = i / (D / 4);
            float w[4], b[4], m[4], o[4];
            traj_load4<T>(wx + d, w);
            traj_load4<T>(bx + d, b);
            traj_load4<T>((r & 1 ? mt : mb) + d, m);
            const float xv = x_s[r];
            if (r & 1) {
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = xv * w[e] + b[e] + m[e];
            } else {
                float w2[4], b2[4], tk[4];
                traj_load4<T>(wy + d, w2);
                traj_load4<T>(by + d, b2);
                traj_load4<T>(tok_s + d, tk);
                const float yv = y_s[r >> 1];
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = xv * w[e] + b[e] + yv * w2[e] + b2[e] + m[e] + tk[e];
            }
            traj_store4<T>(xs + r * ld + d, o);
        }
    }
    // The final norm of a row, its element from mean and 1 / std.
    __device__ __forceinline__ T normed(float x, float mean, float rstd, int d) const {
        return from_f32<T>((x - mean) * rstd * to_f32(ng[d]) + to_f32(nb[d]));
    }
    // The value of component `comp` of a row's raw outputs, from a standard normal variate.
    __device__ __forceinline__ T value(const TrajectoryParams &P, const float *raw, int comp, float normal) const {
        const float mean = raw[3 * comp] + to_f32(mix[comp]);
        const float sraw = raw[3 * comp + 1] + to_f32(mix[P.K + comp]);
        const float sp = sraw > 20.f ? sraw : log1pf(expf(sraw));
        return from_f32<T>(mean + (fminf(sp, P.std_max) + P.std_min) * normal);
    }
};

// Keys and values of token row 2 g + `from`, HL heads of them from `head` on, to row `slot` of the cache of trajectory b0 + g.
template <typename T, int D, int NT, int HL = D / 32>
__device__ __forceinline__ void traj_commit(__attribute__((address_space(1))) char *ck, __attribute__((address_space(1))) char *cv,
                                            const T *kn, const T *vn, int ld, long b0, int valid, int own_rows, int from, int slot, int tid,
                                            int head = 0) {
    constexpr int DH = 32, H = D / DH, CPR = DH * sizeof(T) / 16, PER = HL * CPR;  // 16-byte pieces of a head's row, of HL of them
    for (int i = tid; i < valid * 2 * PER; i += NT) {
        const int c = head * CPR + i % PER, which = i / PER & 1, g = i / (2 * PER);
        __attribute__((address_space(1))) char *const dst =
            (which ? cv : ck) + (((b0 + g) * H + c / CPR) * own_rows + slot) * static_cast<long>(DH * sizeof(T)) + 16 * (c % CPR);
        *(__attribute__((address_space(1))) u32x4 *)dst =
            *reinterpret_cast<const u32x4 *>((which ? vn : kn) + (2 * g + from) * ld + c * (16 / sizeof(T)));
    }
}

// SEVERAL: G > 1.  (One trajectory has no columns to keep apart: doing it all the same costs 3 % of a run.)
template <typename T, int D, int F, bool SEVERAL>
__global__ __launch_bounds__(kTrajWaves * 64) void trajectory_decode_kernel(TrajectoryParams P) {
    typedef TrajOps<T> Ops;
    typedef TrajShape<T, D, F> S;
    constexpr int NW = kTrajWaves, NT = NW * 64, DH = 32, H = D / DH, ROWS = Ops::kRows;
    constexpr bool k16 = sizeof(T) == 2;
    constexpr int LD = D + (k16 ? 8 : 4), LF = F + (k16 ? 8 : 4);  // row strides: 16 bytes off a multiple of 128
    constexpr int VW = D > F ? D : F;
    // keys per block: one step of the second product's contraction.  (Two steps per block, which give the
    // chains between the two products company, lose 12 % at 200 context rows: they round the
    // requests up further, and a request costs the compute unit's address unit 16 clocks whatever it
    // brings.)
    constexpr int BK = k16 ? 32 : 16;
    constexpr int NP = NW > H ? NW / H : 1;         // wavefronts per head
    constexpr int HPW = H > NW ? H / NW : 1;        // heads per wavefront, in turn
    constexpr int VPAD = DH + 16;

    __shared__ __attribute__((aligned(16))) T xs[ROWS * LD];   // layer input; attention output
    __shared__ __attribute__((aligned(16))) T ys[ROWS * LD];   // normed feature stage, then x1; z of the head
    constexpr int QKV = 3 * ROWS * LD, HID = ROWS * LF;
    __shared__ __attribute__((aligned(16))) T qkv[QKV > HID ? QKV : HID];  // q, k, v of the step; hidden layer
    T *const qs = qkv, *const kn = qkv + ROWS * LD, *const vn = qkv + 2 * ROWS * LD, *const hs = qkv;
    __shared__ __attribute__((aligned(16))) T v_lds[k16 ? NW * BK * VPAD : 8];
    __shared__ float red_a[NW * ROWS], red_b[NW * ROWS];
    __shared__ __attribute__((aligned(16))) float part_o[NP > 1 ? NW * ROWS * DH : 4];
    __shared__ float part_m[NP > 1 ? NW * ROWS : 1], part_l[NP > 1 ? NW * ROWS : 1];
    __shared__ float raw_s[ROWS][kTrajHeadOut + 1];
    __shared__ float y_s[Ops::kMax], x_s[2 * Ops::kMax];
    // the parameter vectors of this layer and of the next; cache addresses of every layer
    __shared__ __attribute__((aligned(16))) T pbuf[2][8 * VW];
    __shared__ unsigned long long kv_s[4 * kTrajMaxLayers];
    __shared__ __attribute__((aligned(16))) T cst[TrajConstants<T, D, F>::kElems], tok_s[D];  // and the position token of the coming step
    const TrajConstants<T, D, F> C(cst);

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int tok = Ops::tok(lane), sub = Ops::sub(lane);  // output layout of the products
    const int row16 = lane & 15, quad = lane >> 4;         // operand layout
    const long b0 = static_cast<long>(blockIdx.x) * P.G;
    const int valid = static_cast<int>(min(static_cast<long>(P.G), P.B - b0));
    if constexpr (!SEVERAL)
        if (P.exchange && !traj_given_up<T, D, NT>(P.exchange, b0, tid)) return;

    // ---- the weight tape
    u32x4 ring[S::kRing];
    const char *next = P.tape + wave * P.tape_stride + 16 * lane;
#pragma unroll
    for (int i = 0; i < S::kRing; ++i) {
        ring[i] = *reinterpret_cast<const u32x4 *>(next);
        next += 1024;
    }
    // acc[b] += W_b A^T over KS steps of NB blocks; fragments POS .. POS + KS * NB - 1 of the tape section
    auto product = [&](auto pos_, auto ks_, auto &acc, const T *act, int ld) {
        constexpr int POS = decltype(pos_)::value, KS = decltype(ks_)::value;
        constexpr int NB = sizeof(acc) / sizeof(acc[0]);
        constexpr int KC = KS < 8 ? KS : 8;  // activation operands are read KC steps at a time
        const T *const a = act + (k16 ? row16 : tok) * ld + Ops::kPer * quad;
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k0 = 0; k0 < KS; k0 += KC) {
            u32x4 bf[KC];
#pragma unroll
            for (int k = 0; k < KC; ++k) bf[k] = *reinterpret_cast<const u32x4 *>(a + Ops::kStep * (k0 + k));
#pragma unroll
            for (int k = 0; k < KC; ++k)
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    constexpr int R = S::kRing;
                    const int slot = (POS + (k0 + k) * NB + b) % R;
                    acc[b] = Ops::mma(ring[slot], bf[k], acc[b]);
                    ring[slot] = *reinterpret_cast<const u32x4 *>(next);
                    next += 1024;
                }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) Ops::finish(acc[b]);
    };
    // LayerNorm of v (this lane's features of its token row) into dst
    auto norm_store = [&](auto &v, const T *gam, const T *bet, float eps, T *dst) {
        constexpr int NB = sizeof(v) / sizeof(v[0]);
        constexpr float kLocal = NB * 16;
        float s = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b) s += (v[b][0] + v[b][1]) + (v[b][2] + v[b][3]);
        s = Ops::sum(s);
        const float lmean = s * (1.f / kLocal);
        float q = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float d = v[b][e] - lmean;
                q += d * d;
            }
        q = Ops::sum(q);
        if (lane < ROWS * (k16 ? 1 : 4) && sub == 0) {
            red_a[wave * ROWS + tok] = lmean;
            red_b[wave * ROWS + tok] = q;
        }
        float g[NB][4], be[NB][4];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            traj_load4<T>(gam + 16 * (wave + NW * b) + 4 * sub, g[b]);
            traj_load4<T>(bet + 16 * (wave + NW * b) + 4 * sub, be[b]);
        }
        __syncthreads();
        float lm[NW], lq[NW], sum8[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            lm[w] = red_a[w * ROWS + tok];
            lq[w] = red_b[w * ROWS + tok];
        }
        auto tree = [&](const float (&x)[NW]) { return ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7])); };
        const float mean = tree(lm) * (1.f / NW);
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float d = lm[w] - mean;
            sum8[w] = fmaf(kLocal * d, d, lq[w]);
        }
        const float rstd = __builtin_amdgcn_rsqf(fmaf(tree(sum8), 1.f / D, eps));
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (v[b][e] - mean) * rstd * g[b][e] + be[b][e];
            traj_store4<T>(dst + tok * LD + 16 * (wave + NW * b) + 4 * sub, o);
        }
        __syncthreads();
    };
    // gelu of this lane's 4 values of every block, stored to the hidden tile
    auto gelu_store = [&](auto &acc, const T *bias) {
        constexpr int NB = sizeof(acc) / sizeof(acc[0]);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int col = 16 * (wave + NW * b) + 4 * sub;
            float bi[4];
            traj_load4<T>(bias + col, bi);
            if constexpr (k16) {
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = traj_gelu16(acc[b][e] + bi[e]);
                traj_store4<T>(hs + tok * LF + col, o);
            } else {  // the four rows of lanes hold the same values: each does one of them
                const float a = acc[b][0] + bi[0], c = acc[b][1] + bi[1], d = acc[b][2] + bi[2], f = acc[b][3] + bi[3];
                const float x = quad == 0 ? a : quad == 1 ? c : quad == 2 ? d : f;
                hs[tok * LF + col + quad] = 0.5f * x * (1.f + erff(x * 0.70710678118654752f));
            }
        }
    };

    // ---- attention of this wavefront's head(s): committed rows, then the rows of this step
    const int part = wave / H;  // (only with NP > 1)
    const int head0 = NP > 1 ? wave % H : wave;
    T *const vt = v_lds + (k16 ? wave * BK * VPAD : 0);
    // One block of keys as it comes from memory: K in operand order; V as 16-byte pieces of the
    // row-major tile (16-bit) or as the operand of the second product (float32); which rows they are.
    struct Block {
        u32x4 k[2], v[2];
        int row0, n, g;
    };
    // The layer's caches, as addresses in global memory: made from integers, plain pointers would be
    // generic ones, whose loads count as LDS accesses too — every wait for LDS would wait for the keys.
    typedef __attribute__((address_space(1))) char *Global;
    Global kv[4];
    // Blocks by number: the context's, then trajectory 0's, 1's, ... (the division of the number by
    // the blocks of a trajectory as a multiplication: a loop here costs more than the block's loads)
    int n_own = 0, nb_ctx = (P.n_ctx + BK - 1) / BK, nb_own = 0, n_blocks = 0;
    unsigned own_inv = 0;
    auto set_step = [&](int t) {
        n_own = P.own_base + (t > 0 ? t - 1 : 0);
        nb_own = (n_own + BK - 1) / BK;
        own_inv = nb_own > 1 ? 0xffffffffu / static_cast<unsigned>(nb_own) + 1 : 0;
        n_blocks = nb_ctx + valid * nb_own;
    };
    // (rows past a segment's end re-read its last one)
    auto fetch = [&](int h, int i, Block &r) {
        if (i >= n_blocks) return;
        const int j = i - nb_ctx;
        const int of = nb_own > 1 ? static_cast<int>(__umulhi(static_cast<unsigned>(j), own_inv)) : j;
        const int g = j < 0 ? -1 : of, row0 = BK * (j < 0 ? i : j - of * nb_own);
        r.row0 = row0;
        r.n = g < 0 ? P.n_ctx : n_own;
        r.g = g;
        const int last = r.n - 1;
        const long at = (g < 0 ? static_cast<long>(h) * P.ctx_rows : ((b0 + g) * H + h) * P.own_rows) * DH;
        const Global kp = kv[g < 0 ? 0 : 2] + at * static_cast<long>(sizeof(T)), vp = kv[g < 0 ? 1 : 3] + at * static_cast<long>(sizeof(T));
        typedef const __attribute__((address_space(1))) u32x4 *Global16;
        constexpr unsigned RB = DH * sizeof(T);  // bytes of a row
        if constexpr (k16) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
                r.k[x] = *(Global16)(kp + (static_cast<unsigned>(min(row0 + 16 * x + row16, last)) * RB + 16 * quad));
#pragma unroll
            for (int x = 0; x < 2; ++x)
                r.v[x] = *(Global16)(vp + (static_cast<unsigned>(min(row0 + 16 * x + lane / 4, last)) * RB + 16 * (lane % 4)));
        } else {
            const Global kr = kp + (static_cast<unsigned>(min(row0 + row16, last)) * RB + 16 * quad);
            r.k[0] = *(Global16)kr;
            r.k[1] = *(Global16)(kr + 64);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const __attribute__((address_space(1))) unsigned *vr =
                    (const __attribute__((address_space(1))) unsigned *)(vp + (static_cast<unsigned>(min(row0 + 4 * quad + j, last)) * RB + 4 * row16));
                r.v[0][j] = vr[0];
                r.v[1][j] = vr[16];
            }
        }
    };
    Block r0, r1;
    const int first_block = NP > 1 ? part : 0;  // the wavefront's blocks: this one and every NP-th
    auto first_blocks = [&](int h) {
        fetch(h, first_block, r0);
        fetch(h, first_block + NP, r1);
    };
    auto attention = [&](int h, int t) {
        u32x4 qf[k16 ? 1 : 2];
#pragma unroll
        for (int x = 0; x < (k16 ? 1 : 2); ++x)
            qf[x] = *reinterpret_cast<const u32x4 *>(qs + (k16 ? row16 : tok) * LD + DH * h + Ops::kStep * x + Ops::kPer * quad);
        f32x4 o_acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
        float m_run = -1e30f, l_run = 0.f;
        // 16 bits: the sum of the probabilities as the second product takes them, rounded, from one more product
        // with a row of ones (of the unrounded ones, their rounding would not cancel in the division)
        f32x4 l_acc = {0.f, 0.f, 0.f, 0.f};
        unsigned one2 = 0u;
        if constexpr (k16) one2 = pack2<T>(1.f, 1.f);
        const u32x4 ones = {one2, one2, one2, one2};
        // Scores (lane: keys 4 sub + r of each 16-key part, its token) to probabilities.
        auto fold = [&](auto &sc) {
            constexpr int NX = sizeof(sc) / sizeof(sc[0]);
            float tmax = sc[0][0];
#pragma unroll
            for (int x = 0; x < NX; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, sc[x][r]);
            if (__any(tmax > m_run + Ops::kSlack)) {
                const float m_new = fmaxf(m_run, Ops::max(tmax));
                const float alpha = fast_exp2(m_run - m_new);
                if constexpr (k16) l_acc[0] *= alpha;
                else l_run *= alpha;
#pragma unroll
                for (int db = 0; db < 2; ++db)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o_acc[db][r] *= alpha;
                m_run = m_new;
            }
#pragma unroll
            for (int x = 0; x < NX; ++x) {
#pragma unroll
                for (int r = 0; r < 4; ++r) sc[x][r] = fast_exp2(sc[x][r] - m_run);
                if constexpr (!k16) l_run += (sc[x][0] + sc[x][1]) + (sc[x][2] + sc[x][3]);
            }
        };
        typedef short s16x8 __attribute__((ext_vector_type(8)));
        auto tr_read = [](const T *a) {
            return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(a));
        };
        // float32: the probabilities of keys 4 (lane / 16) + j for this lane's token
        const int p_from = ((lane & 48) | (quad << 2) | (lane & 3)) << 2;
        auto p_operand = [&](const f32x4 &p) {
            u32x4 r;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float pj = p[j];
                r[j] = __builtin_amdgcn_ds_bpermute(p_from, __builtin_bit_cast(int, pj));
            }
            return r;
        };
        // Block i; the wavefront's block after next goes where this one was.  With SEVERAL, a trajectory's block
        // is masked for the columns of the others, and they keep what they have: their probabilities are
        // zeros, but a zero times a value that is not finite is not zero.
        auto compute = [&](Block &r, int i) {
            constexpr int NX = BK / 16;
            const int row0 = r.row0, n = r.n, g = r.g;
            f32x4 sc[NX];
            if constexpr (k16) {
#pragma unroll
                for (int x = 0; x < 2; ++x)
                    *reinterpret_cast<u32x4 *>(vt + (16 * x + lane / 4) * VPAD + 8 * (lane % 4)) = r.v[x];
#pragma unroll
                for (int x = 0; x < NX; ++x) sc[x] = Ops::mma(r.k[x], qf[0], f32x4{0.f, 0.f, 0.f, 0.f});
                fetch(h, i + 2 * NP, r);
            } else {
                sc[0] = Ops::mma(r.k[0], qf[0], f32x4{0.f, 0.f, 0.f, 0.f});
                sc[0] = Ops::mma(r.k[1], qf[1], sc[0]);
                Ops::finish(sc[0]);
            }
            // (with one trajectory the other columns are nobody's)
            const bool mine = !SEVERAL || g < 0 || (tok >> 1) == g;
            auto add = [&](f32x4 &o, const u32x4 &v, const u32x4 &pv) {
                const f32x4 sum = Ops::mma(v, pv, o);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = mine ? sum[e] : o[e];
            };
            if (row0 + BK > n || (SEVERAL && g >= 0)) {
#pragma unroll
                for (int x = 0; x < NX; ++x)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (!mine || row0 + 16 * x + 4 * sub + e >= n) sc[x][e] = -INFINITY;
            }
            fold(sc);
            if constexpr (k16) {
                __builtin_amdgcn_wave_barrier();
                const u32x4 pv = {pack2<T>(sc[0][0], sc[0][1]), pack2<T>(sc[0][2], sc[0][3]),
                                  pack2<T>(sc[1][0], sc[1][1]), pack2<T>(sc[1][2], sc[1][3])};
                l_acc = Ops::mma(ones, pv, l_acc);
#pragma unroll
                for (int db = 0; db < 2; ++db) {
                    const T *a = vt + (4 * quad + (row16 >> 2)) * VPAD + 16 * db + 4 * (lane & 3);
                    const s16x4 lo = tr_read(a), hi = tr_read(a + 16 * VPAD);
                    const s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    add(o_acc[db], __builtin_bit_cast(u32x4, both), pv);
                }
                __builtin_amdgcn_wave_barrier();
            } else {
                const u32x4 pv = p_operand(sc[0]);
#pragma unroll
                for (int db = 0; db < 2; ++db) add(o_acc[db], r.v[db], pv);
                fetch(h, i + 2 * NP, r);
            }
        };
        for (int i = first_block; i < n_blocks; i += 2 * NP) {
            compute(r0, i);
            if (i + NP < n_blocks) compute(r1, i + NP);
        }
        if (t > 0 && (NP == 1 || part == 0)) {  // the buffer rows of this step
            f32x4 sc[1];
            const T *const kr = kn + (k16 ? row16 : lane & 3) * LD + DH * h + Ops::kPer * quad;
            sc[0] = Ops::mma(*reinterpret_cast<const u32x4 *>(kr), qf[0], f32x4{0.f, 0.f, 0.f, 0.f});
            if constexpr (!k16) {
                sc[0] = Ops::mma(*reinterpret_cast<const u32x4 *>(kr + 16), qf[1], sc[0]);
                Ops::finish(sc[0]);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * sub + e != (tok & ~1)) sc[0][e] = -INFINITY;
            // One key per column: its probability to every lane of the column, and the products of the column's
            // own row (a matrix product over the rows of all trajectories would multiply each by all of them).
            float vr[2][4];
#pragma unroll
            for (int db = 0; db < 2; ++db) traj_load4<T>(vn + (tok & ~1) * LD + DH * h + 16 * db + 4 * sub, vr[db]);
            fold(sc);
            float p = Ops::sum((sc[0][0] + sc[0][1]) + (sc[0][2] + sc[0][3]));
            if constexpr (k16) {
                p = to_f32(from_f32<T>(p));
                l_acc[0] += p;
            }
            if (k16 || quad == 0) {  // (float32: the four rows of lanes are partial sums)
#pragma unroll
                for (int db = 0; db < 2; ++db)
#pragma unroll
                    for (int e = 0; e < 4; ++e) o_acc[db][e] = fmaf(p, vr[db][e], o_acc[db][e]);
            }
        }
        float l_tot = k16 ? l_acc[0] : Ops::sum(l_run);
#pragma unroll
        for (int db = 0; db < 2; ++db) Ops::finish(o_acc[db]);
        if constexpr (NP > 1) {  // the other wavefronts' keys of this head
            if (part > 0) {
                if (sub == 0) {
                    part_m[wave * ROWS + tok] = m_run;
                    part_l[wave * ROWS + tok] = l_tot;
                }
#pragma unroll
                for (int db = 0; db < 2; ++db)
                    *reinterpret_cast<f32x4 *>(part_o + (wave * ROWS + tok) * DH + 16 * db + 4 * sub) = o_acc[db];
            }
            __syncthreads();
            if (part == 0) {
#pragma unroll
                for (int p = 1; p < NP; ++p) {
                    const int w = wave + p * H;
                    const float m2 = part_m[w * ROWS + tok], l2 = part_l[w * ROWS + tok];
                    const float m_new = fmaxf(m_run, m2);
                    const float a1 = fast_exp2(m_run - m_new), a2 = fast_exp2(m2 - m_new);
#pragma unroll
                    for (int db = 0; db < 2; ++db) {
                        const f32x4 o2 = *reinterpret_cast<const f32x4 *>(part_o + (w * ROWS + tok) * DH + 16 * db + 4 * sub);
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
                traj_store4<T>(xs + tok * LD + DH * h + 16 * db + 4 * sub, o);
            }
        }
    };

    // ---- constants, the first layer's vectors, the embedding of step 0: target rows; every other row is zero
    constexpr int kPieces = 8 * VW * static_cast<int>(sizeof(T)) / 16;  // of a layer's vectors
    static_assert(kPieces <= NT, "one piece per thread");
    const u32x4 *const vec_src = static_cast<const u32x4 *>(P.vecs);
    if (tid < kPieces) reinterpret_cast<u32x4 *>(pbuf[0])[tid] = vec_src[tid];
    for (int i = tid; i < 4 * P.n_layers; i += NT) kv_s[i] = P.kv[i];
    const T *const xm = static_cast<const T *>(P.x_mean);
    C.template load<NT>(P, tid);
    __syncthreads();
    C.template first_rows<NT>(P, b0, valid, ROWS, xs, LD, tid);
    __syncthreads();

    using std::integral_constant;
    int pp = 0;  // which of the two vector buffers holds this layer's
    for (int t = 0; t < P.Nt; ++t) {
        const bool last_step = t + 1 == P.Nt;
        set_step(t);
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
            const T *const vec = pbuf[pp];
            u32x4 next_vec = {0u, 0u, 0u, 0u};
            if (tid < kPieces) next_vec = vec_src[(l + 1 < P.n_layers ? l + 1 : 0) * kPieces + tid];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const unsigned long long raw = kv_s[4 * l + i];
                const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(raw)),
                               hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(raw >> 32));
                kv[i] = (Global)(static_cast<unsigned long long>(hi) << 32 | lo);
            }
            {   // y = LN1(x + x W_fo^T)
                f32x4 acc[S::ND];
                product(integral_constant<int, 0>{}, integral_constant<int, S::KD>{}, acc, xs, LD);
                float v[S::ND][4];
#pragma unroll
                for (int b = 0; b < S::ND; ++b) {
                    float r[4];
                    traj_load4<T>(xs + tok * LD + 16 * (wave + NW * b) + 4 * sub, r);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[b][e] = acc[b][e] + r[e];
                }
                norm_store(v, vec, vec + VW, P.eps1, ys);
            }
            first_blocks(head0);
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
                        traj_store4<T>(qkv + p * ROWS * LD + tok * LD + 16 * (wave + NW * b) + 4 * sub, o);
                    }
                __syncthreads();
            }
            // the caches: row 2 g is committed at slot t - 1 of trajectory g (its first read is a step
            // away); behind the last one the target row, where the caller keeps it
            if (t > 0) traj_commit<T, D, NT>(kv[2], kv[3], kn, vn, LD, b0, valid, P.own_rows, 0, P.own_base + t - 1, tid);
            if (P.park_target && last_step) traj_commit<T, D, NT>(kv[2], kv[3], kn, vn, LD, b0, valid, P.own_rows, 1, P.own_base + t, tid);
            attention(head0, t);
#pragma unroll
            for (int hh = 1; hh < HPW; ++hh) {
                first_blocks(head0 + NW * hh);
                attention(head0 + NW * hh, t);
            }
            __syncthreads();
            {   // x1 = LN2(y + attn W_o^T)
                f32x4 acc[S::ND];
                product(integral_constant<int, S::kFo + S::kQkv>{}, integral_constant<int, S::KD>{}, acc, xs, LD);
                float v[S::ND][4];
#pragma unroll
                for (int b = 0; b < S::ND; ++b) {
                    float r[4];
                    traj_load4<T>(ys + tok * LD + 16 * (wave + NW * b) + 4 * sub, r);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[b][e] = acc[b][e] + r[e];
                }
                norm_store(v, vec + 2 * VW, vec + 3 * VW, P.eps2, ys);
            }
            {   // h = gelu(x1 W_1^T + b_1)
                f32x4 acc[S::NF];
                product(integral_constant<int, S::kFo + S::kQkv + S::kO>{}, integral_constant<int, S::KD>{}, acc, ys, LD);
                gelu_store(acc, vec + 4 * VW);
                if (tid < kPieces) reinterpret_cast<u32x4 *>(pbuf[pp ^ 1])[tid] = next_vec;
                __syncthreads();
            }
            {   // x = LN3(x1 + h W_2^T + b_2)
                f32x4 acc[S::ND];
                product(integral_constant<int, S::kFo + S::kQkv + S::kO + S::k1>{}, integral_constant<int, S::KF>{}, acc, hs, LF);
                float v[S::ND][4];
#pragma unroll
                for (int b = 0; b < S::ND; ++b) {
                    float r[4], bias[4];
                    traj_load4<T>(vec + 7 * VW + 16 * (wave + NW * b) + 4 * sub, bias);
                    traj_load4<T>(ys + tok * LD + 16 * (wave + NW * b) + 4 * sub, r);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[b][e] = acc[b][e] + r[e] + bias[e];
                }
                norm_store(v, vec + 5 * VW, vec + 6 * VW, P.eps3, xs);
            }
            pp ^= 1;
        }

        // ---- the head on the target rows, one draw per trajectory, the rows of the next step
        {
            constexpr int EPL = D / 64;
            for (int r = wave; r < ROWS; r += NW) {
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
                for (int e = 0; e < EPL; ++e) ys[r * LD + lane * EPL + e] = C.normed(x[e], mean, rstd, lane * EPL + e);
            }
            __syncthreads();
        }
        {
            f32x4 acc[S::NF];
            product(integral_constant<int, 0>{}, integral_constant<int, S::KD>{}, acc, ys, LD);
            gelu_store(acc, C.b1);
            __syncthreads();
        }
        {
            f32x4 acc[1];
            product(integral_constant<int, S::kH1>{}, integral_constant<int, S::KF>{}, acc, hs, LF);
            if (16 * wave < kTrajHeadOut) {
                float bias[4];
                traj_load4<T>(C.b2 + 16 * wave + 4 * sub, bias);
#pragma unroll
                for (int e = 0; e < 4; ++e) raw_s[tok][16 * wave + 4 * sub + e] = acc[0][e] + bias[e];
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
            const T *const mix = C.mix;
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
            const T y = C.value(P, raw, comp, my_n);
            static_cast<T *>(P.preds)[(b0 + tid) * P.Nt + t] = y;
            y_s[tid] = to_f32(y);
        }
        __syncthreads();
        if (last_step) break;
        C.template next_rows<NT>(x_s, y_s, tok_s, valid, xs, LD, tid);
        __syncthreads();
    }
}

}  // namespace artab
