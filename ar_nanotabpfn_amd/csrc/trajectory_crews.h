// The whole-run decode of one trajectory per workgroup (trajectory_decode.h has the scheme, the weights' tapes and the
// rounding model) with two crews of eight wavefronts.  d_model 128 or 256; with several workgroups to a trajectory 512 too.
//
// What bounds a run is one compute unit: its address unit, which a wavefront's 1 KiB request occupies for 16 clocks,
// and the chain of a layer's products, norms and barriers.  A wavefront waits until its request is accepted, so whoever
// computes should not ask: with one crew the requests of a layer (54 per wavefront at d_model 128 and 200 context rows:
// 7000 clocks) and the chain (9000) came one after the other.  Here crew 0 does q/k/v, W_o with LN2 and W_2 with LN3,
// crew 1 W_fo with LN1, the attention and W_1 with the activation; whichever is not computing asks for what it will
// need next.  A wavefront has 128 registers then, about half of them for fragments on their way.
//
// One trajectory has two token rows (its buffer row and its target row).  They stand in all column pairs of a product's
// operand, so that every lane has results that count: the activation, the softmax of several blocks of keys and the
// norms' exchange between the wavefronts are spread over them.
//
// Measured, us per layer and step, one crew / two, 64 trajectories on a shared context: bf16, d_model 128, 8.6 / 6.9 at
// 64 rows, 9.6 / 7.4 at 200, 12.1 / 10.7 at 700, 17.5 / 16.6 at 1500, 26.3 / 26.8 at 3000; d_model 256, 15.4 / 13.1 at 64,
// 17.1 / 15.6 at 200, 21.1 / 20.2 at 600, 22.6 / 22.8 at 768, 32.5 / 32.9 at 1500; float32, d_model 128, 20.2 / 17.5 at 200,
// 54.2 / 48.9 at 2000; d_model 256, 42.6 / 35.0 and 110.5 / 98.3.  Contexts of their own, bf16, d_model 128: 64 trajectories 17.9 /
// 16.6 at 1200, 29.6 / 29.3 at 2000, 35.6 / 35.2 at 2600; 192 of them 26.6 / 25.7 at 1200; 256 13.4 / 11.5 at 300, 17.2 / 17.3 at 500,
// 21.4 / 21.7 at 700, 37.0 / 37.6 at 1500; d_model 256: 64 30.5 / 29.7 at 768, 38.6 / 38.0 at 1000, 44.4 / 44.9 at 1300; 192 45.1 / 44.4 at
// 850; 256 39.2 / 37.5 at 500, 45.8 / 45.6 at 700, 47.6 / 48.4 at 768 (f16 alike).  Long contexts in 16 bits are bound by the stream of keys from the L2,
// which eight wavefronts with twice the registers ask for a little better: crews_serve() draws the line.
// Not kept: crew 0 taking a share of a long context's keys (its registers do not hold them beside the weights: 9.2
// instead of 7.0 ms for 64 x 512 own rows); workgroups half a layer apart (no difference: it is not the memory they
// wait for together, a compute unit gets 55-85 GB/s of keys whatever the others do).
//
// Several workgroups to a trajectory (PARTS): each has its share of the heads, which is its share of the q/k/v weights and
// of the keys, what one compute unit needs longest for; everything behind the attention all of them compute, the same to the
// bit.  Per layer they give each other their heads' output, 1 KiB in 16 bits at d_model 256: dealing out the other products as well
// would take two more exchanges of about 0.9 us each and save 1.4.  64 trajectories of d_model 256 with 600 own rows, bf16, us per
// layer and step: 21.7 with one workgroup, 15.7 with two; 32 on a shared context of 4000 rows 60.9 / 36.1 / 22.9 / 17.4 with 1 / 2 /
// 4 / 8.  artab_trajectory_parts() says how many.
//
// Workgroups that wait for others want them on the chip.  An XCD starts those of a launch in order, so that at most one
// trajectory of it is there in part: seven workgroups at most for the XCD's 32 compute units, and four such launches at once (the
// queues a process has by default) have room.  More of them, a stream with a mask of few compute units, a device with fewer XCDs, or
// kernels of others that stay for long can keep a partner away.  A wait ends after most_polls looks; the workgroup then marks its
// own words, on which the others of the trajectory end too, and the launch behind this one computes the trajectory
// again with one workgroup: caches, draws and variates are the trajectory's own, so nothing of the first attempt is left.
// Where nothing was given up that launch only reads the words.
#pragma once

#include "trajectory_decode.h"

namespace artab {

// Whether these run here (G = 1) and not on one crew: both sides measured above.  The lines of 16 bits lie where a shared
// context crosses; contexts of their own cross later, but for those of nearly every compute unit, which together wait for memory
// and not for their units.
inline bool crews_serve(const TrajectoryParams &P, int D, bool f32) {
    const bool memory = P.own_base > 0 && P.B > 192;
    return P.G == 1 && (D == 128 || D == 256) &&
           (f32 || P.n_ctx + P.own_base + P.Nt / 2 <= (D == 128 ? (memory ? 448 : 2048) : (memory ? 704 : 768)));
}

// The first N of a buffer's fragments.
template <int N, int M>
__device__ __forceinline__ u32x4 (&first(u32x4 (&buf)[M]))[N] {
    static_assert(N <= M, "no more than there are");
    return reinterpret_cast<u32x4 (&)[N]>(buf);
}
// Sum and maximum over a row of 16 lanes.
__device__ __forceinline__ float lanes16_sum(float x) {
    x += row_rotate<8>(x);
    x += row_rotate<4>(x);
    x += row_rotate<2>(x);
    return x + row_rotate<1>(x);
}
__device__ __forceinline__ float lanes16_max(float x) {
    x = fmaxf(x, row_rotate<8>(x));
    x = fmaxf(x, row_rotate<4>(x));
    x = fmaxf(x, row_rotate<2>(x));
    return fmaxf(x, row_rotate<1>(x));
}

template <typename T, int D, int F, int PARTS>
__global__ __launch_bounds__(2 * kTrajWaves * 64) void trajectory_crews_kernel(TrajectoryParams P) {
    typedef TrajOps<T> Ops;
    typedef TrajShape<T, D, F> S;
    using std::integral_constant;
    constexpr int NW = kTrajWaves, NT = 2 * NW * 64, NTC = NW * 64, DH = 32, H = D / DH, NR = 2;  // NR: token rows
    constexpr bool k16 = sizeof(T) == 2;
    constexpr int LD = D + (k16 ? 8 : 4), LF = F + (k16 ? 8 : 4);  // row strides: 16 bytes off a multiple of 128
    constexpr int VW = D > F ? D : F;
    // Keys per block: one step of the second product's contraction.
    constexpr int BK = k16 ? 32 : 16;
    constexpr int HL = H / PARTS;                   // heads of this workgroup
    static_assert(HL <= NW && HL * PARTS == H, "a wavefront per head, or several");
    constexpr int NP = NW / HL;                     // wavefronts per head
    constexpr int VPAD = DH + 16;
    constexpr int GB = 4;  // blocks on their way per wavefront (and, in 16 bits, of one group of score products)
    // fragments of a product that are requested ahead: as many as the registers allow
    constexpr int kMost = 16;
    // q/k/v: 16-feature blocks of this workgroup's heads in one of the three, blocks per wavefront
    constexpr int BL = D / PARTS / 16, NQ = (3 * BL + NW - 1) / NW, kQkv = NQ * S::KD;
    static_assert(PARTS > 1 || NQ == 3 * S::ND, "all heads: the tape's own order");
    constexpr int wFo = S::kFo < kMost ? S::kFo : kMost, wQkv = kQkv < kMost ? kQkv : kMost, wO = S::kO < kMost ? S::kO : kMost,
                  w1 = S::k1 < kMost ? S::k1 : kMost, w2 = S::k2 < kMost ? S::k2 : kMost, wH2 = S::kH2 < w2 ? S::kH2 : w2;
    // where there is room beside others: W_2's together with W_o's, the first of q/k/v's together with W_2's, the keys
    // together with W_fo's
    constexpr bool kW2Early = wO + w2 <= 16, kKeysEarly = 4 * wFo + 8 * GB <= 64, kSpread = kKeysEarly && wFo <= 4;
    constexpr int kQkvEarly = wQkv + w2 <= 20 ? wQkv / 2 : 0, kQkvMid = kQkvEarly + (wQkv - kQkvEarly) / 2;

    __shared__ __attribute__((aligned(16))) T xs[NR * LD];   // layer input; attention output
    __shared__ __attribute__((aligned(16))) T ys[NR * LD];   // normed feature stage, then x1; z of the head
    constexpr int QKV = 3 * NR * LD, HID = NR * LF;
    __shared__ __attribute__((aligned(16))) T qkv[QKV > HID ? QKV : HID];  // q, k, v of the step; hidden layer
    T *const qs = qkv, *const kn = qkv + NR * LD, *const vn = qkv + 2 * NR * LD, *const hs = qkv;
    __shared__ __attribute__((aligned(16))) T v_lds[k16 ? NW * GB * BK * VPAD : 8];
    __shared__ float red_a[NW * NR], red_b[NW * NR];
    __shared__ __attribute__((aligned(16))) float part_o[NP > 1 ? NW * NR * DH : 4];
    __shared__ float part_m[NP > 1 ? NW * NR : 1], part_l[NP > 1 ? NW * NR : 1];
    __shared__ float raw_s[NR][kTrajHeadOut + 1];
    __shared__ float y_s, x_s[2];
    __shared__ float eps_s[3];  // (as kernel arguments they would be fetched again at every norm)
    // the parameter vectors of this layer and of the next; cache addresses of every layer
    __shared__ __attribute__((aligned(16))) T pbuf[2][8 * VW];
    __shared__ unsigned long long kv_s[4 * kTrajMaxLayers];
    __shared__ __attribute__((aligned(16))) T cst[TrajConstants<T, D, F>::kElems], tok_s[D];  // and the position token of the coming step
    const TrajConstants<T, D, F> C(cst);

    const int tid = threadIdx.x, warp = __builtin_amdgcn_readfirstlane(tid >> 6), wave = warp & (NW - 1), lane = tid & 63;
    const int ctid = tid & (NTC - 1);                       // within the crew
    // What a lane is, from an index the compiler cannot trace: it would keep every address it can derive from it
    // through the whole run, in registers that the fragments need.
    struct Lane {
        int lane;
        __device__ __forceinline__ int tok() const { return Ops::tok(lane); }        // output layout of the products
        __device__ __forceinline__ int sub() const { return Ops::sub(lane); }
        __device__ __forceinline__ int row() const { return lane & 1; }              // the token row of its results
        __device__ __forceinline__ bool writes() const { return tok() < NR && (k16 || lane < 16); }  // one of the lanes that hold the same
        __device__ __forceinline__ int row16() const { return lane & 15; }           // operand layout
        __device__ __forceinline__ int quad() const { return lane >> 4; }
    };
    auto here = [&]() { return Lane{opaque(tid & 63)}; };
    // The trajectory, and which of its workgroups this is.  Workgroups are started in order and dealt round-robin over
    // the eight XCDs: those of one trajectory come one after the other on one XCD.
    const int member = PARTS > 1 ? static_cast<int>(blockIdx.x >> 3) % PARTS : 0;
    const long b = PARTS > 1 ? static_cast<long>(blockIdx.x >> 3) / PARTS * 8 + (blockIdx.x & 7) : blockIdx.x;
    if (PARTS > 1 && b >= P.B) return;
    if constexpr (PARTS == 1)
        if (P.exchange && !traj_given_up<T, D, NT>(P.exchange, b, tid)) return;
    // looks that a wait for another workgroup may take; below zero once one was in vain, or another workgroup has given up
    __shared__ int patience_s;

    // Global memory by its address space: made from integers, plain pointers would be generic ones, whose loads count
    // as LDS accesses too, and every wait for LDS would wait for them.
    typedef __attribute__((address_space(1))) char *Global;
    typedef const __attribute__((address_space(1))) u32x4 *Global16;

    // ---- weights
    const Global tape = (Global)(reinterpret_cast<unsigned long long>(P.tape) + wave * static_cast<unsigned long long>(P.tape_stride));
    auto fragment = [&](int at, unsigned lane_byte) {
        const unsigned long long p = reinterpret_cast<unsigned long long>(tape) + static_cast<long>(at) * 1024;
        const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(p)), hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(p >> 32));
        return *(Global16)((Global)(static_cast<unsigned long long>(hi) << 32 | lo) + lane_byte);
    };
    // Where a product's fragments are, by number: one after the other on this wavefront's tape; of q/k/v, where several
    // workgroups share a trajectory, those of its own heads' blocks, on whichever tapes they are.
    auto run_at = [&](int at) { return [=](int n, unsigned lane_byte) { return fragment(at + n, lane_byte); }; };
    auto qkv_block = [&](int i) { return min(wave + NW * i, 3 * BL - 1); };  // (q's blocks, k's, v's; past the end the last one again)
    unsigned long long qkv_tape[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        const int m = qkv_block(i), c = member * BL + m % BL;  // the block's place among all of its matrix
        qkv_tape[i] = reinterpret_cast<unsigned long long>(P.tape) + (c % NW) * static_cast<unsigned long long>(P.tape_stride) +
                      static_cast<unsigned long long>(S::pQkv + m / BL * S::ND + c / NW) * 1024;
    }
    auto qkv_at = [&](int layer_at) {
        if constexpr (PARTS == 1) {
            return run_at(layer_at + S::pQkv);
        } else {
            return [=, &qkv_tape](int n, unsigned lane_byte) {
                const unsigned long long p = qkv_tape[n % NQ] + static_cast<long>(layer_at + n / NQ * 3 * S::ND) * 1024;
                const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(p)), hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(p >> 32));
                return *(Global16)((Global)(static_cast<unsigned long long>(hi) << 32 | lo) + lane_byte);
            };
        }
    };
    // Fragments FROM .. TO - 1 of a product.
    auto ask = [&](auto &buf, auto frag, auto from_, auto to_) {
        constexpr int FROM = decltype(from_)::value, TO = decltype(to_)::value;
        __builtin_amdgcn_sched_barrier(0);
        const unsigned lane_byte = 16 * here().lane;
#pragma unroll
        for (int i = FROM; i < TO; ++i) buf[i] = frag(i, lane_byte);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Values that nobody needs any more, where only one of two paths overwrites them: on the other one their registers
    // would be kept.
    auto forget = [](auto &buf) {
        for (auto &f : buf) {
            u32x4 any;
            asm volatile("" : "=v"(any));
            f = any;
        }
    };
    // acc[i] = W_i A^T over KS steps of NB blocks.  The buffer holds the first fragments; the others follow where there
    // is one free.
    auto product = [&](auto &acc, auto &buf, auto frag, auto ks_, const T *act, int ld) {
        constexpr int KS = decltype(ks_)::value, NB = sizeof(acc) / sizeof(acc[0]), W = sizeof(buf) / sizeof(buf[0]), N = KS * NB;
        constexpr int KC = KS < 4 ? KS : 4;  // activation operands are read KC steps at a time
        const Lane ln = here();
        const T *const a = act + ln.row() * ld + Ops::kPer * ln.quad();
        f32x4 odd[NB];  // (one block alone: two chains of products)
#pragma unroll
        for (int i = 0; i < NB; ++i) acc[i] = odd[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k0 = 0; k0 < KS; k0 += KC) {
            u32x4 bf[KC];
#pragma unroll
            for (int k = 0; k < KC; ++k) bf[k] = *reinterpret_cast<const u32x4 *>(a + Ops::kStep * (k0 + k));
#pragma unroll
            for (int k = 0; k < KC; ++k)
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const int n = (k0 + k) * NB + i;
                    if (NB == 1 && (k & 1)) odd[i] = Ops::mma(buf[n % W], bf[k], odd[i]);
                    else acc[i] = Ops::mma(buf[n % W], bf[k], acc[i]);
                    if (n + W < N) buf[n % W] = frag(n + W, 16 * ln.lane);
                }
            if (N > W) __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (NB == 1) acc[0] += odd[0];
#pragma unroll
        for (int i = 0; i < NB; ++i) Ops::finish(acc[i]);
    };
    // LayerNorm of v (this lane's features of its token row): this wavefront's mean and squares, a barrier, the result.
    auto norm_sums = [&](auto &v) {
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
        const Lane ln = here();
        if (ln.writes() && ln.sub() == 0) {
            red_a[wave * NR + ln.row()] = lmean;
            red_b[wave * NR + ln.row()] = q;
        }
    };
    auto norm_store = [&](auto &v, const T *gam, const T *bet, const float *eps_at, T *dst) {
        constexpr int NB = sizeof(v) / sizeof(v[0]);
        constexpr float kLocal = NB * 16;
        const Lane ln = here();
        const float eps = *eps_at;
        float g[NB][4], be[NB][4];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int col = 16 * (wave + NW * b) + 4 * ln.sub();
            traj_load4<T>(gam + col, g[b]);
            traj_load4<T>(bet + col, be[b]);
        }
        // a row of 16 lanes holds the eight wavefronts' pairs of both token rows
        const float lm = red_a[ln.row16()], lq = red_b[ln.row16()];
        auto wavefronts = [](float x) {  // over the lanes of one parity
            x += row_rotate<2>(x);
            x += row_rotate<4>(x);
            return x + row_rotate<8>(x);
        };
        const float mean = wavefronts(lm) * (1.f / NW), d = lm - mean, squares = wavefronts(fmaf(kLocal * d, d, lq));
        const float rstd = __builtin_amdgcn_rsqf(fmaf(squares, 1.f / D, eps));
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (v[b][e] - mean) * rstd * g[b][e] + be[b][e];
            if (ln.writes()) traj_store4<T>(dst + ln.row() * LD + 16 * (wave + NW * b) + 4 * ln.sub(), o);
        }
    };
    // gelu, stored to the hidden tile.  The values of the two tokens stand in several lanes: in 16 bits all eight of them
    // in the eight column pairs, in float32 in two column pairs of four rows of lanes.  Each lane does one.
    auto gelu_store = [&](auto &acc, const T *bias) {
        static_assert(sizeof(acc) / sizeof(acc[0]) == 2, "two blocks of hidden features per wavefront");
        const Lane ln = here();
        const int tok = ln.tok(), e = k16 ? (tok >> 1) & 3 : ln.quad(), i = k16 ? tok >> 3 : tok >> 1;
        const float a0 = (e & 1) ? acc[0][1] : acc[0][0], a1 = (e & 1) ? acc[0][3] : acc[0][2], c0 = (e & 1) ? acc[1][1] : acc[1][0],
                    c1 = (e & 1) ? acc[1][3] : acc[1][2];
        const float a = (e & 2) ? a1 : a0, c = (e & 2) ? c1 : c0;
        const int col = 16 * (wave + NW * i) + 4 * ln.sub() + e;
        const float x = (i ? c : a) + to_f32(bias[col]);
        hs[ln.row() * LF + col] = from_f32<T>(k16 ? traj_gelu16(x) : 0.5f * x * (1.f + erff(x * 0.70710678118654752f)));
    };

    // ---- attention (crew 1): committed rows, then the rows of this step
    const int part = wave / HL;
    const int head0 = member * HL + wave % HL;
    const int first_block = part;  // the wavefront's blocks: this one and every NP-th
    T *const vt = v_lds + (k16 ? wave * GB * BK * VPAD : 0);
    constexpr unsigned RB = DH * sizeof(T);  // bytes of a row
    Global hk[4];  // the head's rows in the layer's caches: the context's keys and values, the trajectory's
    // Blocks by number: the context's, then the trajectory's.
    const int nb_ctx = (P.n_ctx + BK - 1) / BK;
    int n_own = 0, n_mine = 0, pad = 0;
    auto layer_kv = [&](int l, int i) {
        const unsigned long long raw = kv_s[4 * l + i];
        const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(raw)),
                       hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(raw >> 32));
        return (Global)(static_cast<unsigned long long>(hi) << 32 | lo);
    };
    // What the attention of head h of layer l in step t will read.  n_mine: the wavefront's blocks; its first group
    // leaves out `pad` positions, the later ones are whole.
    auto prepare = [&](int h, int l, int t) {
        n_own = P.own_base + (t > 0 ? t - 1 : 0);
        const int blocks = nb_ctx + (n_own + BK - 1) / BK;
        n_mine = blocks > first_block ? (blocks - first_block + NP - 1) / NP : 0;
        pad = (GB - n_mine % GB) % GB;
        const long ctx = static_cast<long>(h) * P.ctx_rows * RB, own = (b * H + h) * P.own_rows * static_cast<long>(RB);
#pragma unroll
        for (int i = 0; i < 4; ++i) hk[i] = layer_kv(l, i) + (i < 2 ? ctx : own);
    };
    // Block n of the wavefront: the context's or the trajectory's, its first row, the rows of that segment.
    struct Where {
        bool ctx;
        int row0, rows;
    };
    auto where = [&](int n) {
        const int i = first_block + NP * n;
        const bool ctx = i < nb_ctx;
        return Where{ctx, BK * (ctx ? i : i - nb_ctx), ctx ? P.n_ctx : n_own};
    };
    // 16 bytes (float32 values: one) of row `lane_row` of a block; rows past a segment's end re-read its last one
    auto address = [&](const Where &w, int which, int lane_row, int lane_byte) {
        return (w.ctx ? hk[which] : hk[2 + which]) + (static_cast<unsigned>(min(w.row0 + lane_row, w.rows - 1)) * RB + lane_byte);
    };
    // A block as it comes from memory: keys in operand order; values in rows (16-bit) or as the operand of the second
    // product (float32).
    struct Keys {
        u32x4 k[2], v[2];
    };
    auto key_half = [&](const Where &w, int ln, int x) {
        return *(Global16)(k16 ? address(w, 0, 16 * x + (ln & 15), 16 * (ln >> 4)) : address(w, 0, ln & 15, 16 * (ln >> 4) + 64 * x));
    };
    auto value_half = [&](const Where &w, int ln, int x) {
        if constexpr (k16) {
            return *(Global16)address(w, 1, 16 * x + (ln & 15), 16 * (ln >> 4));
        } else {
            u32x4 r;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                r[j] = *(const __attribute__((address_space(1))) unsigned *)address(w, 1, 4 * (ln >> 4) + j, 4 * (ln & 15) + 64 * x);
            return r;
        }
    };
    // The first group (the positions it leaves out are the oldest, so that what is on its way stays countable).
    auto ask_keys = [&](Keys (&r)[GB], auto from_, auto to_) {
        __builtin_amdgcn_sched_barrier(0);
        const int ln = here().lane;
#pragma unroll
        for (int j = decltype(from_)::value; j < decltype(to_)::value; ++j)
            if (j >= pad && j - pad < n_mine) {
                const Where w = where(j - pad);
#pragma unroll
                for (int x = 0; x < 2; ++x) r[j].k[x] = key_half(w, ln, x);
            } else {
                r[j].k[0] = r[j].k[1] = u32x4{0u, 0u, 0u, 0u};
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto ask_values = [&](Keys (&r)[GB], auto from_, auto to_) {
        __builtin_amdgcn_sched_barrier(0);
        const int ln = here().lane;
#pragma unroll
        for (int j = decltype(from_)::value; j < decltype(to_)::value; ++j)
            if (j >= pad && j - pad < n_mine) {
                const Where w = where(j - pad);
#pragma unroll
                for (int x = 0; x < 2; ++x) r[j].v[x] = value_half(w, ln, x);
            } else {
                r[j].v[0] = r[j].v[1] = u32x4{0u, 0u, 0u, 0u};
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    // A head's sums (token tok < NR, dims 4 sub + e of both halves) become its rows of the attention output;
    // with several wavefronts per head through LDS (put, a barrier, take).
    float a_m = -1e30f, a_l = 0.f;
    f32x4 a_o[2];
    auto attention_put = [&]() {
        const Lane ln = here();
        const int tok = ln.tok(), sub = ln.sub();
        if (part > 0 && ln.writes()) {
            if (sub == 0) {
                part_m[wave * NR + tok] = a_m;
                part_l[wave * NR + tok] = a_l;
            }
#pragma unroll
            for (int db = 0; db < 2; ++db) *reinterpret_cast<f32x4 *>(part_o + (wave * NR + tok) * DH + 16 * db + 4 * sub) = a_o[db];
        }
    };
    // ---- what the workgroups of a trajectory give each other: their heads' attention output, as 8-byte words of values and
    // the number of the exchange, stored and read with relaxed device-wide atomics.  A word is its own signal: no fence, no
    // counter, one trip through the memory side.  Two sets of words, in turn: who sends exchange n + 2 has every word of
    // n + 1, and whoever sent those had all words of n.
    constexpr int VPW = k16 ? 2 : 1, WORDS = NR * D / VPW;  // values per word, words per exchange
    static_assert(WORDS <= NTC, "one word per thread of a crew");
    auto words = [&](unsigned tag) { return P.exchange + (2 * b + (tag & 1)) * WORDS; };
    auto send = [&](int row, int col, const float (&o)[4], unsigned tag) {
        if (patience_s < 0) return;  // (what it would send is not the trajectory's)
        unsigned long long *const at = words(tag) + (row * D + col) / VPW;
#pragma unroll
        for (int i = 0; i < 4 / VPW; ++i) {
            unsigned value;
            if constexpr (k16) value = pack2<T>(o[2 * i], o[2 * i + 1]);
            else value = __builtin_bit_cast(unsigned, o[i]);
            __hip_atomic_store(at + i, static_cast<unsigned long long>(tag) << 32 | value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    auto receive = [&](unsigned tag) {
        const int i = ctid, row = i / (WORDS / NR), col = i % (WORDS / NR) * VPW;
        if (i >= WORDS || col / (D / PARTS) == member) return;
        const unsigned long long *const at = words(tag) + i;
        unsigned long long v = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // (every wait ends: the step is then finished with what there is, nobody uses it)
        for (int looks = patience_s; static_cast<unsigned>(v >> 32) != tag; --looks) {
            if (looks <= 0 || static_cast<unsigned>(v >> 32) == kTrajGone) {
                patience_s = -1;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
            v = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const unsigned value = static_cast<unsigned>(v);
        *reinterpret_cast<unsigned *>(xs + row * LD + col) = value;
    };
    auto attention_take = [&](int h, unsigned tag) {
        const Lane ln = here();
        const int tok = ln.tok(), sub = ln.sub();
        if ((NP == 1 || part == 0) && ln.writes()) {
            if constexpr (NP > 1) {  // the other wavefronts' keys of this head
#pragma unroll
                for (int p = 1; p < NP; ++p) {
                    const int w = wave + p * HL;
                    const float m2 = part_m[w * NR + tok], l2 = part_l[w * NR + tok];
                    const float m_new = fmaxf(a_m, m2);
                    const float a1 = fast_exp2(a_m - m_new), a2 = fast_exp2(m2 - m_new);
#pragma unroll
                    for (int db = 0; db < 2; ++db) {
                        const f32x4 o2 = *reinterpret_cast<const f32x4 *>(part_o + (w * NR + tok) * DH + 16 * db + 4 * sub);
#pragma unroll
                        for (int e = 0; e < 4; ++e) a_o[db][e] = a_o[db][e] * a1 + o2[e] * a2;
                    }
                    a_l = a_l * a1 + l2 * a2;
                    a_m = m_new;
                }
            }
            const float inv = a_l > 0.f ? 1.f / a_l : 0.f;
#pragma unroll
            for (int db = 0; db < 2; ++db) {
                const float o[4] = {a_o[db][0] * inv, a_o[db][1] * inv, a_o[db][2] * inv, a_o[db][3] * inv};
                traj_store4<T>(xs + tok * LD + DH * h + 16 * db + 4 * sub, o);
                if constexpr (PARTS > 1) send(tok, DH * h + 16 * db + 4 * sub, o, tag);
            }
        }
    };
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    auto tr_read = [](const T *a) {
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(a));
    };
    // The wavefront's blocks, group by group: `group(more, n0)` takes blocks n0 .. n0 + GB - 1 (those below 0 do not
    // exist) and, with `more`, asks for the next GB.
    auto groups = [&](auto group) {
        int n0 = -pad;
        for (; n0 + GB < n_mine; n0 += GB) group(std::true_type{}, n0);
        if (n0 < n_mine) group(std::false_type{}, n0);
    };

    // One trajectory in 16 bits.  Its two queries stand in all eight column pairs of a score product; of the products of
    // 2 GB 16-key parts, pair x keeps part x's.  A lane then holds four scores of the group, all of them used, where it
    // held 32; the second products take part x's probabilities in pair x's columns and zeros in the others.
    auto attention_16 = [&](int h, int t, auto &keys) {
        const Lane me = here();
        const int lane = me.lane, row16 = me.row16(), quad = me.quad(), pair = row16 >> 1;
        const u32x4 q2 = *reinterpret_cast<const u32x4 *>(qs + (row16 & 1) * LD + DH * h + Ops::kPer * quad);
        const unsigned one2 = pack2<T>(1.f, 1.f);
        const u32x4 ones = {one2, one2, one2, one2};
        f32x4 o_acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}}, l_acc = {0.f, 0.f, 0.f, 0.f};
        // The reference of a token's probabilities, the same in its eight columns.  The step's own buffer row comes
        // first, while the first group is on its way.
        float m_run = -1e30f;
        if (t > 0 && (NP == 1 || part == 0)) {
            const f32x4 sc = Ops::mma(*reinterpret_cast<const u32x4 *>(kn + (row16 & 1) * LD + DH * h + Ops::kPer * quad), q2, f32x4{0.f, 0.f, 0.f, 0.f});
            const float s0 = row_sum(quad == 0 ? sc[0] : 0.f);
            float vr[2][4];
#pragma unroll
            for (int db = 0; db < 2; ++db) traj_load4<T>(vn + DH * h + 16 * db + 4 * quad, vr[db]);
            m_run = fmaxf(s0, -1e30f);
            const float p = pair == 0 ? to_f32(from_f32<T>(fast_exp2(s0 - m_run))) : 0.f;
            l_acc[0] = p;
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int e = 0; e < 4; ++e) o_acc[db][e] = pair == 0 ? p * vr[db][e] : 0.f;
        }
        groups([&](auto more, int n0) {
            const Lane me = here();
            const int pair = me.row16() >> 1;
            // part x's scores stand in every column pair (q2 does); pair x keeps them
            f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < GB; ++j) {
                f32x4 both[2];
#pragma unroll
                for (int x = 0; x < 2; ++x) both[x] = Ops::mma(keys[j].k[x], q2, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float one = (pair & 1) ? both[1][e] : both[0][e];
                    s[e] = j == 0 || (pair >> 1) == j ? one : s[e];
                }
                if constexpr (decltype(more)::value) {
                    const Where w = where(n0 + j + GB);
#pragma unroll
                    for (int x = 0; x < 2; ++x) keys[j].k[x] = key_half(w, lane, x);
                }
            }
            // the values become rows in LDS meanwhile
#pragma unroll
            for (int j = 0; j < GB; ++j) {
#pragma unroll
                for (int x = 0; x < 2; ++x)
                    *reinterpret_cast<u32x4 *>(vt + (j * BK + 16 * x + me.row16()) * VPAD + 8 * me.quad()) = keys[j].v[x];
                if constexpr (decltype(more)::value) {
                    const Where w = where(n0 + j + GB);
#pragma unroll
                    for (int x = 0; x < 2; ++x) keys[j].v[x] = value_half(w, lane, x);
                }
            }
            __builtin_amdgcn_wave_barrier();
            {   // keys past the end of their segment, parts that do not exist
                const int n = n0 + (pair >> 1), i = first_block + NP * n;
                const int rows = i < nb_ctx ? P.n_ctx - BK * i : n_own - BK * (i - nb_ctx);
                const int mine = (n < 0 || pair >= 2 * GB ? 0 : rows) - 16 * (pair & 1) - 4 * me.quad();
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] = e < mine ? s[e] : -INFINITY;
            }
            float top = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
            if (__any(top > m_run + Ops::kSlack)) {
                top = row_max(top);
                top = fmaxf(top, row_rotate<2>(top));
                top = fmaxf(top, row_rotate<4>(top));
                top = fmaxf(fmaxf(top, row_rotate<8>(top)), m_run);
                const float alpha = fast_exp2(m_run - top);
                l_acc[0] *= alpha;
#pragma unroll
                for (int db = 0; db < 2; ++db)
#pragma unroll
                    for (int e = 0; e < 4; ++e) o_acc[db][e] *= alpha;
                m_run = top;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = fast_exp2(s[e] - m_run);
            const unsigned p01 = pack2<T>(s[0], s[1]), p23 = pack2<T>(s[2], s[3]);
            l_acc = Ops::mma(ones, u32x4{p01, p23, 0u, 0u}, l_acc);  // summed as the products take them, rounded
#pragma unroll
            for (int j = 0; j < GB; ++j) {
                const bool lo = pair == 2 * j, hi = pair == 2 * j + 1;
                const u32x4 pv = {lo ? p01 : 0u, lo ? p23 : 0u, hi ? p01 : 0u, hi ? p23 : 0u};
                const T *a = vt + (j * BK + 4 * me.quad() + (me.row16() >> 2)) * VPAD + 4 * (me.lane & 3);
#pragma unroll
                for (int db = 0; db < 2; ++db) {
                    const s16x4 lo4 = tr_read(a + 16 * db), hi4 = tr_read(a + 16 * db + 16 * VPAD);
                    const s16x8 both = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
                    o_acc[db] = Ops::mma(__builtin_bit_cast(u32x4, both), pv, o_acc[db]);
                }
            }
            __builtin_amdgcn_wave_barrier();
        });
        // the eight columns of a token
        auto columns = [](float x) {
            x += row_rotate<2>(x);
            x += row_rotate<4>(x);
            return x + row_rotate<8>(x);
        };
        a_m = m_run;
        a_l = columns(l_acc[0]);
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
            for (int e = 0; e < 4; ++e) a_o[db][e] = columns(o_acc[db][e]);
    };

    // The same in float32: the two tokens are columns 0 and 1 of four (and 2 and 3 again); 16 keys per block.
    auto attention_f32 = [&](int h, int t, auto &keys) {
        const Lane me = here();
        const int lane = me.lane, quad = me.quad(), sub = me.sub();
        u32x4 qf[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) qf[x] = *reinterpret_cast<const u32x4 *>(qs + me.row() * LD + DH * h + Ops::kStep * x + Ops::kPer * quad);
        f32x4 o_acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
        float m_run = -1e30f, l_run = 0.f;
        // Scores (lane: keys 4 sub + r, its token) to probabilities.
        auto fold = [&](f32x4 &sc) {
            const float top = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
            if (__any(top > m_run + Ops::kSlack)) {
                const float m_new = fmaxf(m_run, Ops::max(top)), alpha = fast_exp2(m_run - m_new);
                l_run *= alpha;
#pragma unroll
                for (int db = 0; db < 2; ++db)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o_acc[db][r] *= alpha;
                m_run = m_new;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[r] = fast_exp2(sc[r] - m_run);
            l_run += (sc[0] + sc[1]) + (sc[2] + sc[3]);
        };
        if (t > 0 && (NP == 1 || part == 0)) {  // the step's own buffer row, while the first group is on its way
            const T *const kr = kn + me.row() * LD + DH * h + Ops::kPer * quad;
            f32x4 sc = Ops::mma(*reinterpret_cast<const u32x4 *>(kr), qf[0], f32x4{0.f, 0.f, 0.f, 0.f});
            sc = Ops::mma(*reinterpret_cast<const u32x4 *>(kr + 16), qf[1], sc);
            Ops::finish(sc);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * sub + e != 0) sc[e] = -INFINITY;
            float vr[2][4];
#pragma unroll
            for (int db = 0; db < 2; ++db) traj_load4<T>(vn + DH * h + 16 * db + 4 * sub, vr[db]);
            fold(sc);
            const float p = Ops::sum((sc[0] + sc[1]) + (sc[2] + sc[3]));
            if (quad == 0) {  // (the four rows of lanes are partial sums)
#pragma unroll
                for (int db = 0; db < 2; ++db)
#pragma unroll
                    for (int e = 0; e < 4; ++e) o_acc[db][e] = fmaf(p, vr[db][e], o_acc[db][e]);
            }
        }
        // the probabilities of keys 4 (lane / 16) + j for this lane's token
        const int p_from = ((lane & 48) | (quad << 2) | (lane & 3)) << 2;
        groups([&](auto more, int n0) {
#pragma unroll
            for (int j = 0; j < GB; ++j) {
                if (n0 + j >= 0) {
                    const Where w = where(n0 + j);
                    f32x4 sc = Ops::mma(keys[j].k[0], qf[0], f32x4{0.f, 0.f, 0.f, 0.f});
                    sc = Ops::mma(keys[j].k[1], qf[1], sc);
                    Ops::finish(sc);
                    if (w.row0 + BK > w.rows) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (w.row0 + 4 * sub + e >= w.rows) sc[e] = -INFINITY;
                    }
                    fold(sc);
                    u32x4 pv;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float pe = sc[e];
                        pv[e] = __builtin_amdgcn_ds_bpermute(p_from, __builtin_bit_cast(int, pe));
                    }
#pragma unroll
                    for (int db = 0; db < 2; ++db) o_acc[db] = Ops::mma(keys[j].v[db], pv, o_acc[db]);
                }
                if constexpr (decltype(more)::value) {
                    const Where w = where(n0 + j + GB);
#pragma unroll
                    for (int x = 0; x < 2; ++x) {
                        keys[j].k[x] = key_half(w, lane, x);
                        keys[j].v[x] = value_half(w, lane, x);
                    }
                }
            }
        });
        a_m = m_run;
        a_l = Ops::sum(l_run);
#pragma unroll
        for (int db = 0; db < 2; ++db) {
            Ops::finish(o_acc[db]);
            a_o[db] = o_acc[db];
        }
    };
    auto attention = [&](int h, int t, auto &keys) {
        if constexpr (k16) attention_16(h, t, keys);
        else attention_f32(h, t, keys);
    };

    // ---- constants, the first layer's vectors, the embedding of step 0: the target row; the other one is zero
    constexpr int kPieces = 8 * VW * static_cast<int>(sizeof(T)) / 16;  // of a layer's vectors
    static_assert(kPieces <= NTC, "one piece per thread of a crew");
    const u32x4 *const vec_src = static_cast<const u32x4 *>(P.vecs);
    if (tid < kPieces) reinterpret_cast<u32x4 *>(pbuf[0])[tid] = vec_src[tid];
    for (int i = tid; i < 4 * P.n_layers; i += NT) kv_s[i] = P.kv[i];
    const T *const xm = static_cast<const T *>(P.x_mean);
    C.template load<NT>(P, tid);
    if (tid == 0) {
        eps_s[0] = P.eps1;
        eps_s[1] = P.eps2;
        eps_s[2] = P.eps3;
        if constexpr (PARTS > 1) patience_s = P.most_polls;
    }
    __syncthreads();
    C.template first_rows<NT>(P, b, 1, NR, xs, LD, tid);
    __syncthreads();

    // ---- the run, written once for both crews: every barrier is one of both.
    auto run = [&](auto crew_) {
        constexpr int CREW = decltype(crew_)::value;
        constexpr bool kA = CREW == 0, kB = CREW == 1;
        // fragments on their way
        u32x4 f_qkv[kA ? wQkv : 1], f_o[kA ? wO : 1], f_2[kA ? w2 : 1];
        constexpr int wB = wFo > w1 ? wFo : w1;  // W_fo's, W_1's or the head's
        u32x4 f_b[kB ? wB : 1];
        Keys keys[kB ? GB : 1];
        constexpr integral_constant<int, 0> from0{};
        constexpr integral_constant<int, GB> all_blocks{};
        const int head_at = P.n_layers * S::kLayer;
        if constexpr (kA) ask(f_qkv, qkv_at(0), from0, integral_constant<int, kQkvEarly>{});
        if constexpr (kB) {
            ask(f_b, run_at(S::pFo), from0, integral_constant<int, wFo>{});
            prepare(head0, 0, 0);
            if constexpr (kKeysEarly) {
                ask_keys(keys, from0, all_blocks);
                if constexpr (kSpread) ask_values(keys, from0, integral_constant<int, GB / 2>{});
            }
        }
        int pp = 0;  // which of the two vector buffers holds this layer's
        for (int t = 0; t < P.Nt; ++t) {
            const bool last_step = t + 1 == P.Nt;
            // the variates and feature means of the step's draw, long before they are needed
            float my_u = 0.f, my_n = 0.f;
            T my_x = from_f32<T>(0.f), my_tok = my_x;
            if constexpr (kA) {
                if (wave == 0) {
                    const long at = static_cast<long>(t) * P.B + b;
                    my_u = P.rand_u[at];
                    my_n = P.rand_n_f32 ? static_cast<const float *>(P.rand_n)[at] : to_f32(static_cast<const T *>(P.rand_n)[at]);
                }
                if (ctid < 2 && !last_step) my_x = xm[b * P.Nt + t + ctid];
                if (ctid < D) my_tok = static_cast<const T *>(P.ar_tokens)[static_cast<long>((t + 1) % P.bs) * D + ctid];
            }
            for (int l = 0; l < P.n_layers; ++l) {
                const T *const vec = pbuf[pp];
                int at = l * S::kLayer;
                asm volatile("" : "+s"(at));  // (or every fragment gets a pointer of its own, carried from layer to layer)
                const bool last_layer = l + 1 == P.n_layers;
                float v[S::ND][4];
                auto residual = [&](const T *res) {  // (read ahead of the product)
                    const Lane ln = here();
#pragma unroll
                    for (int b = 0; b < S::ND; ++b) traj_load4<T>(res + ln.row() * LD + 16 * (wave + NW * b) + 4 * ln.sub(), v[b]);
                };
                auto add = [&](const f32x4 (&acc)[S::ND]) {
#pragma unroll
                    for (int b = 0; b < S::ND; ++b)
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[b][e] = acc[b][e] + v[b][e];
                };
                // y = LN1(x + x W_fo^T)
                if constexpr (kB) {
                    f32x4 acc[S::ND];
                    residual(xs);
                    product(acc, first<wFo>(f_b), run_at(at + S::pFo), integral_constant<int, S::KD>{}, xs, LD);
                    add(acc);
                    norm_sums(v);
                } else {
                    ask(f_qkv, qkv_at(at), integral_constant<int, kQkvEarly>{}, integral_constant<int, kQkvMid>{});
                }
                __syncthreads();
                if constexpr (kB) norm_store(v, vec, vec + VW, eps_s, ys);
                else ask(f_qkv, qkv_at(at), integral_constant<int, kQkvMid>{}, integral_constant<int, wQkv>{});
                __syncthreads();
                // q, k, v
                if constexpr (kA) {
                    f32x4 acc[NQ];
                    product(acc, f_qkv, qkv_at(at), integral_constant<int, S::KD>{}, ys, LD);
                    const Lane ln = here();
#pragma unroll
                    for (int i = 0; i < NQ; ++i) {
                        // part of q/k/v and 16-feature block in it
                        const int m = qkv_block(i), p = PARTS == 1 ? i / S::ND : m / BL, c = PARTS == 1 ? wave + NW * (i % S::ND) : member * BL + m % BL;
                        float o[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            o[e] = acc[i][e];
                            if (p == 0) o[e] = to_f32(from_f32<T>(o[e])) * P.qscale;
                        }
                        if (ln.writes()) traj_store4<T>(qkv + p * NR * LD + ln.row() * LD + 16 * c + 4 * ln.sub(), o);
                    }
                } else {
                    if constexpr (!kKeysEarly) ask_keys(keys, from0, all_blocks);
                    ask_values(keys, integral_constant<int, kSpread ? GB / 2 : 0>{}, all_blocks);
                }
                __syncthreads();
                u32x4 next_vec = {0u, 0u, 0u, 0u};
                if constexpr (kA) {
                    ask(f_o, run_at(at + S::pO), from0, integral_constant<int, wO>{});
                    if (ctid < kPieces) next_vec = vec_src[(last_layer ? 0 : l + 1) * kPieces + ctid];
                    if constexpr (kW2Early) ask(f_2, run_at(at + S::p2), from0, integral_constant<int, w2>{});
                    // the caches: row 0 is committed at slot t - 1 (its first read is a step away); behind the last one
                    // the target row, where the caller keeps it
                    auto commit = [&](int from, int slot) {
                        traj_commit<T, D, NTC, HL>(layer_kv(l, 2), layer_kv(l, 3), kn, vn, LD, b, 1, P.own_rows, from, slot, ctid, member * HL);
                    };
                    if (t > 0) commit(0, P.own_base + t - 1);
                    if (P.park_target && last_step) commit(1, P.own_base + t);
                } else {
                    attention(head0, t, keys);
                    if constexpr (NP > 1) attention_put();
                }
                if constexpr (NP > 1) __syncthreads();
                const unsigned tag = static_cast<unsigned>(t * P.n_layers + l) + 1u;  // of this exchange
                if constexpr (kB) attention_take(head0, tag);
                else if constexpr (PARTS > 1) receive(tag);
                __syncthreads();
                // x1 = LN2(y + attn W_o^T)
                if constexpr (kA) {
                    f32x4 acc[S::ND];
                    residual(ys);
                    product(acc, f_o, run_at(at + S::pO), integral_constant<int, S::KD>{}, xs, LD);
                    add(acc);
                    norm_sums(v);
                } else {
                    prepare(head0, last_layer ? 0 : l + 1, last_layer ? t + 1 : t);
                    ask(f_b, run_at(at + S::p1), from0, integral_constant<int, w1 / 2>{});
                }
                __syncthreads();
                if constexpr (kA) norm_store(v, vec + 2 * VW, vec + 3 * VW, eps_s + 1, ys);
                else ask(f_b, run_at(at + S::p1), integral_constant<int, w1 / 2>{}, integral_constant<int, w1>{});
                if constexpr (kB && kSpread) ask_keys(keys, from0, integral_constant<int, GB / 2>{});
                __syncthreads();
                // h = gelu(x1 W_1^T + b_1)
                if constexpr (kB) {
                    f32x4 acc[S::NF];
                    product(acc, first<w1>(f_b), run_at(at + S::p1), integral_constant<int, S::KD>{}, ys, LD);
                    gelu_store(acc, vec + 4 * VW);
                } else {
                    if (ctid < kPieces) reinterpret_cast<u32x4 *>(pbuf[pp ^ 1])[ctid] = next_vec;
                    if constexpr (!kW2Early) ask(f_2, run_at(at + S::p2), from0, integral_constant<int, w2>{});
                    forget(f_qkv);
                    if (kQkvEarly > 0 && !last_layer) ask(f_qkv, qkv_at(at + S::kLayer), from0, integral_constant<int, kQkvEarly>{});
                }
                __syncthreads();
                // x = LN3(x1 + h W_2^T + b_2)
                if constexpr (kA) {
                    f32x4 acc[S::ND];
                    float bias[S::ND][4];
                    residual(ys);
                    const Lane ln = here();
#pragma unroll
                    for (int b = 0; b < S::ND; ++b) traj_load4<T>(vec + 7 * VW + 16 * (wave + NW * b) + 4 * ln.sub(), bias[b]);
                    product(acc, f_2, run_at(at + S::p2), integral_constant<int, S::KF>{}, hs, LF);
                    add(acc);
#pragma unroll
                    for (int b = 0; b < S::ND; ++b)
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[b][e] += bias[b][e];
                    norm_sums(v);
                } else {
                    forget(f_b);
                    if (last_layer) ask(f_b, run_at(head_at), from0, integral_constant<int, w1>{});
                    else ask(f_b, run_at(at + S::kLayer + S::pFo), from0, integral_constant<int, wFo>{});
                    if constexpr (kSpread) ask_keys(keys, integral_constant<int, GB / 2>{}, all_blocks);
                }
                __syncthreads();
                if constexpr (kA) {
                    norm_store(v, vec + 5 * VW, vec + 6 * VW, eps_s + 2, xs);
                } else {
                    if constexpr (kSpread) ask_values(keys, from0, integral_constant<int, GB / 2>{});
                    else if constexpr (kKeysEarly) ask_keys(keys, from0, all_blocks);
                }
                __syncthreads();
                pp ^= 1;
            }

            // ---- the head on the target rows, one draw per trajectory, the rows of the next step
            if constexpr (kA) ask(f_2, run_at(head_at + S::kH1), from0, integral_constant<int, wH2>{});
            {
                constexpr int EPL = D / 64;
                if (const int r = warp; r < NR) {
                    const T *src = xs + r * LD + lane * EPL;
                    float x[EPL], sum = 0.f;
#pragma unroll
                    for (int e = 0; e < EPL; ++e) {
                        x[e] = to_f32(src[e]);
                        sum += x[e];
                    }
                    const float mean = row_sum(lanes16_sum(sum)) / D;
                    float q = 0.f;
#pragma unroll
                    for (int e = 0; e < EPL; ++e) q += (x[e] - mean) * (x[e] - mean);
                    const float rstd = rsqrtf(row_sum(lanes16_sum(q)) / D + P.eps_out);
#pragma unroll
                    for (int e = 0; e < EPL; ++e) ys[r * LD + lane * EPL + e] = C.normed(x[e], mean, rstd, lane * EPL + e);
                }
            }
            __syncthreads();
            if constexpr (kB) {
                f32x4 acc[S::NF];
                product(acc, first<w1>(f_b), run_at(head_at), integral_constant<int, S::KD>{}, ys, LD);
                gelu_store(acc, C.b1);
            }
            __syncthreads();
            if constexpr (kA) {
                f32x4 acc[1];
                product(acc, first<wH2>(f_2), run_at(head_at + S::kH1), integral_constant<int, S::KF>{}, hs, LF);
                const Lane ln = here();
                if (16 * wave < kTrajHeadOut && ln.writes()) {
                    float bias[4];
                    traj_load4<T>(C.b2 + 16 * wave + 4 * ln.sub(), bias);
#pragma unroll
                    for (int e = 0; e < 4; ++e) raw_s[ln.row()][16 * wave + 4 * ln.sub() + e] = acc[0][e] + bias[e];
                }
                if (ctid < 2) x_s[ctid] = to_f32(my_x);
                if (ctid < D) tok_s[ctid] = my_tok;
            } else {
                ask(f_b, run_at(S::pFo), from0, integral_constant<int, wFo>{});
            }
            __syncthreads();
            if constexpr (kA) {
                ask(f_qkv, qkv_at(0), from0, integral_constant<int, kQkvEarly>{});
                if (wave == 0) {  // a lane per component
                    const float *raw = raw_s[1];
                    const T *const mix = C.mix;
                    const int k = min(lane, P.K - 1);
                    const float logit = raw[3 * k + 2] + to_f32(mix[2 * P.K + k]);
                    const float mx = row_max(lanes16_max(logit));
                    const float e = expf(logit - mx);
                    // sums in the components' order
                    float cum = 0.f, upto = 0.f;
                    for (int i = 0; i < P.K; ++i) {
                        cum += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, e), i));
                        upto = lane == i ? cum : upto;
                    }
                    const unsigned long long past = __ballot(lane < P.K && upto > my_u * cum);
                    const int comp = past ? __builtin_ctzll(past) : P.K - 1;
                    const T y = C.value(P, raw, comp, my_n);
                    if (lane == 0) {
                        if (member == 0) static_cast<T *>(P.preds)[b * P.Nt + t] = y;  // (all of them have drawn it)
                        y_s = to_f32(y);
                    }
                }
            }
            __syncthreads();
            // (last written several barriers ago: all threads see the same)
            if (last_step || (PARTS > 1 && __builtin_amdgcn_readfirstlane(patience_s) < 0)) break;
            C.template next_rows<NT>(x_s, &y_s, tok_s, 1, xs, LD, tid);
            __syncthreads();
        }
    };
    if (warp < NW) run(integral_constant<int, 0>{});
    else run(integral_constant<int, 1>{});
    if constexpr (PARTS > 1) {
        if (patience_s < 0) {  // given up: mark this workgroup's words of both sets
            constexpr int MINE = D / PARTS / VPW;
            for (int i = tid; i < 2 * NR * MINE; i += NT)
                __hip_atomic_store(words(0) + i / MINE * (D / VPW) + member * MINE + i % MINE, static_cast<unsigned long long>(kTrajGone) << 32,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

}  // namespace artab
