// Backward pass of the training row attention, one workgroup per (batch entry, head): all visible keys at once.
//
// The two kernels of attention_backward.h each compute the scores, their exponentials and dP.  Where the
// keys that anybody sees fit one workgroup, 32 to a wavefront, one walk over the queries gives all three
// gradients:
//
//   W wavefronts (a group) hold K and V of 32 keys each in registers and, per tile of 32 queries, compute
//       S[q,kv] = (scale log2e Q)[q,:] . K[kv,:]      dP[q,kv] = dO[q,:] . V[kv,:]
//       dV^T[d,kv] += dO^T[d,q] . P[q,kv]             dK^T[d,kv] += Q^T[d,q] . dS[q,kv]
//   as the dK/dV kernel does, and leave dS in LDS; behind the next tile's barrier
//       dQ^T[d,q] = sum over kv of K^T[d,kv] . dS^T[kv,q]
//   is one 16x16x32 product chain per 16 dimensions and 16 queries, dealt over the group's wavefronts: both
//   operands by transposing LDS reads (K lies there once for the whole walk).
//
// delta is made where dO goes to LDS, so that nothing but the results goes through memory; Q lies there twice, as
// it is (for dK) and scaled (for S): P is the forward's P in all three gradients.  G groups share the queries of a
// pair (tile t belongs to group t % G) and add up their dK and dV in LDS at the end, in a fixed order: a training
// step's context has one block of 128 keys, and four wavefronts walking 19 tiles one after the other were a serial
// chain of 1.7 us each.
//
// 16 wavefronts on a compute unit (8 at head_dim 64, where the accumulators take twice the registers): every wait
// of one is behind the work of three others on its SIMD.  64 entries x 4 heads of 608 rows with 96 keys: 49.5 us for the two kernels,
// 22.2 (the tensors once at the rate of a copy: 16.6); with 512 keys 156 -> 86, bound by vector instructions
// (57 % of the cycles) and LDS (40 %), the wavefronts of a barrier in step.  Measured and not kept: 64 keys to a
// wavefront with half the wavefronts (91 us where this form took 79: too few to hide each other's waits).
#pragma once

#include "attention_backward.h"
#include "fused_layer.h"

namespace artab {

template <typename T, int DH, int W, int G>
struct BackwardPair {
    static constexpr int CPR = DH / 8, PIECES = 32 * CPR, TILE = BackwardTile<T, DH>::SIZE, GT = 64 * W, THREADS = GT * G;
    // the queries' pieces go to the first threads of a group, those of dO and O to the next, where it has that many
    static constexpr bool SPLIT = GT >= 2 * PIECES;
    static constexpr int DS = BackwardTile<T, 32>::SIZE;  // elements of a wavefront's dS tile: as one of 32 columns
    static constexpr int kSum = G > 1 ? THREADS * 2 * (DH / 2) * 4 : W * 32 * (DH + 16) * 2;  // bytes of the epilogue
    static constexpr int SUB = 2 * (DH / 16);                // 16 x 16 pieces of a dQ tile
    static constexpr int SPLITS = W > SUB ? W / SUB : 1;     // wavefronts that share one, each with some of the keys
    static constexpr int kParts = SPLITS > 1 ? G * 2 * W * 1024 : 0;
    static constexpr int kStats = G * 2 * 32 * 3 * 4;
    static constexpr int kWalk = (W * TILE + G * 2 * 3 * TILE + G * 2 * W * DS) * 2 + kParts + kStats;
    static constexpr int kLds = kSum > kWalk ? kSum : kWalk;
    static_assert(kLds <= 160 * 1024, "LDS of a compute unit");
    static_assert(GT >= PIECES, "a group stages a tile in one go");
};

template <typename T, int DH, int W, int G>
__global__ __launch_bounds__(64 * W * G) void backward_pair_kernel(BackwardParams P) {
    typedef MfmaOps<T> Ops;
    typedef typename Ops::vec vec;
    typedef BackwardTile<T, DH> Tile;
    typedef BackwardPair<T, DH, W, G> Shape;
    constexpr int KS = DH / 16, DB = DH / 32, TILE = Shape::TILE, CPR = Shape::CPR, PIECES = Shape::PIECES;
    __shared__ __attribute__((aligned(16))) unsigned char lds_raw[Shape::kLds];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave_all % W, group = wave_all / W;
    const int h = blockIdx.x % P.H;
    const long b = blockIdx.x / P.H;
    const int keys = P.Nc + P.Nb, key0 = 32 * wave;

    T *const k_tiles = reinterpret_cast<T *>(lds_raw);                       // [W][TILE]
    T *const stage = k_tiles + W * TILE + group * (2 * 3 * TILE);            // [2][3: Q, scaled Q, dO][TILE]
    T *const ds_tiles = k_tiles + W * TILE + G * 2 * 3 * TILE + group * (2 * W * Shape::DS);  // [2][W][DS]
    float *const stats = reinterpret_cast<float *>(lds_raw + Shape::kWalk - Shape::kStats) + group * (2 * 3 * 32);  // [2][3][32]

    // ---- staging of the group's query tiles
    const int role = Shape::SPLIT ? 64 * wave / PIECES : 0;  // 0: Q (or all), 1: dO and O, others: nothing
    const float c2 = P.scale * kLog2e;
    const T *const q_base = view_row<T>(P.q, b, h, 0), *const g_base = view_row<T>(P.dout, b, h, 0), *const o_base = view_row<T>(P.out, b, h, 0);
    const float *const lse = P.lse + (b * P.H + h) * static_cast<long>(P.R);
    u32x4 q_raw, g_raw, o_raw;
    float st_lse;
    auto fetch = [&](int t) {
        const int piece = (64 * wave) % PIECES + opaque(lane), prow = piece / CPR, pcol = 8 * (piece % CPR);
        const long row = min(32 * t + prow, P.R - 1);
        if (!Shape::SPLIT || role == 0) q_raw = *reinterpret_cast<const u32x4 *>(q_base + row * P.q.sn + pcol);
        if (!Shape::SPLIT || role == 1) {
            g_raw = *reinterpret_cast<const u32x4 *>(g_base + row * P.dout.sn + pcol);
            o_raw = *reinterpret_cast<const u32x4 *>(o_base + row * P.out.sn + pcol);
            st_lse = lse[row];
        }
    };
    auto stash = [&](int slot, int t) {
        const int piece = (64 * wave) % PIECES + opaque(lane), prow = piece / CPR;
        T *const q_tile = stage + slot * (3 * TILE), *const s_tile = q_tile + TILE, *const g_tile = s_tile + TILE;
        if (!Shape::SPLIT || role == 0) {
            Tile::stash(q_tile, piece, q_raw);
            // scale * log2(e) folded into the queries and rounded to the input type, as the forward does (the rounding
            // model of the reference kernel, triton_kernels.py:120-121): P is the forward's P
            u32x4 sc;
#pragma unroll
            for (int e = 0; e < 4; ++e) sc[e] = pack2<T>(unpack_lo<T>(q_raw[e]) * c2, unpack_hi<T>(q_raw[e]) * c2);
            Tile::stash(s_tile, piece, sc);
        }
        if (!Shape::SPLIT || role == 1) {
            Tile::stash(g_tile, piece, g_raw);
            float delta = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                delta = fmaf(unpack_lo<T>(g_raw[e]), unpack_lo<T>(o_raw[e]), delta);
                delta = fmaf(unpack_hi<T>(g_raw[e]), unpack_hi<T>(o_raw[e]), delta);
            }
            // over the CPR lanes of a row: within fours, then the two fours of eight
            delta += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, delta), 0xB1, 0xf, 0xf, true));
            delta += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, delta), 0x4E, 0xf, 0xf, true));
            if constexpr (CPR == 8) delta += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, delta), 0x141, 0xf, 0xf, true));
            if (piece % CPR == 0) {
                float *const s = stats + slot * (3 * 32);
                s[prow] = -st_lse * kLog2e;  // negated: the accumulators start from them
                s[32 + prow] = -delta;
                reinterpret_cast<int *>(s)[64 + prow] = backward_vis_end(P, 32 * t + prow);
            }
        }
    };
    const int tiles = (P.R + 31) / 32, iters = (tiles + G - 1) / G;
    // keys that some row of tile t sees: the buffer's only from the first buffer row to the last attending target
    const int attending = keys + P.attend * P.Nb;
    auto tile_end = [&](int t) { return 32 * t + 32 <= P.Nc || 32 * t >= attending ? P.Nc : keys; };

    fetch(min(group, tiles - 1));
    vec kf[KS], vf[KS];
    {
        const int c = lane & 31, hb = lane >> 5, kj = key0 + c;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            kf[ks] = __builtin_bit_cast(vec, backward_row_piece<T>(P.k, b, h, kj, P.R, ks, hb));
            vf[ks] = __builtin_bit_cast(vec, backward_row_piece<T>(P.v, b, h, kj, P.R, ks, hb));
        }
        if (group == 0) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                *reinterpret_cast<vec *>(k_tiles + wave * TILE + (2 * ks + hb) * Tile::BLOCK + c * 8) = kf[ks];
        }
    }
    stash(0, min(group, tiles - 1));
    if (group + G < tiles) fetch(group + G);

    // (the loads of K and V end here: the compiler would otherwise wait, at their first use in every iteration, for all
    // that is on its way, the next tile among it)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(kf[ks]), "+v"(vf[ks]));
    f32x16 acc_k[DB], acc_v[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc_k[db][v] = acc_v[db][v] = 0.f;

    // dQ of tile t from the dS of a slot.  A wavefront has a 16 x 16 piece (or two of them); where there are more
    // wavefronts than pieces, those of a piece deal the blocks of keys among themselves and leave their sums in
    // LDS, where one of them adds them up behind the next barrier.
    constexpr int SUB = Shape::SUB, SPLITS = Shape::SPLITS, PER = SUB > W ? SUB / W : 1;
    f32x4 *const parts = reinterpret_cast<f32x4 *>(lds_raw + Shape::kWalk - Shape::kStats - Shape::kParts) + group * (2 * W * 64);  // [2][W][64]
    auto dq_store = [&](int t, int sub, const f32x4 &dq, int ln) {
        const int row = 32 * t + 16 * (sub & 1) + (ln & 15);
        if (row < P.R)
            store4f<T>(view_row<T>(P.dq, b, h, row) + 16 * (sub >> 1) + 4 * (ln >> 4), dq[0] * P.scale, dq[1] * P.scale, dq[2] * P.scale,
                       dq[3] * P.scale);
    };
    auto dq_tile = [&](int t, int slot) {
        const int steps = (tile_end(t) + 31) / 32, ln = opaque(lane);
        const int in = ((ln >> 1) & 1) * Tile::BLOCK + (8 * (ln >> 4) + ((ln & 15) >> 2)) * 8 + 4 * (ln & 1);  // (rows 8 quad + l15 / 4 and + 4 of a step's 32 keys)
        const T *const ds = ds_tiles + slot * (W * Shape::DS);
        auto operand = [](const T *p) {
            s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(p));
            s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(p + 4 * 8));
            typedef short s16x8 __attribute__((ext_vector_type(8)));
            s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            return __builtin_bit_cast(vec, both);
        };
#pragma unroll
        for (int x = 0; x < PER; ++x) {
            const int sub = (wave + W * x) % SUB, split = wave / SUB;
            const T *const k_at = k_tiles + (sub >> 1) * (2 * Tile::BLOCK) + in, *const d_at = ds + (sub & 1) * (2 * Tile::BLOCK) + in;
            f32x4 dq = {0.f, 0.f, 0.f, 0.f};
            if (steps == W) {
                constexpr int N = W / SPLITS;
                vec kt[N], dt[N];  // (all on their way before the first is multiplied; the compiler would take turns)
#pragma unroll
                for (int s = 0; s < N; ++s) {
                    kt[s] = operand(k_at + (s * SPLITS + split) * TILE);
                    dt[s] = operand(d_at + (s * SPLITS + split) * Shape::DS);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < N; ++s) dq = Ops::mma16(kt[s], dt[s], dq);
            } else {
                for (int s = split; s < steps; s += SPLITS) dq = Ops::mma16(operand(k_at + s * TILE), operand(d_at + s * Shape::DS), dq);
            }
            if constexpr (SPLITS > 1)
                parts[(slot * W + wave) * 64 + ln] = dq;
            else
                dq_store(t, sub, dq, ln);
        }
    };
    auto dq_sum = [&](int t, int slot) {
        if (t < 0 || wave / SUB != t / G % SPLITS) return;
        const int ln = opaque(lane), sub = wave % SUB;
        const f32x4 *const p = parts + (slot * W + sub) * 64 + ln;
        f32x4 dq = p[0];
#pragma unroll
        for (int i = 1; i < SPLITS; ++i) dq += p[i * SUB * 64];
        dq_store(t, sub, dq, ln);
    };
    // rows of target keys, which nobody sees: zeros, a piece per thread and iteration
    const int zeros = (P.R - keys) * CPR;
    int zero_at = tid;
    auto zero_piece = [&]() {
        if (zero_at >= zeros) return;
        const u32x4 zero = {0u, 0u, 0u, 0u};
        const int row = keys + zero_at / CPR, col = 8 * (zero_at % CPR);
        *reinterpret_cast<u32x4 *>(view_row<T>(P.dk, b, h, row) + col) = zero;
        *reinterpret_cast<u32x4 *>(view_row<T>(P.dv, b, h, row) + col) = zero;
        zero_at += Shape::THREADS;
    };

    for (int it = 0; it < iters; ++it) {
        __syncthreads();  // tile `it` and the last one's dS are complete; everyone has finished reading what is overwritten now
        const int t = it * G + group, slot = it & 1;
        if (t + G < tiles) stash(slot ^ 1, t + G);
        if constexpr (SPLITS > 1) dq_sum(t - 2 * G, slot);
        if (it > 0) dq_tile(t - G, slot ^ 1);  // (every tile but a group's last is followed by an iteration of all groups)
        zero_piece();
        if (t + 2 * G < tiles) fetch(t + 2 * G);
        if (t >= tiles || key0 >= tile_end(t)) continue;
        const T *const q_tile = stage + slot * (3 * TILE), *const s_tile = q_tile + TILE, *const g_tile = s_tile + TILE;
        const float *const st = stats + slot * (3 * 32);
        const int ln = opaque(lane), c = ln & 31, hb = ln >> 5;  // (addresses made of it are not kept over the iterations)
        // rows of the accumulators are queries 8g + 4hb + r of the tile: the accumulators start at
        // -lse2 and -delta of their rows, so that the products leave log2 P and dP - delta
        f32x16 s, dp;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 l4 = *reinterpret_cast<const f32x4 *>(st + 8 * g + 4 * hb);
            const f32x4 d4 = *reinterpret_cast<const f32x4 *>(st + 32 + 8 * g + 4 * hb);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[4 * g + r] = l4[r];
                dp[4 * g + r] = d4[r];
            }
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            s = Ops::mma(Tile::row_operand(s_tile, c, hb, ks), kf[ks], s);
            dp = Ops::mma(Tile::row_operand(g_tile, c, hb, ks), vf[ks], dp);
        }
        u32x4 pb[2], dsb[2];
        // context keys under a full tile of rows: everything is visible (a branch of the whole wavefront)
        if (key0 + 32 <= P.Nc && 32 * t + 32 <= P.R) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float p[4], ds[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    p[r] = fast_exp2(s[4 * g + r]);
                    ds[r] = p[r] * dp[4 * g + r];
                }
                const int x = g >> 1, e = 2 * (g & 1);
                pb[x][e] = pack2<T>(p[0], p[1]);
                pb[x][e + 1] = pack2<T>(p[2], p[3]);
                dsb[x][e] = pack2<T>(ds[0], ds[1]);
                dsb[x][e + 1] = pack2<T>(ds[2], ds[3]);
            }
        } else {
            const int *const end_s = reinterpret_cast<const int *>(st) + 64;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int4 e4 = *reinterpret_cast<const int4 *>(end_s + 8 * g + 4 * hb);
                const int ends[4] = {e4.x, e4.y, e4.z, e4.w};
                float p[4], ds[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool vis = key0 + c < ends[r];
                    const float pr = fast_exp2(s[4 * g + r]);
                    p[r] = vis ? pr : 0.f;
                    ds[r] = vis ? pr * dp[4 * g + r] : 0.f;
                }
                const int x = g >> 1, e = 2 * (g & 1);
                pb[x][e] = pack2<T>(p[0], p[1]);
                pb[x][e + 1] = pack2<T>(p[2], p[3]);
                dsb[x][e] = pack2<T>(ds[0], ds[1]);
                dsb[x][e + 1] = pack2<T>(ds[2], ds[3]);
            }
        }
        vec gt[DB][2], qt[DB][2];  // (all on their way before the first is multiplied; the compiler would take turns)
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                gt[db][x] = Tile::col_operand(g_tile, ln, x, db);
                qt[db][x] = Tile::col_operand(q_tile, ln, x, db);
            }
        // dS as [kv][q] in blocks of 8 queries, as the tiles: the lane's key is a row, four queries a piece
        T *const ds = ds_tiles + (slot * W + wave) * Shape::DS;
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<u32x2 *>(ds + g * Tile::BLOCK + c * 8 + 4 * hb) = u32x2{dsb[g >> 1][2 * (g & 1)], dsb[g >> 1][2 * (g & 1) + 1]};
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                acc_v[db] = Ops::mma(gt[db][x], __builtin_bit_cast(vec, pb[x]), acc_v[db]);
                acc_k[db] = Ops::mma(qt[db][x], __builtin_bit_cast(vec, dsb[x]), acc_k[db]);
            }
    }
    __syncthreads();
    {
        const int t = (iters - 1) * G + group;
        if constexpr (SPLITS > 1) dq_sum(t - G, iters & 1);
        if (t < tiles) dq_tile(t, (iters - 1) & 1);
        if constexpr (SPLITS > 1) {
            __syncthreads();
            if (t < tiles) dq_sum(t, (iters - 1) & 1);
        }
    }
    while (zero_at < zeros) zero_piece();

    __syncthreads();  // LDS is free
    if constexpr (G == 1) {
        T *const out = reinterpret_cast<T *>(lds_raw) + wave * (32 * Tile::PAD);
        if (key0 < keys) {
            backward_store_rows<T, DH>(out, acc_k, P.scale, P.dk, b, h, key0, keys, lane);
            backward_store_rows<T, DH>(out, acc_v, 1.f, P.dv, b, h, key0, keys, lane);
        }
    } else {
        constexpr int REGS = 16 * DB, MINE = REGS / G;
        static_assert(MINE % 4 == 0, "whole pieces of four dimensions");
        float *const sum = reinterpret_cast<float *>(lds_raw);  // [W][2][REGS][G][64]
        if (key0 < keys) {
#pragma unroll
            for (int r = 0; r < REGS; ++r) {
                sum[(((wave * 2 + 0) * REGS + r) * G + group) * 64 + lane] = acc_k[r / 16][r % 16];
                sum[(((wave * 2 + 1) * REGS + r) * G + group) * 64 + lane] = acc_v[r / 16][r % 16];
            }
        }
        __syncthreads();
        const int hb = lane >> 5, kj = key0 + (lane & 31);
        if (kj < keys) {
#pragma unroll
            for (int which = 0; which < 2; ++which)
#pragma unroll
                for (int x = 0; x < MINE; x += 4) {
                    const int r0 = group * MINE + x;
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float *const p = sum + ((wave * 2 + which) * REGS + r0 + e) * G * 64 + lane;
                        v[e] = p[0];
#pragma unroll
                        for (int g = 1; g < G; ++g) v[e] += p[g * 64];
                        if (which == 0) v[e] *= P.scale;
                    }
                    const int d = 32 * (r0 / 16) + 8 * ((r0 % 16) >> 2) + 4 * hb;
                    store4f<T>(view_row<T>(which == 0 ? P.dk : P.dv, b, h, kj) + d, v[0], v[1], v[2], v[3]);
                }
        }
    }
}

}  // namespace artab
