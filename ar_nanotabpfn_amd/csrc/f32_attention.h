// float32 attention on the matrix cores (gfx950, v_mfma_f32_16x16x4_f32), head_dim 32/64/128.
//
// Everything the float32 entry points ask for in one kernel, with the arguments of the portable
// kernel (PortableParams): context, decode (shared context with a buffer per trajectory, or a context
// of its own for each), teacher forcing, prefill, row mask.  Float32 products run at 256 FLOP per
// clock and compute unit (157 TFLOP/s), a sixteenth of the 16-bit rate, so the matrix cores are the
// bound and nothing else may get in their way; the portable kernel, one wavefront per query row,
// re-reads the keys for every row and reached 2 % of that rate.  Measured against it: self-attention of
// 64 x 512 rows, 8 heads of 32: 9587 -> 184 us (93 TFLOP/s; heads of 64: 10438 -> 333 us, 103 TFLOP/s);
// 1024 stacked queries on a context of 16384: 9530 -> 188 us; one query on 512 rows: 82 -> 11 us.
//
// Layout: transposed as in mfma_flash.h, S^T = K Q^T and O^T = V^T P^T, so that a query is a column
// (lane & 15) and the softmax statistics are per-lane values.  With the 16x16x4 form lane (c, g = lane
// / 16) gives contraction element g of row (or column) c:
//   * S^T step 4t + e contracts the dims {16 t + 4 g + e}: K and Q fragments are 16-byte pieces of rows;
//   * the scores of lane (c, g) are the keys {4 g + r}: used as they are as the B operand of step r;
//   * the rows of O^T may be dims in any order: row m of block n is dim (DH/16) m + n, so that a lane
//     reads DH/16 neighbouring floats of a V row and ends up with DH/4 neighbouring floats of the output.
// No operand passes through LDS: a block of 32 keys feeds 2 * 16 QB * DH / 32 products of 32 clocks
// from 256 DH bytes, 4 bytes per clock and SIMD at QB = 2, within what the L1 and L2 deliver.  K of the
// next block is requested behind the first product of this one, V behind the second: each has most
// of a block's time to arrive.
//
// Keys come in 32-row blocks ("tasks") of three kinds: the context, the buffers (of the tile's own
// batch entry, or of each trajectory in turn where the context is shared and the tile stacks
// trajectories: visible to that trajectory's columns only), and the new rows (one per trajectory: a
// block whose rows are trajectories).  SPLIT deals a tile's tasks over the wavefronts of a workgroup
// (and over workgroups, P2.n_split) and merges the partial results in LDS (in a launch of its own);
// otherwise every wavefront has its own tile.
#pragma once

#include <type_traits>

#include "common.h"
#include "portable_kernels.h"

namespace artab {

struct F32Plan {
    int stacked;          // 1: one group per head, rows of all batch entries in one run
    int G, n_groups;      // rows per group; groups per head (1 or B)
    int tiles;            // tiles per group
    int n_split;          // workgroups per tile (SPLIT only)
    float *part_o, *part_lse;  // n_split > 1: [n_split][rows][DH] normalised, [n_split][rows] base-2
    long rows;            // B * H * Lq
};

// HIDES: there are keys that some column may not see (buffers, new rows); without them there is one pass and no watch.
template <int DH, int QB, bool SPLIT, int NW, bool HIDES>
__global__ __launch_bounds__(NW * 64) void f32_attention_kernel(PortableParams P, F32Plan L) {
    constexpr int KT = DH / 16;   // 16-byte pieces per lane and K row; output blocks
    constexpr int COLS = 16 * QB;
    typedef float fvec __attribute__((ext_vector_type(KT < 4 ? KT : 4)));
    constexpr int VN = KT < 4 ? 1 : KT / 4;  // vector loads per V row and lane
    typedef const char __attribute__((address_space(1))) *gptr;  // (scalar base, 32-bit byte offset per lane)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c = lane & 15, g = lane >> 4;

    // workgroup -> (group and head, tile, slice); all tiles of a (group, head) on one XCD
    const int xcd = blockIdx.x & 7;
    int rest = blockIdx.x >> 3;
    const int wg_tiles = SPLIT ? L.tiles : (L.tiles + NW - 1) / NW;
    int slice = 0;
    if (SPLIT) {
        slice = rest % L.n_split;
        rest /= L.n_split;
    }
    int tile = rest % wg_tiles;
    const int kvg = rest / wg_tiles * 8 + xcd;
    if (kvg >= P.H * L.n_groups) return;
    if (!SPLIT) tile = tile * NW + wave;
    const int h = kvg % P.H, grp = kvg / P.H;
    const int row0 = tile * COLS;  // first row of the tile in its group
    if (!SPLIT && row0 >= L.G) return;  // (no barrier below in this form)
    const int live = min(COLS, L.G - row0);
    // batch entry and query index of a row of the group
    auto place = [&](int r, int &b, int &i) {
        const int flat = row0 + min(r, live - 1);
        if (L.stacked) {
            b = flat / P.Lq;
            i = flat - b * P.Lq;
        } else {
            b = grp;
            i = flat;
        }
    };

    if (P.nbuf_dev) {
        // a length read from device memory is clamped to the cache; a new row that would land
        // behind the last slot is attended but not stored
        const int hi = P.capacity - (P.new_row >= 0 ? 1 : 0);
        const int raw = *P.nbuf_dev;
        const int n = raw < 0 ? 0 : (raw > hi ? (hi > 0 ? hi : 0) : raw);
        if (raw != n) P.append = 0;
        P.Nb = n + (P.new_row >= 0 ? 1 : 0);
        if (P.new_row >= 0) P.new_row = n;
    }
    const bool has_new = P.new_row >= 0;
    const int n_buf = P.Nb - (has_new ? 1 : 0);  // rows stored before this call

    const int b_first = L.stacked ? row0 / P.Lq : grp;
    const int n_traj = L.stacked ? (row0 + live - 1) / P.Lq - b_first + 1 : 1;

    // per column: its batch entry within the tile, and the buffer keys it sees
    int traj[QB], limit[QB];
    float q[QB][DH / 4];
#pragma unroll
    for (int j = 0; j < QB; ++j) {
        int b, i;
        place(16 * j + c, b, i);
        traj[j] = b - b_first;
        limit[j] = n_buf;
        if (P.mode == kModeTeacher) limit[j] = min(n_buf, tf_limit(i, P.Nt));
        if (P.mode == kModeRowMask) limit[j] = min(n_buf, row_mask_limit(i, P.rm_nc, n_buf, P.rm_attend));
        const float *row = view_row<float>(P.q, b, h, i) + 4 * g;
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            const f32x4 v = *reinterpret_cast<const f32x4 *>(row + 16 * t);
#pragma unroll
            for (int e = 0; e < 4; ++e) q[j][4 * t + e] = v[e] * P.scale;
        }
    }
    int buf_max = 0;  // buffer keys that any column of the tile sees
#pragma unroll
    for (int j = 0; j < QB; ++j) buf_max = max(buf_max, limit[j]);
    if (P.mode != kModePlain) {
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) buf_max = max(buf_max, __shfl_xor(buf_max, o, 64));
    }
    buf_max = __builtin_amdgcn_readfirstlane(buf_max);

    const int n_ctx_t = (P.Nc + 31) / 32, per_traj = (buf_max + 31) / 32;
    const int n_buf_t = n_traj * per_traj, n_new_t = has_new ? (n_traj + 31) / 32 : 0;
    const int n_tasks = n_ctx_t + n_buf_t + n_new_t;
    int t_first, t_end, t_step;
    if (SPLIT) {
        t_first = static_cast<int>(static_cast<long>(n_tasks) * slice / L.n_split) + wave;
        t_end = static_cast<int>(static_cast<long>(n_tasks) * (slice + 1) / L.n_split);
        t_step = NW;
    } else {
        t_first = 0;
        t_end = n_tasks;
        t_step = 1;
    }

    // a block of keys: where its rows are, and which of them each column sees
    struct Block {
        gptr k, v;
        unsigned k_sn, v_sn, last;  // row strides in bytes; last valid row, counted from the segment's first
        int key0;
        int kind, traj;  // kind 0: context, 1: buffer, 2: new rows
    };
    auto block_of = [&](int t) {
        Block B;
        if (t < n_ctx_t || t >= n_tasks) {
            const int b = L.stacked ? b_first : grp;
            B = {(gptr)view_row<float>(P.kc, b, h, 0), (gptr)view_row<float>(P.vc, b, h, 0), static_cast<unsigned>(4 * P.kc.sn),
                 static_cast<unsigned>(4 * P.vc.sn), static_cast<unsigned>(P.Nc - 1), 32 * min(t, max(n_ctx_t - 1, 0)), 0, 0};
        } else if (t < n_ctx_t + n_buf_t) {
            const int u = t - n_ctx_t, tr = L.stacked ? u / per_traj : 0;
            B = {(gptr)view_row<float>(P.kb, b_first + tr, h, 0), (gptr)view_row<float>(P.vb, b_first + tr, h, 0),
                 static_cast<unsigned>(4 * P.kb.sn), static_cast<unsigned>(4 * P.vb.sn), static_cast<unsigned>(n_buf - 1),
                 32 * (u - tr * per_traj), 1, tr};
        } else {
            B = {(gptr)view_row<float>(P.knew, b_first, h, 0), (gptr)view_row<float>(P.vnew, b_first, h, 0),
                 static_cast<unsigned>(4 * P.knew.sb), static_cast<unsigned>(4 * P.vnew.sb), static_cast<unsigned>(n_traj - 1),
                 32 * (t - n_ctx_t - n_buf_t), 2, 0};
        }
        return B;
    };
    f32x4 kf[2][KT];
    fvec vf[2][4][VN];
    auto request_k = [&](const Block &B) {
#pragma unroll
        for (int sb = 0; sb < 2; ++sb) {
            const unsigned row = min((B.key0 + 16 * sb + c) * B.k_sn, B.last * B.k_sn) + 16 * g;
#pragma unroll
            for (int t = 0; t < KT; ++t)
                kf[sb][t] = *reinterpret_cast<const f32x4 __attribute__((address_space(1))) *>(B.k + (row + 64 * t));
        }
    };
    auto load_v = [&](const Block &B, int key, fvec (&v)[VN]) {  // this lane's piece of a value row
        const unsigned row = min(key * B.v_sn, B.last * B.v_sn) + 4 * KT * c;
#pragma unroll
        for (int n = 0; n < VN; ++n) v[n] = *reinterpret_cast<const fvec __attribute__((address_space(1))) *>(B.v + (row + 16 * n));
    };
    auto request_v = [&](const Block &B) {
#pragma unroll
        for (int sb = 0; sb < 2; ++sb)
#pragma unroll
            for (int r = 0; r < 4; ++r) load_v(B, B.key0 + 16 * sb + 4 * g + r, vf[sb][r]);
    };

    // The wavefront's tasks.  A key that is hidden from a column has probability 0 there, and 0 times a value that
    // is not finite is NaN: the pass that multiplies every value of a block by every column watches for
    // such values in blocks that are hidden from somebody (the context is hidden from nobody; its last
    // block repeats a row that everybody sees) and, if there were any, is followed by a second one,
    // CAREFUL: column after column, with zeros for the values that the column does not see, and with
    // nothing requested ahead, so that it needs no registers that the common pass does not.
    f32x4 o[QB][KT];
    float m[QB], l[QB];
    // (here and below: set inside the lambda, they cost the common kernels up to 30 registers)
#pragma unroll
    for (int j = 0; j < QB; ++j) {
        m[j] = -INFINITY;
        l[j] = 0.f;
#pragma unroll
        for (int n = 0; n < KT; ++n) o[j][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    auto pass = [&](auto careful) {
        constexpr bool CAREFUL = decltype(careful)::value;
        float watch = 0.f;  // NaN: values that are not finite
        int t_now = t_first;
        if (t_now >= t_end) return false;
        Block cur = block_of(t_now);
        if (!CAREFUL) {
            request_k(cur);
            request_v(cur);
        }
        for (; t_now < t_end; t_now += t_step) {
            if (CAREFUL) request_k(cur);
            const int t_next = t_now + t_step < t_end ? t_now + t_step : t_now;
            const Block next = block_of(t_next);
            // (a trajectory's columns are within one block of 16: other blocks sit its buffer out)
            const bool one = L.stacked && cur.kind == 1;
            const int only = one ? (cur.traj * P.Lq) >> 4 : 0;
            f32x4 s[QB][2];
#pragma unroll
            for (int j = 0; j < QB; ++j) {
#pragma unroll
                for (int sb = 0; sb < 2; ++sb) s[j][sb] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (one && only != j) continue;
#pragma unroll
                for (int sb = 0; sb < 2; ++sb)
#pragma unroll
                    for (int t = 0; t < KT; ++t)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            s[j][sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[sb][t][e], q[j][4 * t + e], s[j][sb], 0, 0, 0);
            }
            if (!CAREFUL) request_k(next);
#pragma unroll
            for (int j = 0; j < QB; ++j) {
                if (one && only != j) continue;
                int lo = 0, hi;  // the segment's rows that this column sees
                if (cur.kind == 0) {
                    hi = P.Nc;
                } else if (cur.kind == 1) {
                    hi = !L.stacked || traj[j] == cur.traj ? limit[j] : 0;
                } else {
                    lo = traj[j];
                    hi = traj[j] + 1;
                }
                const bool hidden = __any(hi < cur.key0 + 32 || lo > cur.key0);
                if (hidden) {
#pragma unroll
                    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int key = cur.key0 + 16 * sb + 4 * g + r;
                            if (key < lo || key >= hi) s[j][sb][r] = -INFINITY;
                        }
                }
                float mx = s[j][0][0];  // (no inline assembly on the products' results: the compiler spaces their readers)
#pragma unroll
                for (int x = 1; x < 8; ++x) mx = fmaxf(mx, s[j][x >> 2][x & 3]);
                mx = row_max(mx);
                const float m_new = fmaxf(m[j], mx);
                if (__any(m_new > m[j])) {
                    const float alpha = m[j] == -INFINITY ? 0.f : fast_exp2(m[j] - m_new);
                    m[j] = m_new;
                    l[j] *= alpha;
#pragma unroll
                    for (int n = 0; n < KT; ++n) o[j][n] *= alpha;
                }
                const float m_use = m_new == -INFINITY ? 0.f : m_new;  // a column that has seen no key yet
#pragma unroll
                for (int sb = 0; sb < 2; ++sb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        s[j][sb][r] = fast_exp2(s[j][sb][r] - m_use);
                        l[j] += s[j][sb][r];
                    }
                const bool masked = HIDES && hidden && cur.kind != 0;
                auto value = [&](const fvec (&v)[VN], int n) {
                    if constexpr (KT < 4) return v[0][n];
                    else return v[n / 4][n % 4];
                };
                if constexpr (CAREFUL) {
                    const int n_cols = masked ? 16 : 1;
#pragma unroll 1
                    for (int col = 0; col < n_cols; ++col) {
                        const int lo_c = masked ? __builtin_amdgcn_readlane(lo, col) : 0;
                        const int hi_c = masked ? __builtin_amdgcn_readlane(hi, col) : 0x7fffffff;
                        f32x4 sum[KT];
#pragma unroll
                        for (int n = 0; n < KT; ++n) sum[n] = o[j][n];
#pragma unroll
                        for (int x = 0; x < 8; ++x) {
                            __builtin_amdgcn_sched_barrier(0);
                            const int key = cur.key0 + 16 * (x >> 2) + 4 * g + (x & 3);
                            fvec v[VN];
                            load_v(cur, key, v);
#pragma unroll
                            for (int n = 0; n < KT; ++n)
                                sum[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(key >= lo_c && key < hi_c ? value(v, n) : 0.f,
                                                                              s[j][x >> 2][x & 3], sum[n], 0, 0, 0);
                        }
#pragma unroll
                        for (int n = 0; n < KT; ++n)
#pragma unroll
                            for (int e = 0; e < 4; ++e) o[j][n][e] = !masked || c == col ? sum[n][e] : o[j][n][e];
                    }
                } else {
                    if (masked) {
#pragma unroll
                        for (int x = 0; x < 8; ++x)
#pragma unroll
                            for (int n = 0; n < KT; ++n) watch = fmaf(value(vf[x >> 2][x & 3], n), 0.f, watch);
                    }
#pragma unroll
                    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
#pragma unroll
                            for (int n = 0; n < KT; ++n)
                                o[j][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(value(vf[sb][r], n), s[j][sb][r], o[j][n], 0, 0, 0);
                }
            }
            if (!CAREFUL) request_v(next);
            cur = next;
        }
        return __any(watch != 0.f) != 0;
    };
    const bool again = pass(std::false_type{});
    if constexpr (HIDES) {
        if (again) {
#pragma unroll
            for (int j = 0; j < QB; ++j) {
                m[j] = -INFINITY;
                l[j] = 0.f;
#pragma unroll
                for (int n = 0; n < KT; ++n) o[j][n] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            pass(std::true_type{});
        }
    }
#pragma unroll
    for (int j = 0; j < QB; ++j) l[j] = row_sum(l[j]);

    // ---- results: lane (c, g) holds dims [DH/4 g, DH/4 (g + 1)) of column c, element 4 n' .. of block n
    // being dim KT (4 g + r) + n
    auto out_value = [&](int j, int d) { return o[j][d % KT][d / KT]; };  // d within the lane's DH/4
    if constexpr (SPLIT) {
        __shared__ __attribute__((aligned(16))) float po[NW][COLS][DH + 4];
        __shared__ float pm[NW][COLS], pl[NW][COLS];
#pragma unroll
        for (int j = 0; j < QB; ++j) {
            if (g == 0) {
                pm[wave][16 * j + c] = m[j];
                pl[wave][16 * j + c] = l[j];
            }
#pragma unroll
            for (int x = 0; x < DH / 16; ++x) {
                const f32x4 v = {out_value(j, 4 * x), out_value(j, 4 * x + 1), out_value(j, 4 * x + 2), out_value(j, 4 * x + 3)};
                *reinterpret_cast<f32x4 *>(&po[wave][16 * j + c][DH / 4 * g + 4 * x]) = v;
            }
        }
        __syncthreads();
        for (int idx = threadIdx.x; idx < live * (DH / 4); idx += NW * 64) {
            const int col = idx / (DH / 4), d0 = idx % (DH / 4) * 4;
            float mx = -INFINITY;
#pragma unroll
            for (int w = 0; w < NW; ++w) mx = fmaxf(mx, pm[w][col]);
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            float sum = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const float wt = pm[w][col] == -INFINITY ? 0.f : fast_exp2(pm[w][col] - mx);
                sum += wt * pl[w][col];
                acc += wt * *reinterpret_cast<const f32x4 *>(&po[w][col][d0]);
            }
            const float inv = sum > 0.f ? 1.f / sum : 0.f;  // no visible key: out = 0, lse = -inf
            acc *= inv;
            int b, i;
            place(col, b, i);
            const float lse2 = sum > 0.f ? mx + fast_log2(sum) : -INFINITY;
            const long row = (static_cast<long>(b) * P.H + h) * P.Lq + i;
            if (L.n_split > 1) {
                *reinterpret_cast<f32x4 *>(L.part_o + (slice * L.rows + row) * DH + d0) = acc;
                if (d0 == 0) L.part_lse[slice * L.rows + row] = lse2;
            } else {
                *reinterpret_cast<f32x4 *>(view_row<float>(P.out, b, h, i) + d0) = acc;
                if (P.lse && d0 == 0) P.lse[row] = lse2 * kLn2;
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < QB; ++j) {
            if (16 * j + c >= live) continue;
            const float inv = l[j] > 0.f ? 1.f / l[j] : 0.f;
            f32x4 v[DH / 16];
#pragma unroll
            for (int x = 0; x < DH / 16; ++x)
                v[x] = f32x4{out_value(j, 4 * x), out_value(j, 4 * x + 1), out_value(j, 4 * x + 2), out_value(j, 4 * x + 3)} * inv;
            int b, i;
            place(16 * j + c, b, i);
            const float lse2 = l[j] > 0.f ? m[j] + fast_log2(l[j]) : -INFINITY;
            const long row = (static_cast<long>(b) * P.H + h) * P.Lq + i;
            float *dst = view_row<float>(P.out, b, h, i) + DH / 4 * g;
#pragma unroll
            for (int x = 0; x < DH / 16; ++x) *reinterpret_cast<f32x4 *>(dst + 4 * x) = v[x];
            if (P.lse && g == 0) P.lse[row] = lse2 * kLn2;
        }
    }

    // ---- rows that the call stores: new buffer rows (by the first slice; nobody reads them here), and
    // the prefill's cache rows (row i of K and V by the tile of query i)
    const int first = SPLIT ? threadIdx.x : lane, count = SPLIT ? NW * 64 : 64;
    if (P.append && slice == 0) {
        for (int idx = first; idx < n_traj * (DH / 4); idx += count) {
            const int b = b_first + idx / (DH / 4), d = idx % (DH / 4) * 4;
            // (a trajectory whose queries lie in two tiles is stored by the first of them)
            if (L.stacked ? b * P.Lq < row0 : row0 > 0) continue;
            *reinterpret_cast<f32x4 *>(view_row<float>(P.kb, b, h, P.new_row) + d) =
                *reinterpret_cast<const f32x4 *>(view_row<float>(P.knew, b, h, 0) + d);
            *reinterpret_cast<f32x4 *>(view_row<float>(P.vb, b, h, P.new_row) + d) =
                *reinterpret_cast<const f32x4 *>(view_row<float>(P.vnew, b, h, 0) + d);
        }
    }
    if (P.kcache.p && slice == 0) {
        for (int idx = first; idx < live * (DH / 4); idx += count) {
            const int d = idx % (DH / 4) * 4;
            int b, i;
            place(idx / (DH / 4), b, i);
            if (b >= P.cache_batches) continue;
            *reinterpret_cast<f32x4 *>(view_row<float>(P.kcache, b, h, i) + d) =
                *reinterpret_cast<const f32x4 *>(view_row<float>(P.kc, b, h, i) + d);
            *reinterpret_cast<f32x4 *>(view_row<float>(P.vcache, b, h, i) + d) =
                *reinterpret_cast<const f32x4 *>(view_row<float>(P.vc, b, h, i) + d);
        }
    }
}

// Slices of a tile, merged.
template <int DH>
__global__ __launch_bounds__(256) void f32_combine_kernel(PortableParams P, F32Plan L) {
    const long idx = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    const long row = idx / (DH / 4);
    if (row >= L.rows) return;
    const int d0 = static_cast<int>(idx % (DH / 4)) * 4;
    float mx = -INFINITY;
    for (int s = 0; s < L.n_split; ++s) mx = fmaxf(mx, L.part_lse[s * L.rows + row]);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float sum = 0.f;
    for (int s = 0; s < L.n_split; ++s) {
        const float lse = L.part_lse[s * L.rows + row];
        const float wt = lse == -INFINITY ? 0.f : fast_exp2(lse - mx);
        sum += wt;
        acc += wt * *reinterpret_cast<const f32x4 *>(L.part_o + (s * L.rows + row) * DH + d0);
    }
    const int i = static_cast<int>(row % P.Lq), h = static_cast<int>(row / P.Lq % P.H);
    const long b = row / (static_cast<long>(P.Lq) * P.H);
    *reinterpret_cast<f32x4 *>(view_row<float>(P.out, b, h, i) + d0) = acc * (sum > 0.f ? 1.f / sum : 0.f);
    if (P.lse && d0 == 0) P.lse[row] = sum > 0.f ? (mx + fast_log2(sum)) * kLn2 : -INFINITY;
}

}  // namespace artab
