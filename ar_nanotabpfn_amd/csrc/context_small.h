// Context attention in one launch for calls with few query rows (gfx950; bf16/f16; head_dim 32/64): the queries of
// a group against a context of up to a few thousand rows, output and log-sum-exp.
//
// Bound: latency.  mfma_flash.h gives a group's 64 rows two wavefronts that walk the whole context between them,
// a barrier per 64 keys.  Here a workgroup takes 32 query rows, one column tile of S^T = K Q^T, O^T = V^T P^T, and
// its eight wavefronts deal the 32-key blocks among themselves, no barrier between them: K operands straight from
// memory, V through a wavefront-private tile for the transposing read, two blocks requested ahead, an online
// softmax of its own each; float32 partials are merged in LDS.  (Phase 1 of decode_small.h does the same for
// eight trajectories.)  Every workgroup reads its whole context from the L2, which limits where it is used
// (context_small_applies).
#pragma once

#include "common.h"
#include "mfma_flash.h"

namespace artab {

constexpr int kContextSmallWaves = 8, kContextSmallRows = 32;

struct ContextSmallParams {
    View q, kc, vc, out;
    float *lse;      // [B, H, Lq] or null
    int H, Lq, Nc;
    int G;           // query rows of a group: B * Lq against one context, else Lq
    int tiles;       // of 32 rows, per group
    int stacked;
    float qscale;
    // prefill (queries are the rows of the keys): the tile's K and V rows go to the caches of the first groups
    View kcache, vcache;
    int cache_batches;
};

template <typename T, int DH>
__global__ __launch_bounds__(kContextSmallWaves * 64) void context_small_kernel(ContextSmallParams P) {
    typedef MfmaOps<T> Ops;
    typedef typename Ops::vec vec;
    constexpr int KS = DH / 16, DB = DH / 32, NW = kContextSmallWaves, NCOL = kContextSmallRows;
    constexpr int VPAD = DH + 16;      // row stride = 32 or 96 bytes mod 128 for the transposing reads
    constexpr int CPR = DH / 8;        // 16-byte pieces per row
    constexpr int VP = 32 * CPR / 64;  // V pieces per lane and block
    constexpr int V_BYTES = NW * 32 * VPAD * sizeof(T), O_BYTES = NW * NCOL * DH * 4;
    // the V tiles, and when all wavefronts have left them the partial outputs
    __shared__ __attribute__((aligned(16))) char lds[V_BYTES > O_BYTES ? V_BYTES : O_BYTES];
    __shared__ float part_lse2[NW][NCOL];

    const int h = blockIdx.x % P.H, t = blockIdx.x / P.H, group = t / P.tiles, row0 = (t % P.tiles) * NCOL;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c = lane & 31, hb = lane >> 5;
    const T *const kc_h = view_row<T>(P.kc, group, h, 0), *const vc_h = view_row<T>(P.vc, group, h, 0);
    const auto batch = [&](int r) { return static_cast<long>(P.stacked ? r / P.Lq : group); };
    const auto query = [&](int r) { return P.stacked ? r % P.Lq : r; };

    const int n_blocks = (P.Nc + 31) / 32;
    struct Raw {  // operands of a block: K in MFMA order (row c, 8 elements at 16 ks + 8 hb), V as pieces lane + 64 x
        u32x4 k[KS];
        u32x4 v[VP];
    };
    // rows past the end re-read the last one: their scores are masked, only finite values are needed
    auto fetch = [&](int blk, Raw &r) {
        const T *kr = kc_h + static_cast<long>(min(32 * blk + c, P.Nc - 1)) * P.kc.sn + 8 * hb;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) r.k[ks] = *reinterpret_cast<const u32x4 *>(kr + 16 * ks);
#pragma unroll
        for (int x = 0; x < VP; ++x) {
            const int idx = lane + 64 * x;
            r.v[x] = *reinterpret_cast<const u32x4 *>(vc_h + static_cast<long>(min(32 * blk + idx / CPR, P.Nc - 1)) * P.vc.sn +
                                                      8 * (idx % CPR));
        }
    };
    Raw r0, r1, r2;
    if (wave < n_blocks) fetch(wave, r0);
    if (wave + NW < n_blocks) fetch(wave + NW, r1);

    if (group < P.cache_batches) {
        const int idx = threadIdx.x / CPR, piece = 8 * (threadIdx.x % CPR);
        for (int r = row0 + idx; r < min(row0 + NCOL, P.G); r += NW * 64 / CPR) {
            *reinterpret_cast<u32x4 *>(view_row<T>(P.kcache, group, h, r) + piece) =
                *reinterpret_cast<const u32x4 *>(kc_h + static_cast<long>(r) * P.kc.sn + piece);
            *reinterpret_cast<u32x4 *>(view_row<T>(P.vcache, group, h, r) + piece) =
                *reinterpret_cast<const u32x4 *>(vc_h + static_cast<long>(r) * P.vc.sn + piece);
        }
    }

    vec qreg[KS];
    {
        const bool live = row0 + c < P.G;  // columns past the end carry zero queries, their results are not stored
        const int r = live ? row0 + c : row0;
        const T *qrow = view_row<T>(P.q, batch(r), h, query(r)) + 8 * hb;
        const float qs = live ? P.qscale : 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const u32x4 raw = *reinterpret_cast<const u32x4 *>(qrow + 16 * ks);
            u32x4 sc;  // scale * log2(e) folded in and rounded to the input type, as in mfma_flash.h
#pragma unroll
            for (int e = 0; e < 4; ++e) sc[e] = pack2<T>(unpack_lo<T>(raw[e]) * qs, unpack_hi<T>(raw[e]) * qs);
            qreg[ks] = __builtin_bit_cast(vec, sc);
        }
    }

    f32x16 o_acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) o_acc[db][v] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;  // per column: both lanes of a column hold the same maximum
    T *const vt = reinterpret_cast<T *>(lds) + wave * 32 * VPAD;
    T *const v_wr = vt + (lane / CPR) * VPAD + 8 * (lane % CPR);
    const int v_rd = (4 * hb + ((lane & 15) >> 2)) * VPAD + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    auto compute = [&](int blk, const Raw &r) {
        // (the LDS operations of a wavefront run in order: the last block's reads come first)
#pragma unroll
        for (int x = 0; x < VP; ++x) *reinterpret_cast<u32x4 *>(v_wr + x * (64 / CPR) * VPAD) = r.v[x];
        f32x16 s;
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s = Ops::mma(__builtin_bit_cast(vec, r.k[ks]), qreg[ks], s);
        const int key0 = 32 * blk;
        if (key0 + 32 > P.Nc) {
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (key0 + 8 * (v >> 2) + 4 * hb + (v & 3) >= P.Nc) s[v] = -INFINITY;
        }
        float tmax = s[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) tmax = fmaxf(tmax, s[v]);
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
        const float m_new = fmaxf(m_run, tmax);
        const float m_ref = m_new == -INFINITY ? 0.f : m_new;  // (every score so far -inf: no mass)
        const float alpha = fast_exp2(m_run - m_ref);
        if (__any(alpha != 1.f)) {
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int v = 0; v < 16; ++v) o_acc[db][v] *= alpha;
        }
        m_run = m_new;
        u32x4 pb[2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                pb[tt][e] = pack2<T>(fast_exp2(s[8 * tt + 2 * e] - m_ref), fast_exp2(s[8 * tt + 2 * e + 1] - m_ref));
                l_run = Ops::dot2(pb[tt][e], l_run);  // the mass of the probabilities as the second product takes them
            }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const T *vp = vt + 16 * tt * VPAD + 32 * db + v_rd;
                s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(vp));
                s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(vp + 8 * VPAD));
                typedef short s16x8 __attribute__((ext_vector_type(8)));
                s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                o_acc[db] = Ops::mma(__builtin_bit_cast(vec, both), __builtin_bit_cast(vec, pb[tt]), o_acc[db]);
            }
        __builtin_amdgcn_wave_barrier();
    };
    for (int blk = wave; blk < n_blocks;) {  // three blocks in turn: registers of fixed names
        if (blk + 2 * NW < n_blocks) fetch(blk + 2 * NW, r2);
        compute(blk, r0);
        if ((blk += NW) >= n_blocks) break;
        if (blk + 2 * NW < n_blocks) fetch(blk + 2 * NW, r0);
        compute(blk, r1);
        if ((blk += NW) >= n_blocks) break;
        if (blk + 2 * NW < n_blocks) fetch(blk + 2 * NW, r1);
        compute(blk, r2);
        blk += NW;
    }

    // partials: normalised, with their base-2 log-sum-exp (-inf: no mass)
    float(*const part_o)[NCOL][DH] = reinterpret_cast<float(*)[NCOL][DH]>(lds);
    const float l_tot = l_run + __shfl_xor(l_run, 32, 64), inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    __syncthreads();  // the V tiles are free
    if (hb == 0) part_lse2[wave][c] = l_tot > 0.f ? m_run + fast_log2(l_tot) : (l_tot == 0.f ? -INFINITY : l_tot);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const f32x4 val = {o_acc[db][4 * q4] * inv, o_acc[db][4 * q4 + 1] * inv, o_acc[db][4 * q4 + 2] * inv,
                               o_acc[db][4 * q4 + 3] * inv};
            *reinterpret_cast<f32x4 *>(&part_o[wave][c][32 * db + 8 * q4 + 4 * hb]) = val;
        }
    __syncthreads();
    // merged by 16 threads per column, DH / 16 neighbouring elements each
    constexpr int PER = DH / 16;
    const int col = threadIdx.x / 16, d0 = threadIdx.x % 16 * PER;
    if (row0 + col >= P.G) return;
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) mx = fmaxf(mx, part_lse2[w][col]);
    const float ref = mx == -INFINITY ? 0.f : mx;
    float wsum = 0.f, acc[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) acc[e] = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const float f = fast_exp2(part_lse2[w][col] - ref);
        wsum += f;
#pragma unroll
        for (int e = 0; e < PER; ++e) acc[e] = fmaf(f, part_o[w][col][d0 + e], acc[e]);
    }
    const float norm = wsum > 0.f ? 1.f / wsum : (wsum == 0.f ? 0.f : wsum);
    const int r = row0 + col, i = query(r);
    const long b = batch(r);
    T *orow = view_row<T>(P.out, b, h, i) + d0;
#pragma unroll
    for (int e = 0; e < PER; e += 2) *reinterpret_cast<unsigned *>(orow + e) = pack2<T>(acc[e] * norm, acc[e + 1] * norm);
    if (P.lse && d0 == 0) P.lse[(b * P.H + h) * P.Lq + i] = (ref + fast_log2(wsum)) * kLn2;
}

}  // namespace artab
