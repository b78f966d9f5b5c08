// Launches of the float32 attention kernel (f32_attention.h).
#include "f32_attention.h"
#include "launchers.h"

namespace artab {

// Which form a call takes, from its sizes.  A tile of 32 rows per wavefront (16 where a group has no more)
// keeps the matrix cores busiest and is taken from two such wavefronts per SIMD on; with fewer, a
// tile's keys are dealt over the eight wavefronts of a workgroup, in tiles of 16 rows until there is a
// workgroup for every compute unit, and over several workgroups where even that leaves compute units
// idle and a wavefront would still have two blocks of keys.
F32Shape plan_f32(int H, int Nc, int Dh, int G, int n_groups) {
    F32Shape s;
    const long groups = static_cast<long>(H) * n_groups;
    auto tiles = [&](int cols) { return groups * ((G + cols - 1) / cols); };
    s.qb = G <= 16 || Dh == 128 ? 1 : 2;  // (head_dim 128: registers)
    s.split = tiles(16 * s.qb) < 2048;
    if (s.split && tiles(32) < 256) s.qb = 1;
    s.n_split = 1;
    if (s.split) {
        const long wgs = tiles(16 * s.qb), blocks = (Nc + 31) / 32;
        if (wgs < 256) {
            const long want = (512 + wgs - 1) / wgs, most = blocks / 16;
            const long n = want < most ? want : most;
            s.n_split = static_cast<int>(n < 1 ? 1 : n > 32 ? 32 : n);
        }
    }
    return s;
}

template <int DH, int QB, bool HIDES>
static hipError_t launch_hides(const PortableParams &P, const F32Plan &L, bool split, hipStream_t st) {
    const long kvg8 = (static_cast<long>(P.H) * L.n_groups + 7) / 8;
    if (split) {
        const unsigned grid = static_cast<unsigned>(8 * kvg8 * L.tiles * L.n_split);
        hipLaunchKernelGGL((f32_attention_kernel<DH, QB, true, 8, HIDES>), dim3(grid), dim3(512), 0, st, P, L);
        if (L.n_split > 1)
            hipLaunchKernelGGL(f32_combine_kernel<DH>, dim3(static_cast<unsigned>((L.rows * (DH / 4) + 255) / 256)), dim3(256), 0, st, P, L);
    } else {
        const unsigned grid = static_cast<unsigned>(8 * kvg8 * ((L.tiles + 3) / 4));
        hipLaunchKernelGGL((f32_attention_kernel<DH, QB, false, 4, HIDES>), dim3(grid), dim3(256), 0, st, P, L);
    }
    return hipGetLastError();
}

// A context alone is seen by every column: its calls go without the watch for values that have to be kept apart
// (one query on 4000 rows 13.5 -> 13.1 us).
template <int DH, int QB>
static hipError_t launch(const PortableParams &P, const F32Plan &L, bool split, hipStream_t st) {
    return P.Nb > 0 || P.new_row >= 0 || P.nbuf_dev ? launch_hides<DH, QB, true>(P, L, split, st) : launch_hides<DH, QB, false>(P, L, split, st);
}

hipError_t launch_f32_attention(PortableParams P, bool stacked, void *workspace, size_t workspace_bytes, hipStream_t st) {
    F32Plan L;
    L.stacked = stacked ? 1 : 0;
    L.G = stacked ? P.B * P.Lq : P.Lq;
    L.n_groups = stacked ? 1 : P.B;
    L.rows = static_cast<long>(P.B) * P.H * P.Lq;
    F32Shape s = plan_f32(P.H, P.Nc, P.Dh, L.G, L.n_groups);
    if (s.n_split > 1 && (!workspace || workspace_bytes < f32_workspace_bytes(L.rows, P.Dh, s.n_split) ||
                          reinterpret_cast<uintptr_t>(workspace) % 16))
        s.n_split = 1;  // correct without scratch memory, only less parallel
    L.tiles = (L.G + 16 * s.qb - 1) / (16 * s.qb);
    L.n_split = s.n_split;
    L.part_o = static_cast<float *>(workspace);
    L.part_lse = L.part_o + L.rows * P.Dh * s.n_split;
    P.scale *= kLog2e;
    switch (P.Dh) {
        case 32: return s.qb == 1 ? launch<32, 1>(P, L, s.split, st) : launch<32, 2>(P, L, s.split, st);
        case 64: return s.qb == 1 ? launch<64, 1>(P, L, s.split, st) : launch<64, 2>(P, L, s.split, st);
        default: return launch<128, 1>(P, L, s.split, st);
    }
}

}  // namespace artab
