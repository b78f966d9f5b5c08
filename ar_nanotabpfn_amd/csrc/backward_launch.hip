// Launches of the backward kernels of the training row attention (attention_backward.h):
// template selection by element type and head_dim.
#include "attention_backward_pair.h"
#include "launchers.h"

namespace artab {

template <typename T>
static hipError_t launch_backward_portable(const BackwardParams &P, hipStream_t stream) {
    const long total = static_cast<long>(P.B) * P.H * P.R;
    const dim3 grid(static_cast<unsigned>((total + kPortableWaves - 1) / kPortableWaves)), block(kPortableWaves * 64);
    // the dK/dV kernel reads the delta workspace that the dQ kernel leaves: same stream, in this order
    if (P.Dh <= 64) {
        hipLaunchKernelGGL((backward_dq_portable_kernel<T, 1>), grid, block, 0, stream, P);
        hipLaunchKernelGGL((backward_dkv_portable_kernel<T, 1>), grid, block, 0, stream, P);
    } else if (P.Dh <= 128) {
        hipLaunchKernelGGL((backward_dq_portable_kernel<T, 2>), grid, block, 0, stream, P);
        hipLaunchKernelGGL((backward_dkv_portable_kernel<T, 2>), grid, block, 0, stream, P);
    } else {
        hipLaunchKernelGGL((backward_dq_portable_kernel<T, 4>), grid, block, 0, stream, P);
        hipLaunchKernelGGL((backward_dkv_portable_kernel<T, 4>), grid, block, 0, stream, P);
    }
    return hipGetLastError();
}

template <typename T, int DH, int W, int G>
static hipError_t launch_backward_pair(const BackwardParams &P, hipStream_t stream) {
    hipLaunchKernelGGL((backward_pair_kernel<T, DH, W, G>), dim3(static_cast<unsigned>(P.H) * P.B), dim3(64 * W * G), 0, stream, P);
    return hipGetLastError();
}

template <typename T>
static hipError_t launch_backward_mfma(const BackwardParams &P, hipStream_t stream) {
    // One workgroup per pair (backward_pair_kernel) while the keys that anybody sees fit it.  It stays on one compute
    // unit: with up to 128 keys it is the faster form at any number of pairs (head_dim 32, 96 keys, 608 rows: 21.5 against
    // 18.7 us for 16 pairs, 45.7 against 24.3 for 256); with more, the two kernels' many workgroups win while pairs are few
    // (256 keys, 768 rows: 31.7 against 33.2 at 64 pairs, 36.1 against 34.2 at 96; 512 keys, 1024 rows: 59 against 71 at
    // 96, 106 against 77 at 192; head_dim 64, 256 keys: 58 against 61 at 128, 71 against 64 at 192).  Where pairs need
    // one more round of the chip's 256 compute units, that round has to be half full: 300 pairs of 512 keys 156
    // against 146 us.  Up to 128 keys, two workgroups of half the groups to a unit then (300 pairs, 96 keys: 52 against 32).
    const long pairs = static_cast<long>(P.H) * P.B, rounds = (pairs + 255) / 256;
    const int keys = P.Nc + P.Nb;
    const bool filled = pairs >= 150 * rounds;
    if (P.Dh == 32) {
        if (keys <= 128) return pairs <= 256 ? launch_backward_pair<T, 32, 4, 4>(P, stream) : launch_backward_pair<T, 32, 4, 2>(P, stream);
        if (keys <= 256 && (filled || (pairs >= 80 && rounds == 1))) return launch_backward_pair<T, 32, 8, 2>(P, stream);
        if (keys <= 512 && filled) return launch_backward_pair<T, 32, 16, 1>(P, stream);
    } else {
        if (keys <= 128) return launch_backward_pair<T, 64, 4, 2>(P, stream);
        if (keys <= 256 && filled) return launch_backward_pair<T, 64, 8, 1>(P, stream);
    }
    const long blocks = (P.R + kBackwardRows - 1) / kBackwardRows;
    const dim3 grid(static_cast<unsigned>(blocks * P.H * P.B)), block(kBackwardWaves * 64);
    if (P.Dh == 32) {
        hipLaunchKernelGGL((backward_dq_mfma_kernel<T, 32>), grid, block, 0, stream, P);
        hipLaunchKernelGGL((backward_dkv_mfma_kernel<T, 32>), grid, block, 0, stream, P);
    } else {
        hipLaunchKernelGGL((backward_dq_mfma_kernel<T, 64>), grid, block, 0, stream, P);
        hipLaunchKernelGGL((backward_dkv_mfma_kernel<T, 64>), grid, block, 0, stream, P);
    }
    return hipGetLastError();
}

hipError_t launch_row_mask_backward(const BackwardParams &P, int elem, bool use_mfma, hipStream_t stream) {
    if (static_cast<long>(P.B) * P.H * P.R == 0) return hipSuccess;
    if (use_mfma) return elem == kElemBf16 ? launch_backward_mfma<bf16_t>(P, stream) : launch_backward_mfma<f16_t>(P, stream);
    switch (elem) {
        case kElemBf16: return launch_backward_portable<bf16_t>(P, stream);
        case kElemF16: return launch_backward_portable<f16_t>(P, stream);
        default: return launch_backward_portable<float>(P, stream);
    }
}

}  // namespace artab
