// Launches of the float32 layer kernel (f32_layer.h).
#include "f32_layer.h"
#include "launchers.h"

namespace artab {

// [N, K] float32 -> [N / 16][K / 16][64][4], the fragment order above.
__global__ __launch_bounds__(256) void f32_pack_kernel(const float *w, float *packed, int N, int K) {
    const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= static_cast<long>(N) * K / 4) return;
    const int lane = static_cast<int>(i & 63);
    const long f = i >> 6;
    const int t = static_cast<int>(f % (K / 16)), nb = static_cast<int>(f / (K / 16));
    reinterpret_cast<f32x4 *>(packed)[i] =
        *reinterpret_cast<const f32x4 *>(w + static_cast<long>(16 * nb + (lane & 15)) * K + 16 * t + 4 * (lane >> 4));
}

bool f32_layer_width_ok(int D, int F) { return (D == 128 || D == 256 || D == 512) && F == 256; }

template <int D>
static void launch(const F32LayerParams &P, hipStream_t st) {
    const dim3 grid(static_cast<unsigned>((P.rows + kF32Rows - 1) / kF32Rows)), block(f32_layer_waves(D) * 64);
    launch_observed(kLaunchLayer, f32_layer_kernel<D, 256>, grid, block, 0, st, P);
}

hipError_t launch_f32_layer(const F32LayerParams &P, int D, hipStream_t st) {
    switch (D) {
        case 128: launch<128>(P, st); break;
        case 256: launch<256>(P, st); break;
        default: launch<512>(P, st); break;
    }
    return hipGetLastError();
}

hipError_t launch_f32_pack(const float *w, float *packed, int N, int K, hipStream_t st) {
    const long pieces = static_cast<long>(N) * K / 4;
    hipLaunchKernelGGL(f32_pack_kernel, dim3(static_cast<unsigned>((pieces + 255) / 256)), dim3(256), 0, st, w, packed, N, K);
    return hipGetLastError();
}

}  // namespace artab
