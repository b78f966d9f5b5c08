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

template <int D, int TR>
static void launch(const F32LayerParams &P, hipStream_t st) {
    const dim3 grid(static_cast<unsigned>((P.rows + TR - 1) / TR)), block(f32_layer_waves(D) * 64);
    launch_observed(kLaunchLayer, f32_layer_kernel<D, 256, TR>, grid, block, 0, st, P);
}
// Rows per workgroup: the fewest that one workgroup per compute unit covers, 16 where none does.  A prefill of 12 layers
// and their attention, us with 16 / 8 / 4 rows (256 compute units):
//   d_model 128:  333 rows  331 /  284 /  259, 1000  478 /  427 /  400, 1500  675 /  625 /  638, 2000  952 /  898 /  908, 2500 1183 / 1213 / 1203
//   d_model 256:  333 rows  559 /  417 /  364, 1000  667 /  527 /  477, 1500  904 /  768 /  892, 2000 1025 /  900 / 1016, 2500 1421 / 1522 / 1591
//   d_model 512:  333 rows 1550 / 1002 /  835, 1000 1719 / 1194 / 1057, 1500 2011 / 1497 / 1961, 2000 2396 / 2000 / 2385, 2500 2891 / 3263 / 3503
template <int D>
static void launch(const F32LayerParams &P, hipStream_t st) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    if (P.rows <= 4L * cus) launch<D, 4>(P, st);
    else if (P.rows <= 8L * cus) launch<D, 8>(P, st);
    else launch<D, 16>(P, st);
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
