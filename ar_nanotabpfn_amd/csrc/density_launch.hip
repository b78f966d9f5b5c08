// Launches of the kernels at both ends of a prefill or a density (density_rows.h; include/artab_attention.h).
#include "../../include/artab_attention.h"
#include "density_rows.h"
#include "launchers.h"

namespace artab {
namespace {

bool off_16(const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 != 0; }
template <typename... P>
bool any_null(P... p) {
    return ((p == nullptr) || ...);
}

template <typename T>
int embed(const artab_embed_rows_args &a, hipStream_t st) {
    EmbedRowsParams P{};
    P.x = a.x; P.y = a.y; P.xb = a.x_stride_b; P.xn = a.x_stride_n; P.xc = a.x_stride_c; P.yb = a.y_stride_b; P.yn = a.y_stride_n;
    P.B = a.B; P.N = a.N; P.C = a.C; P.D = a.D; P.one_over_c = 1. / a.C; P.pairs = a.pairs;
    P.w_x = a.w_x; P.b_x = a.b_x; P.w_y = a.w_y; P.b_y = a.b_y; P.markers = a.markers; P.tokens = a.ar_tokens; P.bs = a.bs; P.out = a.out;
    const long threads = static_cast<long>(a.B) * a.N * (a.pairs ? 2 : 1) * (a.D * static_cast<long>(sizeof(T)) / 16);
    hipLaunchKernelGGL((embed_rows_kernel<T>), dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, st, P);
    return hipGetLastError() == hipSuccess ? ARTAB_OK : ARTAB_ERR_LAUNCH;
}

template <typename T>
int density(const artab_density_args &a, hipStream_t st) {
    DensityParams P{};
    P.x = a.x; P.xb = a.x_stride_b; P.norm_g = a.norm_gamma; P.norm_b = a.norm_beta; P.eps = a.eps;
    P.w1 = a.w1; P.b1 = a.b1; P.w2 = a.w2; P.b2 = a.b2; P.mean_bias = a.mean_bias; P.std_bias = a.std_bias; P.weight_bias = a.weight_bias;
    P.K = a.K; P.std_min = a.std_min; P.y = a.y; P.yb = a.y_stride_b; P.yn = a.y_stride_n; P.out = a.out; P.B = a.B; P.Nt = a.Nt;
    const dim3 grid(static_cast<unsigned>((static_cast<long>(a.B) * a.Nt + kDensityRows - 1) / kDensityRows)), block(kDensityWaves * 64);
    if (a.D == 128) hipLaunchKernelGGL((density_kernel<T, 128, 256>), grid, block, 0, st, P);
    else if (a.D == 256) hipLaunchKernelGGL((density_kernel<T, 256, 256>), grid, block, 0, st, P);
    else hipLaunchKernelGGL((density_kernel<T, 512, 256>), grid, block, 0, st, P);
    return hipGetLastError() == hipSuccess ? ARTAB_OK : ARTAB_ERR_LAUNCH;
}

template <typename Fn>
int by_type(int dtype, Fn f) {
    if (dtype == ARTAB_BF16) return f(bf16_t{});
    if (dtype == ARTAB_F16) return f(f16_t{});
    if (dtype == ARTAB_F32) return f(float{});
    return ARTAB_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace artab

extern "C" {

int artab_embed_rows(const artab_embed_rows_args *a, int dtype, void *stream) {
    using namespace artab;
    if (!a) return ARTAB_ERR_NULL_POINTER;
    if (dtype != ARTAB_BF16 && dtype != ARTAB_F16 && dtype != ARTAB_F32) return ARTAB_ERR_UNSUPPORTED;
    if (a->D < 8 || a->D % 8) return ARTAB_ERR_UNSUPPORTED;
    if (a->B < 0 || a->N < 0 || a->C < 1 || (a->pairs && a->bs < 1) || (a->D && static_cast<int64_t>(a->B) * a->N >= (int64_t{1} << 32) / a->D))
        return ARTAB_ERR_BAD_SHAPE;  // (2^33 / D rows: fewer than 2^31 threads)
    if (a->B == 0 || a->N == 0) return ARTAB_OK;
    if (any_null(a->x, a->y, a->w_x, a->b_x, a->w_y, a->b_y, a->markers, static_cast<const void *>(a->out)) || (a->pairs && !a->ar_tokens))
        return ARTAB_ERR_NULL_POINTER;
    for (const void *p : {a->w_x, a->b_x, a->w_y, a->b_y, a->markers, a->ar_tokens, static_cast<const void *>(a->out)})
        if (off_16(p)) return ARTAB_ERR_BAD_STRIDE;
    return by_type(dtype, [&](auto t) { return embed<decltype(t)>(*a, static_cast<hipStream_t>(stream)); });
}

int artab_density_supported(int D, int F, int K) {
    return (D == 128 || D == 256 || D == 512) && F == 256 && K >= 1 && 3 * K <= artab::kDensityMaxOut;
}

int artab_density(const artab_density_args *a, int dtype, void *stream) {
    using namespace artab;
    if (!a) return ARTAB_ERR_NULL_POINTER;
    if (!artab_density_supported(a->D, a->F, a->K)) return ARTAB_ERR_UNSUPPORTED;
    if (a->B < 0 || a->Nt < 0 || static_cast<int64_t>(a->B) * a->Nt >= (1 << 30)) return ARTAB_ERR_BAD_SHAPE;
    if (a->B == 0 || a->Nt == 0) return dtype == ARTAB_BF16 || dtype == ARTAB_F16 || dtype == ARTAB_F32 ? ARTAB_OK : ARTAB_ERR_UNSUPPORTED;
    if (any_null(a->x, a->norm_gamma, a->norm_beta, a->w1, a->b1, a->w2, a->b2, a->mean_bias, a->std_bias, a->weight_bias, a->y,
                 static_cast<const void *>(a->out)))
        return ARTAB_ERR_NULL_POINTER;
    if (off_16(a->w1) || off_16(a->w2)) return ARTAB_ERR_BAD_STRIDE;
    return by_type(dtype, [&](auto t) { return density<decltype(t)>(*a, static_cast<hipStream_t>(stream)); });
}

}  // extern "C"
