// Launches of the whole-run decode kernel (trajectory_decode.h), one object per element type:
// -DARTAB_TRAJ_TYPE=0 (bf16, with the type-dispatching entry points) | 1 (f16) | 2 (float32).
#include "launchers.h"
#include "trajectory_crews.h"

#ifndef ARTAB_TRAJ_TYPE
#error "define ARTAB_TRAJ_TYPE (0, 1 or 2)"
#endif

namespace artab {

#if ARTAB_TRAJ_TYPE == 0
typedef bf16_t TrajT;
#elif ARTAB_TRAJ_TYPE == 1
typedef f16_t TrajT;
#else
typedef float TrajT;
#endif

namespace {

// Runs `f` with the shape of (D, F) as a compile-time type; false where none is built.  The widths D are those
// whose activation tiles fit the LDS of one compute unit; F is the feed-forward width that the model's default
// and the training configuration have, others would be further instances (a model with one of them takes
// the step-by-step launches).
template <typename T, typename Fn>
bool with_shape(int D, int F, Fn f) {
    if (F == 256) {
        switch (D) {
            case 128: f(std::integral_constant<int, 128>{}, std::integral_constant<int, 256>{}); return true;
            case 256: f(std::integral_constant<int, 256>{}, std::integral_constant<int, 256>{}); return true;
            case 512:
                if constexpr (sizeof(T) == 2) {
                    f(std::integral_constant<int, 512>{}, std::integral_constant<int, 256>{});
                    return true;
                }
                return false;
            default: return false;
        }
    }
    return false;
}

template <typename T>
TrajectoryTapeLayout tape_layout(int D, int F, int n_layers) {
    TrajectoryTapeLayout t{};
    if (n_layers > kTrajMaxLayers) return t;
    with_shape<T>(D, F, [&](auto d, auto f) {
        typedef TrajShape<T, decltype(d)::value, decltype(f)::value> S;
        t.layer = S::kLayer;
        t.head = S::kHead;
        t.ring = S::kRing;
        t.max_group = TrajOps<T>::kMax;
        t.stride = (static_cast<long>(n_layers) * S::kLayer + S::kHead + S::kRing) * 1024;
        // first fragment, fragments per contraction step, blocks per wavefront of every matrix
        t.fo = {0, S::ND, 0, S::ND};
        for (int p = 0; p < 3; ++p) t.qkv[p] = {S::kFo, 3 * S::ND, p * S::ND, S::ND};
        t.o = {S::kFo + S::kQkv, S::ND, 0, S::ND};
        t.w1 = {S::kFo + S::kQkv + S::kO, S::NF, 0, S::NF};
        t.w2 = {S::kFo + S::kQkv + S::kO + S::k1, S::ND, 0, S::ND};
        t.h1 = {0, S::NF, 0, S::NF};
        t.h2 = {S::kH1, 1, 0, 1};
    });
    return t;
}

template <typename T>
hipError_t tape_matrix(const void *w, char *tape, long stride, int N, int K, const TrajectoryTapeLayout::Matrix &m,
                       int section, hipStream_t st) {
    const long frags = static_cast<long>(kTrajWaves) * m.per_wave * (K / TrajOps<T>::kStep);
    hipLaunchKernelGGL((trajectory_tape_kernel<T>), dim3(static_cast<unsigned>((frags + 3) / 4)), dim3(256), 0, st,
                       static_cast<const T *>(w), tape, stride, N, K, m.per_wave, section + m.first, m.step, m.offset);
    return hipGetLastError();
}

// Several workgroups to a trajectory: the heads are dealt over them.
template <typename T, int D, int F, int PARTS>
hipError_t launch_parts(const TrajectoryParams &P, hipStream_t st) {
    if constexpr (traj_parts_built(D, PARTS)) {
        const long words = 2L * P.B * traj_exchange_words<T>(D);
        hipLaunchKernelGGL(trajectory_exchange_kernel, dim3(static_cast<unsigned>((words + 255) / 256)), dim3(256), 0, st, P.exchange, words);
        hipLaunchKernelGGL((trajectory_crews_kernel<T, D, F, PARTS>), dim3(static_cast<unsigned>((P.B + 7) / 8 * 8 * PARTS)),
                           dim3(2 * kTrajWaves * 64), 0, st, P);
        return hipGetLastError();
    }
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t decode_parts(const TrajectoryParams &P, int D, int F, int parts, hipStream_t st) {
    hipError_t e = hipErrorInvalidValue;
    with_shape<T>(D, F, [&](auto d, auto f) {
        constexpr int kD = decltype(d)::value, kF = decltype(f)::value;
        e = parts == 2 ? launch_parts<T, kD, kF, 2>(P, st) : parts == 4 ? launch_parts<T, kD, kF, 4>(P, st)
            : parts == 8 ? launch_parts<T, kD, kF, 8>(P, st) : hipErrorInvalidValue;
    });
    return e;
}

template <typename T>
hipError_t decode(const TrajectoryParams &P, int D, int F, int parts, hipStream_t st) {
    hipError_t e = hipErrorInvalidValue;
    if (parts > 1) {  // and, behind it, one workgroup to each trajectory that has been given up
        e = decode_parts<T>(P, D, F, parts, st);
        if (e != hipSuccess) return e;
    }
    with_shape<T>(D, F, [&](auto d, auto f) {
        const dim3 grid(static_cast<unsigned>((P.B + P.G - 1) / P.G)), block(kTrajWaves * 64);
        if constexpr (decltype(d)::value <= 256) {
            if (crews_serve(P, D, sizeof(T) == 4)) {
                hipLaunchKernelGGL((trajectory_crews_kernel<T, decltype(d)::value, decltype(f)::value, 1>), grid, dim3(2 * kTrajWaves * 64), 0, st, P);
                e = hipGetLastError();
                return;
            }
        }
        if (P.G > 1) {
            hipLaunchKernelGGL((trajectory_decode_kernel<T, decltype(d)::value, decltype(f)::value, true>), grid, block, 0, st, P);
            e = hipGetLastError();
        } else if constexpr (sizeof(T) == 2) {  // (in float32 the crews take all of them)
            hipLaunchKernelGGL((trajectory_decode_kernel<T, decltype(d)::value, decltype(f)::value, false>), grid, block, 0, st, P);
            e = hipGetLastError();
        }
    });
    return e;
}

}  // namespace

#define ARTAB_TRAJ_FORMS(suffix)                                                                                      \
    TrajectoryTapeLayout trajectory_tape_layout_##suffix(int D, int F, int n_layers) {                                \
        return tape_layout<TrajT>(D, F, n_layers);                                                                    \
    }                                                                                                                 \
    hipError_t launch_trajectory_tape_##suffix(const void *w, char *tape, long stride, int N, int K,                  \
                                               const TrajectoryTapeLayout::Matrix &m, int section, hipStream_t st) { \
        return tape_matrix<TrajT>(w, tape, stride, N, K, m, section, st);                                             \
    }                                                                                                                 \
    hipError_t launch_trajectory_decode_##suffix(const TrajectoryParams &P, int D, int F, int parts, hipStream_t st) { \
        return decode<TrajT>(P, D, F, parts, st);                                                                     \
    }

#if ARTAB_TRAJ_TYPE == 0
ARTAB_TRAJ_FORMS(bf16)

// Repeats the first `bytes` bytes of every tape behind its end.
static __global__ void trajectory_tape_wrap_kernel(char *tape, long tape_stride, long bytes) {
    const long chunk = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
    const long per = bytes / 16;
    if (chunk >= per * kTrajWaves) return;
    char *t = tape + chunk / per * tape_stride;
    const long at = chunk % per * 16;
    *reinterpret_cast<u32x4 *>(t + tape_stride - bytes + at) = *reinterpret_cast<const u32x4 *>(t + at);
}

hipError_t launch_trajectory_tape_wrap(char *tape, long stride, long bytes, hipStream_t st) {
    const long chunks = bytes / 16 * kTrajWaves;
    hipLaunchKernelGGL(trajectory_tape_wrap_kernel, dim3(static_cast<unsigned>((chunks + 255) / 256)), dim3(256), 0, st, tape,
                       stride, bytes);
    return hipGetLastError();
}
#elif ARTAB_TRAJ_TYPE == 1
ARTAB_TRAJ_FORMS(f16)
#else
ARTAB_TRAJ_FORMS(f32)
#endif

}  // namespace artab
