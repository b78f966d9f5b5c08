// The layer stack of a training step: buffers and launches of the kernels of train_layers.h around the row
// attention (include/artab_attention.h, artab_train_*).
#include "../../include/artab_attention.h"
#include "launchers.h"
#include "train_head.h"
#include "train_layers.h"

namespace artab {
namespace {

constexpr int kParams = 16;  // per layer, in the order of artab_train_args.params
enum ParamIndex : int { kPFeatV, kPFeatOut, kPQ, kPK, kPV, kPO, kPW1, kPBias1, kPW2, kPBias2, kPG1, kPB1, kPG2, kPB2, kPG3, kPB3 };

struct Arena {  // deals out 256-byte aligned pieces of one allocation (or only counts them)
    char *base;
    size_t used = 0;
    explicit Arena(void *p) : base(static_cast<char *>(p)) {}
    template <typename T>
    T *take(size_t n) {
        T *r = base ? reinterpret_cast<T *>(base + used) : nullptr;
        used += (n * sizeof(T) + 255) / 256 * 256;
        return r;
    }
};

struct SavedLayer {
    float *r1, *r2, *r3, *lse;
    float2 *stats1, *stats2, *stats3;
    bf16_t *qkv, *attn;
};
struct Saved {
    bf16_t *packed;
    float *fo;
    char *layers;
    size_t layer_bytes, bytes;
    SavedLayer layer(const artab_train_args &a, int l) const {
        const size_t M = static_cast<size_t>(a.B) * a.R;
        Arena s(layers ? layers + l * layer_bytes : nullptr);
        return take(a, M, s);
    }
    static SavedLayer take(const artab_train_args &a, size_t M, Arena &s) {
        SavedLayer v;
        v.r1 = s.take<float>(M * a.D);
        v.r2 = s.take<float>(M * a.D);
        v.r3 = s.take<float>(M * a.D);
        v.lse = s.take<float>(M * a.H);
        v.stats1 = s.take<float2>(M);
        v.stats2 = s.take<float2>(M);
        v.stats3 = s.take<float2>(M);
        v.qkv = s.take<bf16_t>(M * 3 * a.D);
        v.attn = s.take<bf16_t>(M * a.D);
        return v;
    }
};
size_t packed_elems(int D, int F) { return 2 * (5 * static_cast<size_t>(D) * D + 2 * static_cast<size_t>(D) * F); }

Saved saved_layout(const artab_train_args &a) {
    Saved v;
    Arena s(a.saved);
    v.packed = s.take<bf16_t>(a.n_layers * packed_elems(a.D, a.F));
    v.fo = s.take<float>(static_cast<size_t>(a.n_layers) * a.D * a.D);
    v.layers = a.saved ? s.base + s.used : nullptr;
    Arena one(nullptr);
    Saved::take(a, static_cast<size_t>(a.B) * a.R, one);
    v.layer_bytes = one.used;
    v.bytes = s.used + v.layer_bytes * a.n_layers;
    return v;
}

// offsets (floats) inside a layer's gradients
struct GradLayout {
    long qkv, fo, o, w1, w2, vec_b, vec_a, out, v, total;
    GradLayout(int D, int F) {
        const long dd = static_cast<long>(D) * D, df = static_cast<long>(D) * F;
        qkv = 0; fo = 3 * dd; o = 4 * dd; w1 = 5 * dd; w2 = w1 + df;
        vec_b = w2 + df;           // g3, b3, bias2, g2, b2, bias1
        vec_a = vec_b + 5 * D + F; // g1, b1
        out = vec_a + 2 * D; v = out + dd;
        total = v + dd;
    }
};

// Workgroups of the backward kernel: as many as are resident, three to a compute unit at d_model 128, two at 256.
// (Of 1216 tiles some then have two, some one; 608 workgroups of two each: 83 us instead of 74, some compute units
// with six tiles, some with four.)
int backward_groups(long M, int D) {
    const long resident = D == 128 ? 768 : 512, tiles = (M + kTrainRows - 1) / kTrainRows;
    return static_cast<int>(tiles < resident ? tiles : resident);
}
int grad_jobs(int D, int F) { return (5 * D * D + 2 * D * F) / (128 * 128); }
// Row slices of the weight-gradient products: enough that pieces times slices give every compute unit a
// workgroup, none shorter than 256 rows.
int grad_slices(long M, int jobs) {
    const long most = (M + 255) / 256, want = (256 + jobs - 1) / jobs;
    return static_cast<int>(want < most ? want : most);
}
constexpr int kFinalGroups = 512;

struct Scratch {
    float *dx, *dr2, *delta, *part_w, *part_c, *part_f;
    bf16_t *d3, *x2, *h, *du, *d2, *dattn, *dqkv, *x1, *d1, *x;
    size_t bytes;
};
Scratch scratch_layout(const artab_train_args &a) {
    const size_t M = static_cast<size_t>(a.B) * a.R, D = a.D, F = a.F;
    const int groups = backward_groups(M, a.D), jobs = grad_jobs(a.D, a.F);
    Scratch v;
    Arena s(a.scratch);
    v.dx = s.take<float>(M * D);
    v.dr2 = s.take<float>(M * D);
    v.delta = s.take<float>(M * a.H);
    v.part_w = s.take<float>(static_cast<size_t>(grad_slices(M, jobs)) * jobs * 16384);
    v.part_c = s.take<float>(groups * (7 * D + F));
    v.part_f = s.take<float>(kFinalGroups * 2 * D);
    v.d3 = s.take<bf16_t>(M * D);
    v.x2 = s.take<bf16_t>(M * D);
    v.h = s.take<bf16_t>(M * F);
    v.du = s.take<bf16_t>(M * F);
    v.d2 = s.take<bf16_t>(M * D);
    v.dattn = s.take<bf16_t>(M * D);
    v.dqkv = s.take<bf16_t>(M * 3 * D);
    v.x1 = s.take<bf16_t>(M * D);
    v.d1 = s.take<bf16_t>(M * D);
    v.x = s.take<bf16_t>(M * D);
    v.bytes = s.used;
    return v;
}

TrainWeights weights(const artab_train_args &a, int first) {
    TrainWeights w{};
    for (int i = 0; i < kTrainPackLayers && first + i < a.n_layers; ++i) {
        const float *const *p = a.params + static_cast<size_t>(first + i) * kParams;
        w.v[i] = p[kPFeatV]; w.out[i] = p[kPFeatOut];
        w.q[i] = p[kPQ]; w.k[i] = p[kPK]; w.vr[i] = p[kPV]; w.o[i] = p[kPO];
        w.w1[i] = p[kPW1]; w.w2[i] = p[kPW2];
    }
    return w;
}

struct HeadViews {
    artab_view q, k, v, out;
};
HeadViews head_views(const artab_train_args &a, bf16_t *qkv, bf16_t *out) {
    const int64_t D = a.D, Dh = a.D / a.H;
    auto part = [&](int i) { return artab_view{qkv + i * D, a.R * 3 * D, Dh, 3 * D}; };
    return {part(0), part(1), part(2), artab_view{out, a.R * D, Dh, D}};
}

#define TRAIN_TRY(expr)             \
    do {                            \
        const int rc_ = (expr);     \
        if (rc_ != ARTAB_OK) return rc_; \
    } while (0)

template <int D, int F>
int forward(const artab_train_args &a, hipStream_t st) {
    const Saved S = saved_layout(a);
    const long M = static_cast<long>(a.B) * a.R;
    for (int l0 = 0; l0 < a.n_layers; l0 += kTrainPackLayers) {
        const TrainWeights W = weights(a, l0);
        const unsigned n = static_cast<unsigned>(a.n_layers - l0 < kTrainPackLayers ? a.n_layers - l0 : kTrainPackLayers);
        float *fo = S.fo + static_cast<long>(l0) * D * D;
        hipLaunchKernelGGL((train_fold_kernel<D>), dim3(D / 16, n), dim3(D), 0, st, W, fo);
        hipLaunchKernelGGL((train_pack_kernel<D, F>), dim3(static_cast<unsigned>((train_packed_elems<D, F>() / 8 + 255) / 256), n), dim3(256),
                           0, st, W, fo, S.packed + l0 * train_packed_elems<D, F>());
    }
    const dim3 grid(static_cast<unsigned>((M + kTrainRows - 1) / kTrainRows)), block(kTrainWaves * 64);
    for (int l = 0; l <= a.n_layers; ++l) {  // launch l: behind the attention of layer l - 1, in front of that of layer l
        TrainForward A{};
        A.M = M;
        if (l == 0) {
            A.x = a.x;
        } else {
            const float *const *p = a.params + static_cast<size_t>(l - 1) * kParams;
            const SavedLayer v = S.layer(a, l - 1);
            A.attn = v.attn; A.r1 = v.r1; A.stats1 = v.stats1; A.g1 = p[kPG1]; A.b1 = p[kPB1]; A.packed = S.packed + (l - 1) * train_packed_elems<D, F>();
            A.g2 = p[kPG2]; A.b2 = p[kPB2]; A.bias1 = p[kPBias1]; A.bias2 = p[kPBias2]; A.eps2 = a.eps2; A.eps3 = a.eps3;
            A.r2 = v.r2; A.stats2 = v.stats2; A.r3 = v.r3; A.stats3 = v.stats3; A.g3 = p[kPG3]; A.b3 = p[kPB3];
        }
        if (l == a.n_layers) {
            hipLaunchKernelGGL((train_forward_kernel<D, F, true, false>), grid, block, 0, st, A);
            break;
        }
        const float *const *p = a.params + static_cast<size_t>(l) * kParams;
        const SavedLayer v = S.layer(a, l);
        A.next_packed = S.packed + l * train_packed_elems<D, F>(); A.next_g1 = p[kPG1]; A.next_b1 = p[kPB1]; A.next_eps1 = a.eps1;
        A.next_r1 = v.r1; A.next_stats1 = v.stats1; A.next_qkv = v.qkv;
        if (l == 0)
            hipLaunchKernelGGL((train_forward_kernel<D, F, false, true>), grid, block, 0, st, A);
        else
            hipLaunchKernelGGL((train_forward_kernel<D, F, true, true>), grid, block, 0, st, A);
        const HeadViews h = head_views(a, v.qkv, v.attn);
        TRAIN_TRY(artab_row_mask_attention(&h.q, &h.k, &h.v, &h.out, v.lse, a.B, a.H, a.R, a.context_len, a.buffer_len, a.attending_chunks,
                                           D / a.H, 0.f, ARTAB_BF16, ARTAB_IMPL_AUTO, st));
    }
    const float *const *p = a.params + static_cast<size_t>(a.n_layers - 1) * kParams;
    const SavedLayer v = S.layer(a, a.n_layers - 1);
    TrainFinal Z{};
    Z.r3 = v.r3; Z.stats3 = v.stats3; Z.g3 = p[kPG3]; Z.b3 = p[kPB3]; Z.g = a.norm_gamma; Z.b = a.norm_beta; Z.eps = a.eps_out;
    Z.z = a.z; Z.B = a.B; Z.R = a.R; Z.first = a.first_row;
    const long rows = static_cast<long>(a.B) * (a.R - a.first_row);
    hipLaunchKernelGGL((train_final_kernel<D, false>), dim3(static_cast<unsigned>((rows + 3) / 4 < 2048 ? (rows + 3) / 4 : 2048)), dim3(256), 0, st, Z);
    return hipGetLastError() == hipSuccess ? ARTAB_OK : ARTAB_ERR_LAUNCH;
}

// Weight gradients of a launch: C[n][k] = sum_m P[m][n] Q[m][k] in pieces, and the workgroups' column sums.
struct GradProducts {
    TrainGradJobs jobs{};
    TrainReduce reduce{};
    GradProducts(long M, int slices, float *part) {
        jobs.part = part; jobs.M = M; jobs.rows_per_slice = ((M + slices - 1) / slices + 63) / 64 * 64;
        reduce.part = part; reduce.slices = slices;
    }
    void add(const bf16_t *P, int ldp, const bf16_t *Q, int ldq, int N, int K, float *out) {
        for (int n = 0; n < N; n += 128)
            for (int k = 0; k < K; k += 128) {
                const int i = jobs.jobs++;
                jobs.p[i] = P + n; jobs.q[i] = Q + k; jobs.ldp[i] = ldp; jobs.ldq[i] = ldq;
                reduce.out[i] = out + static_cast<long>(n) * K + k; reduce.ld[i] = K;
            }
    }
    void launch(hipStream_t st) {
        reduce.jobs = jobs.jobs;
        int columns = 0;
        for (int i = 0; i < reduce.n_cols; ++i) columns += reduce.cols[i].n;
        hipLaunchKernelGGL(train_weight_grad_kernel, dim3(jobs.jobs, reduce.slices), dim3(512), 0, st, jobs);
        hipLaunchKernelGGL(train_reduce_kernel, dim3(jobs.jobs * 16 + columns / kTrainReduceCols), dim3(256), 0, st, reduce);
    }
};

template <int D, int F>
int backward(const artab_train_args &a, hipStream_t st) {
    const Saved S = saved_layout(a);
    const Scratch X = scratch_layout(a);
    const GradLayout G(D, F);
    const long M = static_cast<long>(a.B) * a.R;
    const int groups = backward_groups(M, a.D), jobs = grad_jobs(D, F), slices = grad_slices(M, jobs);
    const dim3 block(kTrainWaves * 64);
    {
        const float *const *p = a.params + static_cast<size_t>(a.n_layers - 1) * kParams;
        const SavedLayer v = S.layer(a, a.n_layers - 1);
        TrainFinal Z{};
        Z.r3 = v.r3; Z.stats3 = v.stats3; Z.g3 = p[kPG3]; Z.b3 = p[kPB3]; Z.g = a.norm_gamma; Z.b = a.norm_beta; Z.eps = a.eps_out;
        Z.dz = a.dz; Z.dx = X.dx; Z.part = X.part_f; Z.B = a.B; Z.R = a.R; Z.first = a.first_row;
        hipLaunchKernelGGL((train_final_kernel<D, true>), dim3(kFinalGroups), dim3(256), 0, st, Z);
        TrainReduce T{};
        T.cols[0] = {X.part_f, a.grads + a.n_layers * G.total, kFinalGroups, 2 * D, 2 * D};
        T.n_cols = 1;
        hipLaunchKernelGGL(train_reduce_kernel, dim3(2 * D / kTrainReduceCols), dim3(256), 0, st, T);
    }
    for (int l = a.n_layers; l >= 0; --l) {  // launch l: the front of layer l, then the back of layer l - 1
        TrainBackward A{};
        GradProducts products(M, slices, X.part_w);
        A.M = M; A.dr2 = X.dr2; A.part = X.part_c; A.dx = l > 0 ? X.dx : a.dx;
        if (l < a.n_layers) {
            const float *const *p = a.params + static_cast<size_t>(l) * kParams;
            const SavedLayer v = S.layer(a, l);
            const HeadViews h = head_views(a, v.qkv, v.attn), d = head_views(a, X.dqkv, X.dattn);
            TRAIN_TRY(artab_row_mask_attention_backward(&h.q, &h.k, &h.v, &h.out, &d.out, v.lse, X.delta, &d.q, &d.k, &d.v, a.B, a.H, a.R,
                                                        a.context_len, a.buffer_len, a.attending_chunks, D / a.H, 0.f, ARTAB_BF16, ARTAB_IMPL_AUTO, st));
            A.dqkv = X.dqkv; A.r1 = v.r1; A.stats1 = v.stats1; A.g1 = p[kPG1]; A.b1 = p[kPB1]; A.packed = S.packed + l * train_packed_elems<D, F>();
            A.x1 = X.x1; A.d1 = X.d1; A.x = X.x; A.r3 = a.x;
            float *g = a.grads + l * G.total;
            products.add(X.dqkv, 3 * D, X.x1, D, 3 * D, D, g + G.qkv);
            products.add(X.d1, D, X.x, D, D, D, g + G.fo);
            products.reduce.cols[products.reduce.n_cols++] = {X.part_c + 5 * D + F, g + G.vec_a, groups, 7 * D + F, 2 * D};
        }
        if (l > 0) {
            const float *const *p = a.params + static_cast<size_t>(l - 1) * kParams;
            const SavedLayer v = S.layer(a, l - 1);
            A.r3 = v.r3; A.stats3 = v.stats3; A.g3 = p[kPG3]; A.b3 = p[kPB3]; A.r2 = v.r2; A.stats2 = v.stats2; A.g2 = p[kPG2]; A.b2 = p[kPB2];
            A.bias1 = p[kPBias1]; A.back_packed = S.packed + (l - 1) * train_packed_elems<D, F>();
            A.d3 = X.d3; A.x2 = X.x2; A.h = X.h; A.du = X.du; A.d2 = X.d2; A.dattn = X.dattn;
            float *g = a.grads + (l - 1) * G.total;
            products.add(X.d2, D, v.attn, D, D, D, g + G.o);
            products.add(X.du, F, X.x2, D, F, D, g + G.w1);
            products.add(X.d3, D, X.h, F, D, F, g + G.w2);
            products.reduce.cols[products.reduce.n_cols++] = {X.part_c, g + G.vec_b, groups, 7 * D + F, 5 * D + F};
        }
        if (l == a.n_layers)
            hipLaunchKernelGGL((train_backward_kernel<D, F, false, true>), dim3(groups), block, 0, st, A);
        else if (l == 0)
            hipLaunchKernelGGL((train_backward_kernel<D, F, true, false>), dim3(groups), block, 0, st, A);
        else
            hipLaunchKernelGGL((train_backward_kernel<D, F, true, true>), dim3(groups), block, 0, st, A);
        products.launch(st);
    }
    for (int l0 = 0; l0 < a.n_layers; l0 += kTrainPackLayers) {
        const unsigned n = static_cast<unsigned>(a.n_layers - l0 < kTrainPackLayers ? a.n_layers - l0 : kTrainPackLayers);
        hipLaunchKernelGGL((train_unfold_kernel<D>), dim3(2 * (D / 16), n), dim3(D), 0, st, weights(a, l0), a.grads + l0 * G.total, G.total,
                           G.fo, G.out, G.v);
    }
    return hipGetLastError() == hipSuccess ? ARTAB_OK : ARTAB_ERR_LAUNCH;
}

bool supported(const artab_train_args *a) {
    if (!a || a->B < 1 || a->R < 1 || a->H < 1 || a->n_layers < 1) return false;
    if ((a->D != 128 && a->D != 256) || a->F != 256 || a->D % a->H) return false;
    const int Dh = a->D / a->H;
    if (Dh != 32 && Dh != 64) return false;
    return a->context_len >= 1 && a->buffer_len >= 0 && a->context_len + a->buffer_len <= a->R && a->attending_chunks >= 0 &&
           a->first_row >= 0 && a->first_row < a->R && static_cast<int64_t>(a->B) * a->R < (1 << 30);
}

// The kernels read and write 16-byte pieces.
template <typename... P>
bool off_16(P... p) {
    return ((reinterpret_cast<uintptr_t>(p) % 16 != 0) || ...);
}
int check_parameters(const artab_train_args *a) {
    const void *const *p = reinterpret_cast<const void *const *>(a->params);
    for (int i = 0; i < 16 * a->n_layers; ++i) {
        if (!p[i]) return ARTAB_ERR_NULL_POINTER;
        if (off_16(p[i])) return ARTAB_ERR_BAD_STRIDE;
    }
    return off_16(a->x, a->saved, a->norm_gamma, a->norm_beta) ? ARTAB_ERR_BAD_STRIDE : ARTAB_OK;
}

constexpr int kEmbedSlices = 8;

bool embed_supported(const artab_train_embed_args *a) {
    return a && a->B >= 1 && (a->D == 128 || a->D == 256) && a->feat >= 1 && a->n_context >= 1 && a->n_buffer >= 0 && a->n_target >= 1 &&
           static_cast<int64_t>(a->B) * (a->n_context + a->n_buffer + a->n_target) < (1 << 30);
}

template <int D>
int embed(const artab_train_embed_args &a, hipStream_t st) {
    TrainEmbed P{};
    P.x[0] = a.x_context; P.x[1] = a.x_buffer; P.x[2] = a.x_target; P.y[0] = a.y_context; P.y[1] = a.y_buffer;
    P.n[0] = a.n_context; P.n[1] = a.n_buffer; P.n[2] = a.n_target; P.feat = a.feat;
    P.w_x = a.w_x; P.b_x = a.b_x; P.w_y = a.w_y; P.b_y = a.b_y; P.markers = a.markers; P.tokens = a.tokens;
    P.out = a.out; P.xy = reinterpret_cast<float2 *>(a.xy); P.B = a.B; P.R = a.n_context + a.n_buffer + a.n_target;
    const long n = static_cast<long>(P.B) * P.R * (D / 4);
    hipLaunchKernelGGL((train_embed_kernel<D>), dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st, P);
    return hipGetLastError() == hipSuccess ? ARTAB_OK : ARTAB_ERR_LAUNCH;
}

template <int D>
int embed_backward(const artab_train_embed_args &a, hipStream_t st) {
    TrainEmbedBackward P{};
    P.dx = a.out; P.xy = reinterpret_cast<const float2 *>(a.xy); P.B = a.B; P.R = a.n_context + a.n_buffer + a.n_target;
    P.n_ctx = a.n_context; P.n_buf = a.n_buffer; P.slices = kEmbedSlices;
    Arena s(a.scratch);
    P.part = s.take<float>(static_cast<size_t>(a.B) * kEmbedSlices * 5 * D);
    float *sums = s.take<float>(5 * D);
    P.d_tokens = a.grads + 7 * D;
    hipLaunchKernelGGL((train_embed_backward_kernel<D>), dim3(a.B > a.n_buffer ? a.B : a.n_buffer, kEmbedSlices + 1), dim3(256), 0, st, P);
    TrainReduce T{};
    T.cols[0] = {P.part, sums, a.B * kEmbedSlices, 5 * D, 5 * D};
    T.n_cols = 1;
    hipLaunchKernelGGL(train_reduce_kernel, dim3(5 * D / kTrainReduceCols), dim3(256), 0, st, T);
    hipLaunchKernelGGL(train_embed_finish_kernel, dim3(1), dim3(D), 0, st, sums, a.grads, D);
    return hipGetLastError() == hipSuccess ? ARTAB_OK : ARTAB_ERR_LAUNCH;
}

// ---- the head

bool head_supported(const artab_train_head_args *a) {
    return a && a->rows >= 1 && a->rows < (1 << 30) && (a->D == 128 || a->D == 256) && a->F == 256 && a->K >= 1 && 3 * a->K <= kHeadCols;
}
int head_cols(const artab_train_head_args &a) { return 3 * a.K <= 64 ? 64 : 128; }
int head_groups(long M) {  // as many workgroups as are resident (three to a compute unit), or fewer
    const long tiles = (M + kTrainRows - 1) / kTrainRows;
    return static_cast<int>(tiles < 768 ? tiles : 768);
}
int head_jobs(const artab_train_head_args &a) { return (a.F / 128) * (a.D / 128) + a.F / 128; }

struct HeadSaved {
    float *y;  // a copy: the caller's may change before the backward pass, as under modules
    bf16_t *packed;
    float *part_loss;
    size_t bytes;
};
HeadSaved head_saved(const artab_train_head_args &a) {
    Arena s(a.saved);
    HeadSaved v;
    v.y = s.take<float>(a.rows);
    v.packed = s.take<bf16_t>(2 * static_cast<size_t>(a.F) * (a.D + head_cols(a)));
    v.part_loss = s.take<float>(head_groups(a.rows));
    v.bytes = s.used;
    return v;
}
struct HeadScratch {
    bf16_t *zb, *h, *du, *draw;
    float *part, *part_w;
    size_t bytes;
};
HeadScratch head_scratch(const artab_train_head_args &a) {
    Arena s(a.scratch);
    HeadScratch v;
    const size_t M = a.rows;
    const int jobs = head_jobs(a);
    v.zb = s.take<bf16_t>(M * a.D);
    v.h = s.take<bf16_t>(M * a.F);
    v.du = s.take<bf16_t>(M * a.F);
    v.draw = s.take<bf16_t>(M * kHeadCols);
    v.part = s.take<float>(static_cast<size_t>(head_groups(a.rows)) * (a.F + kHeadCols));
    v.part_w = s.take<float>(static_cast<size_t>(grad_slices(M, jobs)) * jobs * 16384);
    v.bytes = s.used;
    return v;
}

TrainHead head_params(const artab_train_head_args &a) {
    TrainHead P{};
    P.z = a.z; P.w1 = a.w1; P.b1 = a.b1; P.w2 = a.w2; P.b2 = a.b2;
    P.mean_bias = a.mean_bias; P.std_bias = a.std_bias; P.weight_bias = a.weight_bias; P.std_min = a.std_min; P.K = a.K; P.M = a.rows;
    const HeadSaved S = head_saved(a);
    P.packed = S.packed; P.part_loss = S.part_loss; P.kept_y = S.y;
    return P;
}

template <int D, int NP>
int head_forward(const artab_train_head_args &a, hipStream_t st) {
    constexpr int F = 256;
    TrainHead P = head_params(a);
    P.y = a.y;
    const int groups = head_groups(a.rows);
    hipLaunchKernelGGL((train_head_pack_kernel<D, F, NP>), dim3(static_cast<unsigned>((train_head_packed_elems<D, F, NP>() / 8 + 255) / 256)),
                       dim3(256), 0, st, P);
    hipLaunchKernelGGL((train_head_kernel<D, F, NP, false>), dim3(groups), dim3(kTrainWaves * 64), 0, st, P);
    hipLaunchKernelGGL(train_head_loss_kernel, dim3(1), dim3(256), 0, st, P.part_loss, groups, P.M, a.loss);
    return hipGetLastError() == hipSuccess ? ARTAB_OK : ARTAB_ERR_LAUNCH;
}
template <int D, int NP>
int head_backward(const artab_train_head_args &a, hipStream_t st) {
    constexpr int F = 256;
    TrainHead P = head_params(a);
    const HeadScratch X = head_scratch(a);
    const int groups = head_groups(a.rows), jobs = head_jobs(a), slices = grad_slices(P.M, jobs);
    P.dloss = a.dloss; P.dz = a.dz; P.zb = X.zb; P.h = X.h; P.du = X.du; P.draw = X.draw; P.part = X.part;
    hipLaunchKernelGGL((train_head_kernel<D, F, NP, true>), dim3(groups), dim3(kTrainWaves * 64), 0, st, P);
    GradProducts products(P.M, slices, X.part_w);
    products.add(X.du, F, X.zb, D, F, D, a.grads);
    products.add(X.draw, kHeadCols, X.h, F, kHeadCols, F, a.grads + static_cast<long>(F) * D);
    products.reduce.cols[products.reduce.n_cols++] = {X.part, a.grads + static_cast<long>(F) * (D + kHeadCols), groups, F + kHeadCols, F + kHeadCols};
    products.launch(st);
    return hipGetLastError() == hipSuccess ? ARTAB_OK : ARTAB_ERR_LAUNCH;
}

}  // namespace
}  // namespace artab

extern "C" {

size_t artab_train_embed_scratch_bytes(const artab_train_embed_args *a) {
    if (!artab::embed_supported(a)) return 0;
    artab::Arena s(nullptr);
    s.take<float>(static_cast<size_t>(a->B) * artab::kEmbedSlices * 5 * a->D);
    s.take<float>(5 * a->D);
    return s.used;
}
int artab_train_embed(const artab_train_embed_args *a, void *stream) {
    if (!artab::embed_supported(a)) return ARTAB_ERR_UNSUPPORTED;
    if (!a->x_context || !a->y_context || (a->n_buffer && (!a->x_buffer || !a->y_buffer || !a->tokens)) || !a->x_target || !a->w_x || !a->b_x ||
        !a->w_y || !a->b_y || !a->markers || !a->out || !a->xy)
        return ARTAB_ERR_NULL_POINTER;
    if (artab::off_16(a->w_x, a->b_x, a->w_y, a->b_y, a->markers, a->tokens, a->out, a->xy)) return ARTAB_ERR_BAD_STRIDE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return a->D == 128 ? artab::embed<128>(*a, st) : artab::embed<256>(*a, st);
}
int artab_train_embed_backward(const artab_train_embed_args *a, void *stream) {
    if (!artab::embed_supported(a)) return ARTAB_ERR_UNSUPPORTED;
    if (!a->out || !a->xy || !a->grads || !a->scratch) return ARTAB_ERR_NULL_POINTER;
    if (artab::off_16(a->out, a->xy, a->grads, a->scratch)) return ARTAB_ERR_BAD_STRIDE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return a->D == 128 ? artab::embed_backward<128>(*a, st) : artab::embed_backward<256>(*a, st);
}

size_t artab_train_head_saved_bytes(const artab_train_head_args *a) {
    if (!artab::head_supported(a)) return 0;
    artab_train_head_args b = *a;
    b.saved = nullptr;
    return artab::head_saved(b).bytes;
}
size_t artab_train_head_scratch_bytes(const artab_train_head_args *a) {
    if (!artab::head_supported(a)) return 0;
    artab_train_head_args b = *a;
    b.scratch = nullptr;
    return artab::head_scratch(b).bytes;
}
int artab_train_head_forward(const artab_train_head_args *a, void *stream) {
    if (!artab::head_supported(a)) return ARTAB_ERR_UNSUPPORTED;
    if (!a->z || !a->y || !a->w1 || !a->b1 || !a->w2 || !a->b2 || !a->mean_bias || !a->std_bias || !a->weight_bias || !a->saved || !a->loss)
        return ARTAB_ERR_NULL_POINTER;
    if (artab::off_16(a->z, a->w1, a->b1, a->w2, a->saved)) return ARTAB_ERR_BAD_STRIDE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool narrow = artab::head_cols(*a) == 64;
    if (a->D == 128) return narrow ? artab::head_forward<128, 64>(*a, st) : artab::head_forward<128, 128>(*a, st);
    return narrow ? artab::head_forward<256, 64>(*a, st) : artab::head_forward<256, 128>(*a, st);
}
int artab_train_head_backward(const artab_train_head_args *a, void *stream) {
    if (!artab::head_supported(a)) return ARTAB_ERR_UNSUPPORTED;
    if (!a->z || !a->w1 || !a->b1 || !a->w2 || !a->b2 || !a->mean_bias || !a->std_bias || !a->weight_bias || !a->saved || !a->dloss ||
        !a->dz || !a->grads || !a->scratch)
        return ARTAB_ERR_NULL_POINTER;
    if (artab::off_16(a->z, a->w1, a->b1, a->w2, a->saved, a->dz, a->grads, a->scratch)) return ARTAB_ERR_BAD_STRIDE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool narrow = artab::head_cols(*a) == 64;
    if (a->D == 128) return narrow ? artab::head_backward<128, 64>(*a, st) : artab::head_backward<128, 128>(*a, st);
    return narrow ? artab::head_backward<256, 64>(*a, st) : artab::head_backward<256, 128>(*a, st);
}

size_t artab_train_saved_bytes(const artab_train_args *a) {
    if (!artab::supported(a)) return 0;
    artab_train_args b = *a;
    b.saved = nullptr;
    return artab::saved_layout(b).bytes;
}
size_t artab_train_scratch_bytes(const artab_train_args *a) {
    if (!artab::supported(a)) return 0;
    artab_train_args b = *a;
    b.scratch = nullptr;
    return artab::scratch_layout(b).bytes;
}
int artab_train_forward(const artab_train_args *a, void *stream) {
    if (!artab::supported(a)) return ARTAB_ERR_UNSUPPORTED;
    if (!a->x || !a->params || !a->saved || !a->z || !a->norm_gamma || !a->norm_beta) return ARTAB_ERR_NULL_POINTER;
    const int rc = artab::off_16(a->z) ? ARTAB_ERR_BAD_STRIDE : artab::check_parameters(a);
    if (rc != ARTAB_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return a->D == 128 ? artab::forward<128, 256>(*a, st) : artab::forward<256, 256>(*a, st);
}
int artab_train_backward(const artab_train_args *a, void *stream) {
    if (!artab::supported(a)) return ARTAB_ERR_UNSUPPORTED;
    if (!a->x || !a->params || !a->saved || !a->dz || !a->dx || !a->grads || !a->scratch || !a->norm_gamma || !a->norm_beta)
        return ARTAB_ERR_NULL_POINTER;
    const int rc = artab::off_16(a->dz, a->dx, a->grads, a->scratch) ? ARTAB_ERR_BAD_STRIDE : artab::check_parameters(a);
    if (rc != ARTAB_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return a->D == 128 ? artab::backward<128, 256>(*a, st) : artab::backward<256, 256>(*a, st);
}

}  // extern "C"
