// Batched elementwise optimizer steps: Grokfast (EMA filter + amplification,
// optionally fused with its AdamW update) and SuperGrok v1.5 (device-side
// global-norm clip, mu EMA, 2->H->1 sharpness meta-net, Adam, progressive
// weight decay; SAM perturb / sharpness restore helpers).
//
// Every entry point covers all tensors with one launch per stage: a tile of
// elements is mapped to (tensor, offset) by a search in a prefix table, so
// small parameter sets cost one or two launches instead of several per tensor
// (the reference launches per tensor and syncs the host for the gradient norm).
#include "sg_elemwise.hpp"

namespace sgew {
namespace {

// ---- Grokfast (aux: ema) -------------------------------------------------------
// HBM bound (40 B an element in fp32): four elements per lane and access.
template <bool ADAM, class BT>
__global__ __launch_bounds__(THREADS) void k_grokfast(BT B, float alpha, float lamb, float beta1, float om_beta1, float beta2,
                                                       float om_beta2, float eps, float decay) {
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    const float om_alpha = 1.0f - alpha;
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float g[V], e[V];
        ldt<V>(R.grad, R.dtype, i, g);
        ldf<V>(R.aux, i, e);
#pragma unroll
        for (int c = 0; c < V; c++) {
            e[c] = sg_fma(alpha, e[c], om_alpha * g[c]);
            g[c] = sg::round_to(R.dtype, sg_fma(lamb, e[c], g[c]));       // AdamW consumes the gradient as stored
        }
        stf<V>(R.aux, i, e);
        stt<V>(R.grad, R.dtype, i, g);
        if (ADAM) adam_update<V>(R, i, g, beta1, om_beta1, beta2, om_beta2, eps, decay);
    });
}

// ---- SuperGrok v1.5 (aux: mu, aux2: sharpness) -----------------------------------
template <int GELU, class BT>
__global__ __launch_bounds__(THREADS) void k_sg15(BT B, const float* __restrict__ W1, const float* __restrict__ b1,
                                                   const float* __restrict__ W2, const float* __restrict__ b2, int H,
                                                   float clip_norm, float rescale, float lamb_eff, float beta2, float eps, float decay) {
    __shared__ float sW1[2 * MAX_HIDDEN], sb1[MAX_HIDDEN], sW2[MAX_HIDDEN];
    load_net(W1, b1, W2, H, sW1, sb1, sW2);
    const Clip clip = global_norm(B, clip_norm);        // (its barriers cover the weights)
    const MetaNet<GELU> net = {sW1, sb1, sW2, b2[0], H, (const __attribute__((address_space(4))) MetaPoly*)B.table};

    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    const float alpha = R.alpha, beta1 = R.beta1;
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float g[V], s[V], mu[V];
        clipped_grad<V>(R, i, clip, g);
        ldsharp<V>(R, i, s);
        ldf<V>(R.aux, i, mu);
#pragma unroll
        for (int c = 0; c < V; c++) mu[c] = sg_fma(alpha, mu[c], (1.0f - alpha) * g[c]);
        stf<V>(R.aux, i, mu);
#pragma unroll
        for (int c = 0; c < V; c++) g[c] = sg_fma(lamb_eff, mu[c], sg_fma(rescale, net(g[c], s[c]), g[c]));
        adam_update<V>(R, i, g, beta1, 1.0f - beta1, beta2, 1.0f - beta2, eps, decay);
    });
}

template <class BT>
__global__ __launch_bounds__(THREADS) void k_sam_perturb(BT B, float rho) {
    const Clip n = global_norm(B, 0.0f);
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    const float r = rho / (n.norm + 1e-12f);
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float p[V], g[V];
        ldt<V>(R.param, R.dtype, i, p);
        ldt<V>(R.grad, R.dtype, i, g);
#pragma unroll
        for (int c = 0; c < V; c++) p[c] = sg_fma(r, g[c], p[c]);
        stt<V>(R.param, R.dtype, i, p);
    });
}

// grad: the normal gradient, aux2: the SAM gradient, ea: sharpness, easq: backup (both in the tensor's type)
template <class BT>
__global__ __launch_bounds__(THREADS) void k_restore(BT B) {
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float a[V], b[V], p[V];
        ldt<V>(R.aux2, R.dtype, i, a);
        ldt<V>(R.grad, R.dtype, i, b);
        ldt<V>(R.easq, R.dtype, i, p);
#pragma unroll
        for (int c = 0; c < V; c++) a[c] = sg_abs(a[c] - b[c]);
        stt<V>(R.ea, R.dtype, i, a);
        stt<V>(R.param, R.dtype, i, p);
    });
}

}  // namespace
}  // namespace sgew

extern "C" {

size_t sg_elemwise_workspace_bytes(int num_tensors, const int64_t* numels) {
    if (num_tensors < 0 || (num_tensors > 0 && !numels)) return 0;
    sgew::Layout L;
    if (sgew::make_layout(num_tensors, numels, &L)) return 0;
    return L.bytes;
}

int sg_grokfast_ema(int num_tensors, const SgGrokfastTensor* tensors, float alpha, float lamb, void* workspace,
                    size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    if (!tensors) return sg::fail("NULL argument");
    std::vector<Rec> recs;
    recs.reserve(num_tensors);
    for (int i = 0; i < num_tensors; i++) {
        const SgGrokfastTensor& t = tensors[i];
        if (t.numel == 0) continue;
        if (!t.grad || !t.ema) return sg::fail("tensor %d: NULL pointer", i);
        if (check_dtype(i, t.dtype) || check_numel(i, t.numel)) return 1;
        recs.push_back({nullptr, t.grad, nullptr, nullptr, t.ema, nullptr, (int32_t)t.numel, (int16_t)t.dtype,
                        vec4_ok(t.dtype, bits(t.grad), bits(t.ema)), 0, 0.0f, 1.0f, 0.0f, 0.0f});
    }
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, false, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        hipLaunchKernelGGL((k_grokfast<false, BT>), dim3(B.tiles), dim3(THREADS), 0, st, B, alpha, lamb, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f);
        SG_LAUNCH_CHECK("k_grokfast<ema>");
        return 0;
    });
}

int sg_grokfast_adamw_step(int num_tensors, const SgGrokfastAdamTensor* tensors, float alpha, float lamb, double lr,
                           double beta1, double beta2, double eps, double weight_decay, void* workspace,
                           size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    if (!tensors) return sg::fail("NULL argument");
    std::vector<Rec> recs;
    recs.reserve(num_tensors);
    int last_step = 0;
    double bc1 = 1.0, bc2 = 1.0;
    for (int i = 0; i < num_tensors; i++) {
        const SgGrokfastAdamTensor& t = tensors[i];
        if (t.numel == 0) continue;
        if (!t.param || !t.grad || !t.ema || !t.exp_avg || !t.exp_avg_sq) return sg::fail("tensor %d: NULL pointer", i);
        if (check_dtype(i, t.dtype) || check_numel(i, t.numel)) return 1;
        if (t.step < 1) return sg::fail("tensor %d: step must be >= 1", i);
        // bias corrections in double, as the Python helper computes them (tensors of a group are nearly always at one step)
        if (t.step != last_step) {
            bc1 = 1.0 - std::pow(beta1, (double)t.step);
            bc2 = 1.0 - std::pow(beta2, (double)t.step);
            last_step = t.step;
        }
        recs.push_back({t.param, t.grad, t.exp_avg, t.exp_avg_sq, t.ema, nullptr, (int32_t)t.numel, (int16_t)t.dtype,
                        vec4_ok(t.dtype, bits(t.param) | bits(t.grad), bits(t.ema) | bits(t.exp_avg) | bits(t.exp_avg_sq)), 0,
                        (float)(lr / bc1), (float)bc2, 0.0f, 0.0f});
    }
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, false, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        hipLaunchKernelGGL((k_grokfast<true, BT>), dim3(B.tiles), dim3(THREADS), 0, st, B, alpha, lamb, (float)beta1,
                           (float)(1.0 - beta1), (float)beta2, (float)(1.0 - beta2), (float)eps, (float)(1.0 - lr * weight_decay));
        SG_LAUNCH_CHECK("k_grokfast<adamw>");
        return 0;
    });
}

int sg15_fused_step(int num_tensors, const Sg15Tensor* tensors, const Sg15Net* net, float lamb_eff, float beta2, float lr,
                    float wd_eff, float eps, float grad_clip_norm, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    if (!tensors || !net || !net->W1 || !net->b1 || !net->W2 || !net->b2) return sg::fail("NULL argument");
    if (net->hidden < 1 || net->hidden > MAX_HIDDEN) return sg::fail("hidden_dim %d outside [1,%d]", net->hidden, MAX_HIDDEN);
    if (net->gelu_mode != 0 && net->gelu_mode != 1) return sg::fail("bad gelu_mode %d", net->gelu_mode);
    std::vector<Rec> recs;
    recs.reserve(num_tensors);
    for (int i = 0; i < num_tensors; i++) {
        const Sg15Tensor& t = tensors[i];
        if (t.numel == 0) continue;
        if (!t.param || !t.grad || !t.sharpness || !t.exp_avg || !t.exp_avg_sq || !t.mu) return sg::fail("tensor %d: NULL pointer", i);
        const int dtype = t.dtype & ~SG_SHARP_F32;
        const bool s32 = t.dtype != dtype;
        if (check_dtype(i, dtype) || check_numel(i, t.numel)) return 1;
        recs.push_back({t.param, t.grad, t.exp_avg, t.exp_avg_sq, t.mu, t.sharpness, (int32_t)t.numel, (int16_t)dtype,
                        vec4_ok(dtype, bits(t.param) | bits(t.grad) | (s32 ? 0 : bits(t.sharpness)),
                                bits(t.exp_avg) | bits(t.exp_avg_sq) | bits(t.mu) | (s32 ? bits(t.sharpness) : 0)), (int8_t)s32,
                        lr / t.bc1, t.bc2, t.alpha, t.beta1});
    }
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, true, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        const float decay = 1.0f - lr * wd_eff;
        const auto run = [&](auto gelu) {
            hipLaunchKernelGGL((k_sg15<decltype(gelu)::value, BT>), dim3(B.tiles), dim3(THREADS), 0, st, B, net->W1, net->b1, net->W2,
                               net->b2, net->hidden, grad_clip_norm, net->rescale, lamb_eff, beta2, eps, decay);
        };
        if (net->gelu_mode == 0) {
            launch_sumsq(B, st, PrepMetaPoly{net->W1, net->b1, net->W2, net->b2, net->hidden});
            run(std::integral_constant<int, 0>{});
        } else {
            launch_sumsq(B, st);
            run(std::integral_constant<int, 1>{});
        }
        SG_LAUNCH_CHECK("k_sg15");
        return 0;
    });
}

int sg15_sam_perturb(int num_tensors, const Sg15SamTensor* tensors, float rho, void* workspace, size_t workspace_bytes,
                     void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    if (!tensors) return sg::fail("NULL argument");
    std::vector<Rec> recs;
    recs.reserve(num_tensors);
    for (int i = 0; i < num_tensors; i++) {
        const Sg15SamTensor& t = tensors[i];
        if (t.numel == 0) continue;
        if (!t.param || !t.grad) return sg::fail("tensor %d: NULL pointer", i);
        if (check_dtype(i, t.dtype) || check_numel(i, t.numel)) return 1;
        recs.push_back({t.param, const_cast<void*>(t.grad), nullptr, nullptr, nullptr, nullptr, (int32_t)t.numel, (int16_t)t.dtype,
                        vec4_ok(t.dtype, bits(t.param) | bits(t.grad), 0), 0, 0.0f, 1.0f, 0.0f, 0.0f});
    }
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, true, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        launch_sumsq(B, st);
        hipLaunchKernelGGL(k_sam_perturb<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B, rho);
        SG_LAUNCH_CHECK("k_sam_perturb");
        return 0;
    });
}

int sg15_sharpness_restore(int num_tensors, const Sg15RestoreTensor* tensors, void* workspace, size_t workspace_bytes,
                           void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    if (!tensors) return sg::fail("NULL argument");
    std::vector<Rec> recs;
    recs.reserve(num_tensors);
    for (int i = 0; i < num_tensors; i++) {
        const Sg15RestoreTensor& t = tensors[i];
        if (t.numel == 0) continue;
        if (!t.param || !t.sharpness || !t.backup || !t.sam_grad || !t.normal_grad) return sg::fail("tensor %d: NULL pointer", i);
        if (check_dtype(i, t.dtype) || check_numel(i, t.numel)) return 1;
        recs.push_back({t.param, const_cast<void*>(t.normal_grad), static_cast<float*>(t.sharpness),
                        static_cast<float*>(const_cast<void*>(t.backup)), nullptr, t.sam_grad, (int32_t)t.numel, (int16_t)t.dtype,
                        vec4_ok(t.dtype, bits(t.param) | bits(t.sharpness) | bits(t.backup) | bits(t.sam_grad) | bits(t.normal_grad), 0), 0,
                        0.0f, 1.0f, 0.0f, 0.0f});
    }
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, false, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        hipLaunchKernelGGL(k_restore<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B);
        SG_LAUNCH_CHECK("k_restore");
        return 0;
    });
}

}  // extern "C"
