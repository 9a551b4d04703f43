// The reference's remaining fused optimizer steps: GrokAdamW, NeuralGrok,
// Prodigy, Lion, SuperGrok v1.1 and the LookSAM helpers.  Replaces the bodies of
// grokadamw_fused_step, neuralgrok_fused_step, prodigy_fused_step,
// lion_fused_step, supergrok11_fused_step and looksam_* of the reference's
// csrc/ops.cpp:209-656 with their per-optimizer kernels.
//
// Same batching as the other elementwise steps: one launch per stage covers
// every tensor.  Everything the reference reads back to the host between stages -
// the global gradient norm, Prodigy's numerator/denominator, v1.1's cosine
// gate per tensor, LookSAM's per-tensor norms - is reduced on the device
// (partial sums in double, added up in a fixed order by the consumer) so a
// step enqueues without a host sync.
#include <mutex>

#include "sg_elemwise.hpp"

namespace sgew {
namespace {

// ---- GrokAdamW (aux: ema, or NULL for plain AdamW) -------------------------------
template <class BT>
__global__ __launch_bounds__(THREADS) void k_grokadamw(BT B, float clip_norm, float alpha, float lamb, float beta1, float beta2,
                                                        float eps, float decay) {
    Clip clip = {0.0f, 1.0f, false};
    if (clip_norm > 0.0f) clip = global_norm(B, clip_norm);
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float g[V];
        clipped_grad<V>(R, i, clip, g);
        if (R.aux) {
            float e[V];
            ldf<V>(R.aux, i, e);
#pragma unroll
            for (int c = 0; c < V; c++) {
                e[c] = sg_fma(alpha, e[c], (1.0f - alpha) * g[c]);
                g[c] = sg_fma(lamb, e[c], g[c]);
            }
            stf<V>(R.aux, i, e);
        }
        adam_update<V>(R, i, g, beta1, 1.0f - beta1, beta2, 1.0f - beta2, eps, decay);
    });
}

// ---- NeuralGrok ------------------------------------------------------------------
// The amplifier  sum_h W2 relu(W1 g + b1)  is a straight line  A g + B  between two neighbouring thresholds -b1/W1 of
// its units.  One block tabulates the lines of all H + 1 intervals per call (in double, while the other blocks of its
// launch reduce the gradient norm); an element finds its interval by a search of the thresholds in LDS and evaluates
// one fma.  Evaluating the units one by one is 3 vector instructions and LDS operands for each of 128 units: 332 us
// for 25 M elements against 140 us for the step's memory traffic.
// Error: A and B are rounded once, so the amplifier is within 2^-24 (|A g| + |B| + |A g + B|).  Close to a far threshold the
// first two cancel and a unit-by-unit sum, which rounds only what is left of them, can be closer there; over module-made
// weights (128 units) and gradients of deviation 1e-3, 1 and 1000 the largest error against float64 is 6e-9, 4e-8 and 4e-5, unit
// by unit 9e-8, 2e-7 and 2e-4.
constexpr int AMP_SLOTS = 511;         // thresholds, padded with +inf to 2^k - 1 (at most MAX_HIDDEN = 256 real ones)
struct AmpTable {
    float t[AMP_SLOTS + 1];
    float A[MAX_HIDDEN + 1], B[MAX_HIDDEN + 1];
    float lo, hi;                      // the interval of small gradients: lo < g <= hi
    int at, direct;                    // its index; direct: non-finite weights, no table
};
static_assert(sizeof(AmpTable) <= TABLE_BYTES, "table fits its place in the workspace");
inline int amp_slots(int H) {          // smallest 2^k - 1 >= H
    int s = 1;
    while (s < H) s = 2 * s + 1;
    return s;
}
// The table's block works while the others read the gradients, and in a small call they wait for it.  One lane per unit:
// its rank is a count over all thresholds (four per LDS read), and the line of the interval below rank k is the units
// that rise below it plus those that fall above it, a running sum from either end.  Both are sums of the active
// units alone, never a difference, in double.  Adding up the H units of each interval by itself was a chain of 128
// terms: the launch took 29.7 us over 0.42 M gradients and 31.9 us over 25 M; now 7.1
// and 19.6 us (6.5 and 20.4 without a table).
struct PrepAmp {
    static constexpr bool any = true;
    const float *W1, *b1, *W2;
    int H, slots;
    template <class BT>
    __device__ void operator()(const BT& B) const {
        static_assert(MAX_HIDDEN == THREADS, "one lane per unit");
        constexpr int WAVES = THREADS / 64;
        __shared__ float4 st[MAX_HIDDEN / 4];
        __shared__ float sorted[MAX_HIDDEN], sw1[MAX_HIDDEN], sb1[MAX_HIDDEN], sw2[MAX_HIDDEN];
        __shared__ double tot[WAVES][4];
        AmpTable* out = static_cast<AmpTable*>(B.table);
        const int h = threadIdx.x, lane = h & 63, wave = h >> 6;
        float w = 0.0f, b = 0.0f, u = 0.0f, t = __builtin_inff();
        bool bad = false;
        if (h < H) {
            w = W1[h];
            b = b1[h];
            u = W2[h];
            t = w == 0.0f ? __builtin_inff() : -b / w;           // a unit that does not look at g has no threshold
            bad = !sg_isfinite(w) || !sg_isfinite(b) || !sg_isfinite(u);
        }
        reinterpret_cast<float*>(st)[h] = t;                     // (+inf past H)
        bad = __syncthreads_or(bad ? 1 : 0) != 0;
        int r = h;                                               // the lanes past H stay where they are
        if (h < H) {
            r = 0;
#pragma unroll 4
            for (int k = 0; k < H; k += 4) {
                const float4 o = st[k / 4];
                r += (o.x < t || (o.x == t && k < h)) ? 1 : 0;
                r += (o.y < t || (o.y == t && k + 1 < h)) ? 1 : 0;
                r += (o.z < t || (o.z == t && k + 2 < h)) ? 1 : 0;
                r += (o.w < t || (o.w == t && k + 3 < h)) ? 1 : 0;
            }
        }
        r &= MAX_HIDDEN - 1;                                     // (in range whatever the weights)
        sorted[r] = t;
        sw1[r] = w;
        sb1[r] = b;
        sw2[r] = u;
        const int at = __syncthreads_count(t < 0.0f ? 1 : 0);
        for (int k = h; k < slots; k += THREADS) out->t[k] = k < H ? sorted[k] : __builtin_inff();
        // From here on lane h holds the unit of rank h.  A unit with w = 0 and b > 0 is always active: its threshold +inf
        // puts it above every interval that a finite gradient reaches, with those that fall.
        w = sw1[h];
        b = sb1[h];
        u = sw2[h];
        const double ua = (double)u * (double)w, uc = (double)u * (double)b;
        const bool rises = w > 0.0f, falls = w < 0.0f || (w == 0.0f && b > 0.0f);
        double ra = rises ? ua : 0.0, rc = rises ? uc : 0.0, fa = falls ? ua : 0.0, fc = falls ? uc : 0.0;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const double xa = __shfl_up(ra, d), xc = __shfl_up(rc, d), ya = __shfl_down(fa, d), yc = __shfl_down(fc, d);
            if (lane >= d) { ra += xa; rc += xc; }
            if (lane + d < 64) { fa += ya; fc += yc; }
        }
        if (lane == 63) { tot[wave][0] = ra; tot[wave][1] = rc; }
        if (lane == 0) { tot[wave][2] = fa; tot[wave][3] = fc; }
        __syncthreads();
        double pa = 0.0, pc = 0.0;                               // the waves below this one
        for (int v = 0; v < WAVES; v++) {
            if (v < wave) { pa += tot[v][0]; pc += tot[v][1]; }
            if (v > wave) { fa += tot[v][2]; fc += tot[v][3]; }
        }
        const double ea = __shfl_up(ra, 1), ec = __shfl_up(rc, 1);
        const double la = pa + (lane > 0 ? ea : 0.0), lc = pc + (lane > 0 ? ec : 0.0);
        if (h < H) {                                             // interval h: thresholds 0 .. h-1 lie below g
            out->A[h] = (float)(la + fa);
            out->B[h] = (float)(lc + fc);
        }
        if (h == H - 1) {
            out->A[H] = (float)(pa + ra);
            out->B[H] = (float)(pc + rc);
        }
        if (h == 0) {
            out->at = at;
            out->lo = at > 0 ? sorted[at - 1] : -__builtin_inff();
            out->hi = at < H ? sorted[at] : __builtin_inff();
            out->direct = bad ? 1 : 0;
        }
    }
};

template <class BT>
__global__ __launch_bounds__(THREADS) void k_neuralgrok(BT B, const float* __restrict__ W1, const float* __restrict__ b1,
                                                         const float* __restrict__ W2, const float* __restrict__ b2, int H, int slots,
                                                         float clip_norm, float alpha_amp, float beta_amp, float beta1, float beta2,
                                                         float eps, float decay) {
    __shared__ float st[AMP_SLOTS + 1], sA[MAX_HIDDEN + 1], sB[MAX_HIDDEN + 1];
    const AmpTable* T = static_cast<const AmpTable*>(B.table);
    for (int k = threadIdx.x; k < slots; k += THREADS) st[k] = T->t[k];
    for (int k = threadIdx.x; k <= H; k += THREADS) { sA[k] = T->A[k]; sB[k] = T->B[k]; }
    const Clip clip = global_norm(B, clip_norm);                 // (its barriers cover the table)
    const float lo = T->lo, hi = T->hi, A0 = T->A[T->at], B0 = T->B[T->at];
    const bool direct = T->direct != 0;
    const float bias2 = b2[0];
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    const auto amplifier = [&](float g) {
        if (direct || !sg_isfinite(g)) {                         // unit by unit, as written
            float acc = 0.0f;
            for (int h = 0; h < H; h++) acc = sg_fma(W2[h], sg_max(sg_fma(W1[h], g, b1[h]), 0.0f), acc);
            return acc;
        }
        if (g > lo && g <= hi) return sg_fma(A0, g, B0);
        int pos = 0;
        for (int step = (slots + 1) >> 1; step > 0; step >>= 1)
            if (g > st[pos + step - 1]) pos += step;
        return sg_fma(sA[pos], g, sB[pos]);
    };
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float g[V];
        clipped_grad<V>(R, i, clip, g);
#pragma unroll
        for (int c = 0; c < V; c++) g[c] = g[c] * sg_fma(alpha_amp, amplifier(g[c]) + bias2, beta_amp);
        adam_update<V>(R, i, g, beta1, 1.0f - beta1, beta2, 1.0f - beta2, eps, decay);
    });
}

// ---- Lion ------------------------------------------------------------------------
template <class BT>
__global__ __launch_bounds__(THREADS) void k_lion(BT B, float lr, float beta1, float beta2, float wd) {
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float g[V], m[V], p[V];
        ldt<V>(R.grad, R.dtype, i, g);
        ldf<V>(R.ea, i, m);
        ldt<V>(R.param, R.dtype, i, p);
#pragma unroll
        for (int c = 0; c < V; c++) {
            const float interp = sg_fma(beta1, m[c], (1.0f - beta1) * g[c]);
            const float s = interp > 0.0f ? 1.0f : (interp < 0.0f ? -1.0f : 0.0f);
            p[c] = sg_fma(-lr, sg_fma(wd, p[c], s), p[c]);
            m[c] = sg_fma(beta2, m[c], (1.0f - beta2) * g[c]);
        }
        stt<V>(R.param, R.dtype, i, p);
        stf<V>(R.ea, i, m);
    });
}

// ---- Prodigy (aux: s, aux2: initial parameter, fp32) --------------------------------
template <class BT>
__global__ __launch_bounds__(THREADS) void k_prodigy_partial(BT B, int blocks) {
    double nsum = 0.0, dsum = 0.0;
    for (int tile = blockIdx.x; tile < B.tiles; tile += blocks) {
        int start, cnt;
        const Rec& R = tile_rec(B, tile, &start, &cnt);
        const float* p0 = static_cast<const float*>(R.aux2);
        float num = 0.0f, den = 0.0f;
        for_tile(R, start, cnt, [&](auto v, int i) {
            constexpr int V = decltype(v)::value;
            float g[V], p[V], q[V], sv[V];
            ldt<V>(R.grad, R.dtype, i, g);
            ldt<V>(R.param, R.dtype, i, p);
            ldf<V>(p0, i, q);
            ldf<V>(R.aux, i, sv);
#pragma unroll
            for (int c = 0; c < V; c++) {
                num = sg_fma(g[c], p[c] - q[c], num);
                den += sv[c];
            }
        });
        nsum += (double)num;
        dsum += (double)den;
    }
    tile_sums<2>(B, nsum, dsum);
}
// one block: the two sums and this call's d_lr, for the Adam kernel (table) and for the host (pinned, may be NULL)
template <class BT>
__global__ __launch_bounds__(THREADS) void k_prodigy_dlr(BT B, int blocks, float d_lr, float* host) {
    double s[2];
    add_tiles<2>(B, 0, blocks, s);
    if (threadIdx.x != 0) return;
    const float num = (float)s[0], den = (float)s[1];
    if (den > 1e-30f) d_lr = sg_max(d_lr, sg_abs(num) / (den + 1e-12f));
    *static_cast<float*>(B.table) = d_lr;
    if (host) __hip_atomic_store(host, d_lr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
template <class BT>
__global__ __launch_bounds__(THREADS) void k_prodigy(BT B, float beta1, float beta2, float lr, float wd, float eps) {
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    const float d_lr = *static_cast<const float*>(B.table);
    const float decay = 1.0f - (lr * d_lr) * wd, eps_eff = d_lr * eps;
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float dg[V], sv[V];
        ldt<V>(R.grad, R.dtype, i, dg);
        ldf<V>(R.aux, i, sv);
#pragma unroll
        for (int c = 0; c < V; c++) {
            dg[c] = d_lr * dg[c];
            sv[c] = sg_fma(beta2, sv[c], ((1.0f - beta2) * dg[c]) * dg[c]);
        }
        stf<V>(R.aux, i, sv);
        adam_update<V>(R, i, dg, beta1, 1.0f - beta1, beta2, 1.0f - beta2, eps_eff, decay);
    });
}

// What a call needs to hand d_lr back to the host: a word of pinned memory that the kernel writes and an event behind
// it, so that the host waits for the reduction alone while the update runs on.  A copy into the caller's pageable
// memory would wait for the whole step.  Slots are kept for later calls, at most MAX_SLOTS of them; a call takes one
// for itself, so threads and streams do not meet.
struct HostSlot {
    float* word = nullptr;
    hipEvent_t done = nullptr;
    int device = -1;
};
constexpr size_t MAX_SLOTS = 16;
std::mutex g_slot_mutex;
std::vector<HostSlot> g_slots;
void drop_slot(HostSlot& s) {
    if (s.done) (void)hipEventDestroy(s.done);
    if (s.word) (void)hipHostFree(s.word);
    s = HostSlot();
}
int take_slot(HostSlot* out) {
    int dev = -1;
    SG_HIP_CHECK(hipGetDevice(&dev));
    {
        std::lock_guard<std::mutex> lock(g_slot_mutex);
        for (size_t i = 0; i < g_slots.size(); i++)
            if (g_slots[i].device == dev) {
                *out = g_slots[i];
                g_slots.erase(g_slots.begin() + i);
                return 0;
            }
    }
    HostSlot s;
    s.device = dev;
    SG_HIP_CHECK(hipHostMalloc(&s.word, 64, hipHostMallocMapped | hipHostMallocCoherent));
    if (hipError_t e = hipEventCreateWithFlags(&s.done, hipEventDisableTiming)) {
        drop_slot(s);
        return sg::fail("hipEventCreateWithFlags: %s", hipGetErrorString(e));
    }
    *out = s;
    return 0;
}
void give_slot(HostSlot s) {
    std::lock_guard<std::mutex> lock(g_slot_mutex);
    if (g_slots.size() < MAX_SLOTS) g_slots.push_back(s);
    else drop_slot(s);
}

// ---- SuperGrok v1.1 (aux: mu, aux2: sharpness) ------------------------------------------
// The smart gradient of an element lies in the scratch at its tile's place: tile * B.tile + offset within the tile.
template <int GELU, class BT>
__global__ __launch_bounds__(THREADS) void k_sg11_smart(BT B, const float* __restrict__ W1, const float* __restrict__ b1,
                                                         const float* __restrict__ W2, const float* __restrict__ b2, int H,
                                                         float clip_norm, float rescale, double* norm_partials, float* smart) {
    __shared__ float sW1[2 * MAX_HIDDEN], sb1[MAX_HIDDEN], sW2[MAX_HIDDEN];
    load_net(W1, b1, W2, H, sW1, sb1, sW2);
    const Clip clip = global_norm(B, clip_norm);        // (its barriers cover the weights)
    const MetaNet<GELU> net = {sW1, sb1, sW2, b2[0], H, (const __attribute__((address_space(4))) MetaPoly*)B.table};
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    float* const out = smart + (int64_t)blockIdx.x * B.tile - start;
    const float alpha = R.alpha;
    float dot = 0.0f, ss = 0.0f, mm = 0.0f;
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
        for (int c = 0; c < V; c++) {
            g[c] = sg_fma(rescale, net(g[c], s[c]), g[c]);
            dot = sg_fma(g[c], mu[c], dot);
            ss = sg_fma(g[c], g[c], ss);
            mm = sg_fma(mu[c], mu[c], mm);
        }
        stf<V>(out, i, g);
    });
    BatchCommon C = B;
    C.partials = norm_partials;
    tile_sums<3>(C, (double)dot, (double)ss, (double)mm);
}

template <class BT>
__global__ __launch_bounds__(THREADS) void k_sg11_adam(BT B, float beta2, float eps, float decay, float lamb, float ramp,
                                                        float temperature, const float* smart) {
    int start, cnt, ti;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt, &ti);
    const float* const in = smart + (int64_t)blockIdx.x * B.tile - start;
    // cosine gate of this tensor (compute_cosine_gate_fused; csrc/ops.cpp:272-278)
    double s[3];
    tensor_sums<3>(B, R, ti, start, s);
    const float cosv = (float)s[0] / ((float)sqrt(s[1]) * (float)sqrt(s[2]) + 1e-8f);
    const float gate = 1.0f / (1.0f + sg_exp(-temperature * cosv));
    const float lamb_eff = ramp > 0.0f ? (ramp * gate) * lamb : 0.0f;
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float fg[V], mu[V];
        ldf<V>(in, i, fg);
        ldf<V>(R.aux, i, mu);
#pragma unroll
        for (int c = 0; c < V; c++) fg[c] = sg_fma(lamb_eff, mu[c], fg[c]);
        adam_update<V>(R, i, fg, R.beta1, 1.0f - R.beta1, beta2, 1.0f - beta2, eps, decay);
    });
}

// ---- LookSAM ----------------------------------------------------------------------------------------------
// Rec roles: restore  param=param, aux2=backup;  directions  aux=v (fp32), grad=sam_grad, aux2=normal_grad;
//            adjust   grad=grad, aux=v (fp32)
template <class BT>
__global__ __launch_bounds__(THREADS) void k_ls_restore(BT B) {
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float p[V];
        ldt<V>(R.aux2, R.dtype, i, p);
        stt<V>(R.param, R.dtype, i, p);
    });
}

template <class BT>
__global__ __launch_bounds__(THREADS) void k_ls_diff_sumsq(BT B) {
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    float acc = 0.0f;
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float a[V], b[V];
        ldt<V>(R.grad, R.dtype, i, a);
        ldt<V>(R.aux2, R.dtype, i, b);
#pragma unroll
        for (int c = 0; c < V; c++) {
            const float d = sg::round_to(R.dtype, a[c] - b[c]);     // as the reference forms it: subtracted in the gradients' own type
            acc = sg_fma(d, d, acc);
        }
    });
    tile_sums<1>(B, (double)acc);
}

template <class BT>
__global__ __launch_bounds__(THREADS) void k_ls_direction(BT B) {
    int start, cnt, ti;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt, &ti);
    double s[1];
    tensor_sums<1>(B, R, ti, start, s);
    const float norm = (float)sqrt(s[0]);
    if (!(norm >= 1e-12f)) return;          // that tensor's direction stays as it was
    const float inv = 1.0f / norm;
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float a[V], b[V];
        ldt<V>(R.grad, R.dtype, i, a);
        ldt<V>(R.aux2, R.dtype, i, b);
#pragma unroll
        for (int c = 0; c < V; c++) a[c] = (a[c] - b[c]) * inv;      // the device branch widens both gradients before subtracting (csrc/ops.cpp:621-623)
        stf<V>(R.aux, i, a);
    });
}

// sum of squares of each tensor's gradient
template <class BT>
__global__ __launch_bounds__(THREADS) void k_grad_sumsq(BT B) {
    int start, cnt;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt);
    float acc = 0.0f;
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float g[V];
        ldt<V>(R.grad, R.dtype, i, g);
#pragma unroll
        for (int c = 0; c < V; c++) acc = sg_fma(g[c], g[c], acc);
    });
    tile_sums<1>(B, (double)acc);
}

template <class BT>
__global__ __launch_bounds__(THREADS) void k_ls_adjust(BT B, float la) {
    int start, cnt, ti;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt, &ti);
    double s[1];
    tensor_sums<1>(B, R, ti, start, s);
    const float scale = la * (float)sqrt(s[0]);
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float d[V], g[V];
        ldf<V>(R.aux, i, d);
        ldt<V>(R.grad, R.dtype, i, g);
#pragma unroll
        for (int c = 0; c < V; c++) g[c] = sg_fma(scale, sg::round_to(R.dtype, d[c]), g[c]);    // the direction is converted to the gradient's type first (csrc/ops.cpp:646)
        stt<V>(R.grad, R.dtype, i, g);
    });
}

// ---- SuperGrok v2 pre-pass: per-tensor norm clip + non-finite guard ------------------------------------------
// Rec roles: grad = input gradient, param = output (a new tensor, as the reference makes one)
template <class BT>
__global__ __launch_bounds__(THREADS) void k_sg2_clip(BT B, float max_norm) {
    int start, cnt, ti;
    const Rec& R = tile_rec(B, blockIdx.x, &start, &cnt, &ti);
    double s[1];
    tensor_sums<1>(B, R, ti, start, s);
    // a NaN norm compares false (no clip); an infinite one gives scale 0 and the guard below zeroes what 0*inf leaves
    const float norm = (float)sqrt(s[0]);
    const float scale = (norm > max_norm) ? max_norm / (norm + 1e-12f) : 1.0f;
    for_tile(R, start, cnt, [&](auto v, int i) {
        constexpr int V = decltype(v)::value;
        float g[V];
        ldt<V>(R.grad, R.dtype, i, g);
#pragma unroll
        for (int c = 0; c < V; c++) {
            if (scale != 1.0f) g[c] = sg::round_to(R.dtype, g[c] * scale);      // the product is a tensor of the gradient's type
            g[c] = sg::finite_or_zero(g[c]);
        }
        stt<V>(R.param, R.dtype, i, g);
    });
}

// ---- host side ---------------------------------------------------------------------------------------------
enum Need { N_PARAM = 1, N_GRAD = 2, N_EA = 4, N_EASQ = 8, N_AUX = 16, N_AUX2 = 32, AUX2_F32 = 64, SHARP = 128 };      // SHARP: aux2 is a sharpness array

int collect(int n, const SgFamilyTensor* ts, int need, float lr, std::vector<Rec>* recs) {
    if (!ts) return sg::fail("NULL argument");
    recs->reserve(n);
    for (int i = 0; i < n; i++) {
        const SgFamilyTensor& t = ts[i];
        if (t.numel == 0) continue;
        if (((need & N_PARAM) && !t.param) || ((need & N_GRAD) && !t.grad) || ((need & N_EA) && !t.exp_avg) ||
            ((need & N_EASQ) && !t.exp_avg_sq) || ((need & N_AUX) && !t.aux) || ((need & N_AUX2) && !t.aux2))
            return sg::fail("tensor %d: NULL pointer", i);
        const int dtype = (need & SHARP) ? t.dtype & ~SG_SHARP_F32 : t.dtype;
        const bool s32 = t.dtype != dtype, aux2_f32 = s32 || (need & AUX2_F32);
        if (check_dtype(i, dtype) || check_numel(i, t.numel)) return 1;
        if ((need & N_EASQ) && (!(t.bc1 > 0.0f) || !(t.bc2 > 0.0f))) return sg::fail("bias corrections must be positive (step >= 1)");
        const uintptr_t typed = bits(t.param) | bits(t.grad) | (aux2_f32 ? 0 : bits(t.aux2));
        const uintptr_t f32 = bits(t.exp_avg) | bits(t.exp_avg_sq) | bits(t.aux) | (aux2_f32 ? bits(t.aux2) : 0);
        recs->push_back({t.param, t.grad, t.exp_avg, t.exp_avg_sq, t.aux, t.aux2, (int32_t)t.numel, (int16_t)dtype,
                         vec4_ok(dtype, typed, f32), (int8_t)s32, (need & N_EASQ) ? lr / t.bc1 : 0.0f, t.bc2, t.alpha, t.beta1});
    }
    return 0;
}

int looksam_collect(int n, const SgLookSamTensor* ts, int mode, std::vector<Rec>* recs) {
    if (!ts) return sg::fail("NULL argument");
    recs->reserve(n);
    for (int i = 0; i < n; i++) {
        const SgLookSamTensor& t = ts[i];
        if (t.numel == 0) continue;
        if (!t.a || !t.b || (mode == 1 && !t.c)) return sg::fail("tensor %d: NULL pointer", i);
        if (check_dtype(i, t.dtype) || check_numel(i, t.numel)) return 1;
        Rec r = {};
        r.numel = (int32_t)t.numel;
        r.dtype = (int16_t)t.dtype;
        if (mode == 0) { r.param = t.a; r.aux2 = t.b; r.vec4 = vec4_ok(t.dtype, bits(t.a) | bits(t.b), 0); }
        if (mode == 1) {
            r.aux = static_cast<float*>(t.a); r.grad = const_cast<void*>(t.b); r.aux2 = t.c;
            r.vec4 = vec4_ok(t.dtype, bits(t.b) | bits(t.c), bits(t.a));
        }
        if (mode == 2) {
            r.grad = t.a; r.aux = const_cast<float*>(static_cast<const float*>(t.b));
            r.vec4 = vec4_ok(t.dtype, bits(t.a), bits(t.b));
        }
        recs->push_back(r);
    }
    return 0;
}

}  // namespace
}  // namespace sgew

extern "C" {

size_t sg_family_workspace_bytes(int num_tensors, const int64_t* numels) {
    if (num_tensors < 0 || (num_tensors > 0 && !numels)) return 0;
    sgew::Layout L;
    if (sgew::make_layout(num_tensors, numels, &L)) return 0;
    // v1.1: smart gradients by tile, and partial sums of the norm apart from those of the cosine gate
    return L.bytes + sizeof(float) * (size_t)L.tiles * L.tile + sizeof(double) * 3 * (size_t)(L.tiles + 1) + 512;
}

int sg_grokadamw_step(int num_tensors, const SgFamilyTensor* tensors, float alpha, float lamb, float beta1, float beta2, float lr,
                      float wd, float eps, float grad_clip_norm, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    std::vector<Rec> recs;
    // the EMA buffer may be NULL for every tensor when lamb == 0: the step is then plain AdamW
    if (collect(num_tensors, tensors, N_PARAM | N_GRAD | N_EA | N_EASQ | (lamb != 0.0f ? N_AUX : 0), lr, &recs)) return 1;
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, grad_clip_norm > 0.0f, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        if (grad_clip_norm > 0.0f) launch_sumsq(B, st);
        hipLaunchKernelGGL(k_grokadamw<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B, grad_clip_norm, alpha, lamb, beta1, beta2, eps,
                           1.0f - lr * wd);
        SG_LAUNCH_CHECK("k_grokadamw");
        return 0;
    });
}

int sg_neuralgrok_step(int num_tensors, const SgFamilyTensor* tensors, const SgAmplifier* amp, float alpha_amp, float beta_amp,
                       float beta1, float beta2, float lr, float wd, float eps, float grad_clip_norm, void* workspace,
                       size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    if (!amp || !amp->W1 || !amp->b1 || !amp->W2 || !amp->b2) return sg::fail("NULL argument");
    if (amp->hidden < 1 || amp->hidden > MAX_HIDDEN) return sg::fail("hidden_dim %d outside [1,%d]", amp->hidden, MAX_HIDDEN);
    std::vector<Rec> recs;
    if (collect(num_tensors, tensors, N_PARAM | N_GRAD | N_EA | N_EASQ, lr, &recs)) return 1;
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, true, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        const int slots = amp_slots(amp->hidden);
        launch_sumsq(B, st, PrepAmp{amp->W1, amp->b1, amp->W2, amp->hidden, slots});
        hipLaunchKernelGGL(k_neuralgrok<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B, amp->W1, amp->b1, amp->W2, amp->b2, amp->hidden, slots,
                           grad_clip_norm, alpha_amp, beta_amp, beta1, beta2, eps, 1.0f - lr * wd);
        SG_LAUNCH_CHECK("k_neuralgrok");
        return 0;
    });
}

int sg_prodigy_step(int num_tensors, const SgFamilyTensor* tensors, float d_lr, float beta1, float beta2, float lr, float wd, float eps,
                    float* d_lr_out, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (d_lr_out) *d_lr_out = d_lr;
    if (num_tensors <= 0) return 0;
    std::vector<Rec> recs;
    if (collect(num_tensors, tensors, N_PARAM | N_GRAD | N_EA | N_EASQ | N_AUX | N_AUX2 | AUX2_F32, lr, &recs)) return 1;
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    HostSlot slot;
    if (d_lr_out && take_slot(&slot)) return 1;
    const int rc = with_batch(recs, workspace, workspace_bytes, st, true, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        const int blocks = partial_blocks(B.tiles);
        hipLaunchKernelGGL(k_prodigy_partial<BT>, dim3(blocks), dim3(THREADS), 0, st, B, blocks);
        hipLaunchKernelGGL(k_prodigy_dlr<BT>, dim3(1), dim3(THREADS), 0, st, B, blocks, d_lr, slot.word);
        if (d_lr_out) SG_HIP_CHECK(hipEventRecord(slot.done, st));
        hipLaunchKernelGGL(k_prodigy<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B, beta1, beta2, lr, wd, eps);
        SG_LAUNCH_CHECK("k_prodigy");
        if (d_lr_out) {
            SG_HIP_CHECK(hipEventSynchronize(slot.done));
            *d_lr_out = *static_cast<volatile float*>(slot.word);
        }
        return 0;
    });
    if (d_lr_out) {
        if (rc == 0) give_slot(slot);
        else drop_slot(slot);
    }
    return rc;
}

int sg_lion_step(int num_tensors, const SgFamilyTensor* tensors, float lr, float beta1, float beta2, float wd, void* workspace,
                 size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    std::vector<Rec> recs;
    if (collect(num_tensors, tensors, N_PARAM | N_GRAD | N_EA, lr, &recs)) return 1;
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, false, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        hipLaunchKernelGGL(k_lion<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B, lr, beta1, beta2, wd);
        SG_LAUNCH_CHECK("k_lion");
        return 0;
    });
}

int sg11_fused_step(int num_tensors, const SgFamilyTensor* tensors, const Sg15Net* net, float beta2, float lr, float wd, float eps,
                    float lamb, float ramp, float gate_temperature, float grad_clip_norm, void* workspace, size_t workspace_bytes,
                    void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    if (!net || !net->W1 || !net->b1 || !net->W2 || !net->b2) return sg::fail("NULL argument");
    if (net->hidden < 1 || net->hidden > MAX_HIDDEN) return sg::fail("hidden_dim %d outside [1,%d]", net->hidden, MAX_HIDDEN);
    if (net->gelu_mode != 0 && net->gelu_mode != 1) return sg::fail("bad gelu_mode %d", net->gelu_mode);
    std::vector<Rec> recs;
    if (collect(num_tensors, tensors, N_PARAM | N_GRAD | N_EA | N_EASQ | N_AUX | N_AUX2 | SHARP, lr, &recs)) return 1;
    if (recs.empty()) return 0;
    // scratch behind the bookkeeping region: partial sums of the cosine gates, then the smart gradients
    std::vector<int64_t> numels(recs.size());
    for (size_t i = 0; i < recs.size(); i++) numels[i] = recs[i].numel;
    Layout L;
    if (make_layout((int)recs.size(), numels.data(), &L)) return 1;
    const size_t gate_bytes = sg::align_up(sizeof(double) * 3 * (size_t)(L.tiles + 1), 256);
    const size_t need = L.bytes + gate_bytes + sizeof(float) * (size_t)L.tiles * L.tile;
    if (!workspace || workspace_bytes < need) return sg::fail("workspace too small: need %zu bytes, got %zu", need, workspace_bytes);
    double* gates = reinterpret_cast<double*>(static_cast<unsigned char*>(workspace) + L.bytes);
    float* smart = reinterpret_cast<float*>(static_cast<unsigned char*>(workspace) + L.bytes + gate_bytes);
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, true, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        const auto run = [&](auto gelu) {
            hipLaunchKernelGGL((k_sg11_smart<decltype(gelu)::value, BT>), dim3(B.tiles), dim3(THREADS), 0, st, B, net->W1, net->b1, net->W2,
                               net->b2, net->hidden, grad_clip_norm, net->rescale, gates, smart);
        };
        if (net->gelu_mode == 0) {
            launch_sumsq(B, st, PrepMetaPoly{net->W1, net->b1, net->W2, net->b2, net->hidden});
            run(std::integral_constant<int, 0>{});
        } else {
            launch_sumsq(B, st);
            run(std::integral_constant<int, 1>{});
        }
        BT G = B;
        G.partials = gates;
        launch_tensor_sums<3>(G, st);
        hipLaunchKernelGGL(k_sg11_adam<BT>, dim3(B.tiles), dim3(THREADS), 0, st, G, beta2, eps, 1.0f - lr * wd, lamb, ramp, gate_temperature,
                           smart);
        SG_LAUNCH_CHECK("k_sg11_adam");
        return 0;
    });
}

int sg2_clip_grads(int num_tensors, const Sg2ClipTensor* tensors, float max_norm, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    if (!tensors) return sg::fail("NULL argument");
    std::vector<Rec> recs;
    recs.reserve(num_tensors);
    for (int i = 0; i < num_tensors; i++) {
        const Sg2ClipTensor& t = tensors[i];
        if (t.numel == 0) continue;
        if (!t.grad || !t.out) return sg::fail("tensor %d: NULL pointer", i);
        if (check_dtype(i, t.dtype) || check_numel(i, t.numel)) return 1;
        Rec r = {};
        r.grad = const_cast<void*>(t.grad);
        r.param = t.out;
        r.numel = (int32_t)t.numel;
        r.dtype = (int16_t)t.dtype;
        r.vec4 = vec4_ok(t.dtype, bits(t.grad) | bits(t.out), 0);
        recs.push_back(r);
    }
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, true, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        hipLaunchKernelGGL(k_grad_sumsq<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B);
        launch_tensor_sums<1>(B, st);
        hipLaunchKernelGGL(k_sg2_clip<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B, max_norm);
        SG_LAUNCH_CHECK("k_sg2_clip");
        return 0;
    });
}

int sg_looksam_restore(int num_tensors, const SgLookSamTensor* tensors, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    std::vector<Rec> recs;
    if (looksam_collect(num_tensors, tensors, 0, &recs)) return 1;
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, false, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        hipLaunchKernelGGL(k_ls_restore<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B);
        SG_LAUNCH_CHECK("k_ls_restore");
        return 0;
    });
}

int sg_looksam_directions(int num_tensors, const SgLookSamTensor* tensors, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    std::vector<Rec> recs;
    if (looksam_collect(num_tensors, tensors, 1, &recs)) return 1;
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, true, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        hipLaunchKernelGGL(k_ls_diff_sumsq<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B);
        launch_tensor_sums<1>(B, st);
        hipLaunchKernelGGL(k_ls_direction<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B);
        SG_LAUNCH_CHECK("k_ls_direction");
        return 0;
    });
}

int sg_looksam_adjust(int num_tensors, const SgLookSamTensor* tensors, float la, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace sgew;
    if (num_tensors <= 0) return 0;
    std::vector<Rec> recs;
    if (looksam_collect(num_tensors, tensors, 2, &recs)) return 1;
    if (recs.empty()) return 0;
    hipStream_t st = (hipStream_t)stream;
    return with_batch(recs, workspace, workspace_bytes, st, true, [&](const auto& B) {
        using BT = std::decay_t<decltype(B)>;
        hipLaunchKernelGGL(k_grad_sumsq<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B);
        launch_tensor_sums<1>(B, st);
        hipLaunchKernelGGL(k_ls_adjust<BT>, dim3(B.tiles), dim3(THREADS), 0, st, B, la);
        SG_LAUNCH_CHECK("k_ls_adjust");
        return 0;
    });
}

}  // extern "C"
