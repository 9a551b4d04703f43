// Shared plumbing of the elementwise fused steps: the per-call tensor records
// and their tile prefix, tile -> tensor lookup, typed four-element access and
// the deterministic device-side reductions (partial sums in double, added up
// in a fixed order by every block that needs the result).
#ifndef SG_ELEMWISE_HPP_
#define SG_ELEMWISE_HPP_
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "sg_common.hpp"

namespace sgew {
namespace {

// Elements per workgroup.  Large calls use 4096 (16 per lane: few, long workgroups stream best); small calls use
// shorter tiles so that there are several workgroups per CU and few elements in series per lane.  A function of the
// call's total size only, so the workspace layout, the records and the kernels agree.
inline int tile_for(int64_t total) { return total >= (8 << 20) ? 4096 : (total >= (1 << 20) ? 1024 : 256); }
constexpr int THREADS = 256;
constexpr int MAX_HIDDEN = 256;
constexpr int MAX_PARTIALS = 1024;     // blocks of a whole-call reduction: what one consumer block adds up in four loads per lane

// One tensor as the kernels see it; which pointer is what depends on the step (see the collectors of each file).
struct Rec {
    void* param;
    void* grad;
    float* ea;
    float* easq;
    float* aux;
    const void* aux2;
    int32_t numel;
    int16_t dtype;
    int8_t vec4;           // every pointer allows four elements per lane and access
    int8_t sharp32;        // aux2 (sharpness) is fp32, rounded to dtype when read
    float step_size, bc2, alpha, beta1;
};
static_assert(sizeof(Rec) == 72, "Rec layout");

struct Layout {
    int n, tiles, tile, widest;      // widest: tiles of the largest tensor
    size_t off_recs, off_prefix, off_partials, off_tred, off_table, bytes;
    int64_t total;
};
constexpr size_t TABLE_BYTES = 8192;   // meta-net table of a call (MetaPoly or AmpTable)

inline int make_layout(int n, const int64_t* numels, Layout* L) {
    int64_t tiles = 0, total = 0, widest = 0;
    for (int i = 0; i < n; i++) {
        if (numels[i] < 0 || numels[i] > 0x7fffffff) return sg::fail("tensor %d: bad numel %lld", i, (long long)numels[i]);
        total += numels[i];
    }
    const int TILE = tile_for(total);
    for (int i = 0; i < n; i++) {
        const int64_t t = (numels[i] + TILE - 1) / TILE;
        tiles += t;
        widest = t > widest ? t : widest;
    }
    if (tiles > 0x7fffffff) return sg::fail("too many elements");
    L->tile = TILE;
    L->n = n;
    L->tiles = (int)tiles;
    L->widest = (int)widest;
    size_t o = 0;
    auto take = [&](size_t b) { size_t r = o; o = sg::align_up(o + b, 256); return r; };
    // records and tile prefix table back to back: one upload (calls of more tensors than travel as kernel arguments)
    L->off_recs = take(sizeof(Rec) * (size_t)n + sizeof(int) * (size_t)(n + 1));
    L->off_prefix = L->off_recs + sizeof(Rec) * (size_t)n;
    L->off_partials = take(sizeof(double) * 3 * (size_t)(tiles + 1));     // up to three sums per tile
    L->off_tred = take(sizeof(double) * 3 * (size_t)(n + 1));             // per-tensor sums
    L->off_table = take(TABLE_BYTES);
    L->total = total;
    L->bytes = o;
    return 0;
}

struct BatchCommon {
    int n, tiles, tile;
    int folded;           // consumers of per-tensor sums add up the tensor's tiles themselves (no k_sum_tiles launch)
    double* partials;
    double* tred;         // [n][3]
    void* table;
};
// The records of a call as kernel arguments.  A launch of a copy kernel that only carries the table costs 1.6 us of
// its own and about as much again before the next kernel starts, a third of a Grokfast step on 14 tensors.  CAP: the
// argument block stays below 4 KB.
constexpr int CAP = SG_ELEMWISE_ARG_TENSORS;
struct BatchArg : BatchCommon {
    Rec recs[CAP];
    int prefix[CAP];      // first tile of tensor i + 1
};
static_assert(sizeof(BatchArg) + 128 <= 4096, "kernel arguments stay below 4 KB");
// Calls of more tensors: the table lies in the workspace.
struct BatchPtr : BatchCommon {
    const Rec* recs;
    const int* prefix;    // [n + 1]
};

// Calls f(batch) with the records as kernel arguments where they fit, else uploaded into the workspace.  scratch:
// whether the step uses partial sums or a table.
template <class F>
int with_batch(const std::vector<Rec>& recs, void* workspace, size_t ws_bytes, hipStream_t st, bool scratch, F&& f) {
    const int n = (int)recs.size();
    std::vector<int64_t> numels(n);
    for (int i = 0; i < n; i++) numels[i] = recs[i].numel;
    Layout L;
    if (make_layout(n, numels.data(), &L)) return 1;
    if ((scratch || n > CAP) && (!workspace || ws_bytes < L.bytes)) return sg::fail("workspace too small: need %zu bytes, got %zu", L.bytes, ws_bytes);
    if (((uintptr_t)workspace & 255u) != 0) return sg::fail("workspace must be 256-byte aligned");
    unsigned char* ws = static_cast<unsigned char*>(workspace);
    BatchCommon c;
    c.n = n;
    c.tiles = L.tiles;
    c.tile = L.tile;
    // up to 512 tiles a tensor: 6 KB read per consumer block and sum, against a launch of its own (4.5 us)
    c.folded = L.widest <= 512 ? 1 : 0;
    c.partials = reinterpret_cast<double*>(ws + L.off_partials);
    c.tred = reinterpret_cast<double*>(ws + L.off_tred);
    c.table = ws + L.off_table;
    if (n <= CAP) {
        BatchArg B;
        static_cast<BatchCommon&>(B) = c;
        std::memcpy(B.recs, recs.data(), sizeof(Rec) * (size_t)n);
        int run = 0;
        for (int i = 0; i < n; i++) B.prefix[i] = run += (int)((numels[i] + L.tile - 1) / L.tile);
        return f(B);
    }
    std::vector<uint32_t> blob((sizeof(Rec) * (size_t)n + sizeof(int) * (size_t)(n + 1)) / 4, 0u);
    std::memcpy(blob.data(), recs.data(), sizeof(Rec) * (size_t)n);
    int* prefix = reinterpret_cast<int*>(blob.data() + sizeof(Rec) * (size_t)n / 4);
    for (int i = 0; i < n; i++) prefix[i + 1] = prefix[i] + (int)((numels[i] + L.tile - 1) / L.tile);
    if (sg::upload_words(ws + L.off_recs, blob.data(), blob.size() * 4, st)) return 1;
    BatchPtr B;
    static_cast<BatchCommon&>(B) = c;
    B.recs = reinterpret_cast<const Rec*>(ws + L.off_recs);
    B.prefix = reinterpret_cast<const int*>(ws + L.off_prefix);
    return f(B);
}

// tensor index of a tile; *first: its first tile
__device__ __forceinline__ int tile_tensor(const BatchArg& B, int tile, int* first) {
    // at most 64 tensors: one load and a ballot in place of a chain of dependent loads
    const int lane = threadIdx.x & 63;
    const int end = lane < B.n ? B.prefix[lane] : 0x7fffffff;
    const int ti = __popcll(__ballot(end <= tile));
    *first = ti > 0 ? __builtin_amdgcn_readlane(end, ti - 1) : 0;
    return ti;
}
__device__ __forceinline__ int tile_tensor(const BatchPtr& B, int tile, int* first) {
    const int ti = sg::upper_seg(sg::as_const(B.prefix), B.n, tile);
    *first = B.prefix[ti];
    return ti;
}
template <class BT>
__device__ __forceinline__ const Rec& tile_rec(const BT& B, int tile, int* start, int* cnt, int* tensor = nullptr) {
    int first;
    const int ti = tile_tensor(B, tile, &first);
    const Rec& R = B.recs[ti];
    *start = (tile - first) * B.tile;
    *cnt = min(B.tile, R.numel - *start);
    if (tensor) *tensor = ti;
    return R;
}

// ---- one or four elements per lane -------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
template <int V>
__device__ __forceinline__ void ldf(const float* p, int i, float (&x)[V]) {
    if constexpr (V == 4) {
        const f32x4 v = *(const SG_GLOBAL f32x4*)(p + i);
#pragma unroll
        for (int c = 0; c < 4; c++) x[c] = v[c];
    } else {
        x[0] = ((const SG_GLOBAL float*)p)[i];
    }
}
template <int V>
__device__ __forceinline__ void stf(float* p, int i, const float (&x)[V]) {
    if constexpr (V == 4) *(SG_GLOBAL f32x4*)(p + i) = f32x4{x[0], x[1], x[2], x[3]};
    else ((SG_GLOBAL float*)p)[i] = x[0];
}
// typed: the tensor's own storage type
template <int V>
__device__ __forceinline__ void ldt(const void* p, int dtype, int i, float (&x)[V]) {
    if constexpr (V == 4) {
        if (dtype == SG_F32) return ldf<4>(static_cast<const float*>(p), i, x);
        const u16x4 v = *(const SG_GLOBAL u16x4*)(static_cast<const uint16_t*>(p) + i);
#pragma unroll
        for (int c = 0; c < 4; c++) x[c] = dtype == SG_F16 ? __half2float(__ushort_as_half(v[c])) : sg::bf16_bits_to_f(v[c]);
    } else {
        x[0] = sg::load_elem(p, dtype, i);
    }
}
template <int V>
__device__ __forceinline__ void stt(void* p, int dtype, int i, const float (&x)[V]) {
    if constexpr (V == 4) {
        if (dtype == SG_F32) return stf<4>(static_cast<float*>(p), i, x);
        u16x4 v;
#pragma unroll
        for (int c = 0; c < 4; c++) v[c] = dtype == SG_F16 ? __half_as_ushort(__float2half_rn(x[c])) : sg::f_to_bf16_bits(x[c]);
        *(SG_GLOBAL u16x4*)(static_cast<uint16_t*>(p) + i) = v;
    } else {
        sg::store_elem(p, dtype, i, x[0]);
    }
}
// sharpness of a tensor: in its type, or in fp32 and rounded to it
template <int V>
__device__ __forceinline__ void ldsharp(const Rec& R, int i, float (&x)[V]) {
    if (!R.sharp32) return ldt<V>(R.aux2, R.dtype, i, x);
    ldf<V>(static_cast<const float*>(R.aux2), i, x);
#pragma unroll
    for (int c = 0; c < V; c++) x[c] = sg::round_to(R.dtype, x[c]);
}

// Runs body(V, i) over the elements of a tile: four consecutive ones per lane where the tensor's pointers allow
// 16-byte (8-byte for 16-bit types) accesses, single ones for the ragged end and for other tensors.
template <class B>
__device__ __forceinline__ void for_tile(const Rec& R, int start, int cnt, B body) {
    int done = 0;
    if (R.vec4) {
        done = cnt & ~3;
        for (int k = threadIdx.x * 4; k < done; k += THREADS * 4) body(std::integral_constant<int, 4>{}, start + k);
    }
    for (int k = done + threadIdx.x; k < cnt; k += THREADS) body(std::integral_constant<int, 1>{}, start + k);
}

// ---- deterministic sums -------------------------------------------
// blocks of a whole-call reduction over `tiles` tiles
inline int partial_blocks(int tiles) { return tiles < MAX_PARTIALS ? tiles : MAX_PARTIALS; }

struct NoExtra {
    static constexpr bool any = false;
    template <class BT> __device__ void operator()(const BT&) const {}
};
// Sum of squares of all gradients, one partial sum per block (block b takes tiles b, b + blocks, ...).  One more
// block, where a step has a table to prepare from its meta-net's weights, does that meanwhile.
template <class BT, class Extra>
__global__ __launch_bounds__(THREADS) void k_sumsq(BT B, int blocks, Extra extra) {
    if (Extra::any && (int)blockIdx.x == blocks) {
        extra(B);
        return;
    }
    __shared__ double sm[4];
    float acc = 0.0f;
    double sum = 0.0;
    for (int tile = blockIdx.x; tile < B.tiles; tile += blocks) {
        int start, cnt;
        const Rec& R = tile_rec(B, tile, &start, &cnt);
        for_tile(R, start, cnt, [&](auto v, int i) {
            constexpr int V = decltype(v)::value;
            float g[V];
            ldt<V>(R.grad, R.dtype, i, g);
#pragma unroll
            for (int c = 0; c < V; c++) acc = sg_fma(g[c], g[c], acc);
        });
        sum += (double)acc;
        acc = 0.0f;
    }
    const double tot = sg::block_sum(sum, sm);
    if (threadIdx.x == 0) B.partials[blockIdx.x] = tot;
}
template <class BT, class Extra = NoExtra>
void launch_sumsq(const BT& B, hipStream_t st, Extra extra = Extra()) {
    const int blocks = partial_blocks(B.tiles);
    hipLaunchKernelGGL((k_sumsq<BT, Extra>), dim3(blocks + (Extra::any ? 1 : 0)), dim3(THREADS), 0, st, B, blocks, extra);
}

// Global norm (called by every block of the consumer) and the clip coefficient of clip_grad_norms_device_side.
struct Clip {
    float norm, coef;
    bool on;
};
template <class BT>
__device__ __forceinline__ Clip global_norm(const BT& B, float clip_norm) {
    __shared__ double sm[4];
    const int blocks = B.tiles < MAX_PARTIALS ? B.tiles : MAX_PARTIALS;
    double acc = 0.0;
    for (int k = threadIdx.x; k < blocks; k += THREADS) acc += B.partials[k];
    Clip c;
    c.norm = (float)sqrt(sg::block_sum(acc, sm));
    c.on = clip_norm > 0.0f && c.norm > clip_norm;
    c.coef = c.on ? clip_norm / (c.norm + 1e-6f) : 1.0f;
    return c;
}

// ---- per-tensor sums: up to three per tile, then per tensor -------------
template <int S, class BT>
__device__ __forceinline__ void tile_sums(const BT& B, double a, double b = 0.0, double c = 0.0) {
    __shared__ double sm[4];
    const double v[3] = {a, b, c};
#pragma unroll
    for (int s = 0; s < S; s++) {
        const double t = sg::block_sum(v[s], sm);
        if (threadIdx.x == 0) B.partials[3 * (size_t)blockIdx.x + s] = t;
    }
}
template <int S, class BT>
__device__ __forceinline__ void add_tiles(const BT& B, int lo, int hi, double (&out)[S]) {
    __shared__ double sm[4];
    double acc[S] = {};
    for (int k = lo + (int)threadIdx.x; k < hi; k += THREADS)
#pragma unroll
        for (int s = 0; s < S; s++) acc[s] += B.partials[3 * (size_t)k + s];
#pragma unroll
    for (int s = 0; s < S; s++) out[s] = sg::block_sum(acc[s], sm);
}
// block t: sums of tensor t's tiles into tred[t]
template <int S, class BT>
__global__ __launch_bounds__(THREADS) void k_sum_tiles(BT B) {
    const int t = blockIdx.x;
    int lo, hi;
    if constexpr (std::is_same_v<BT, BatchArg>) { lo = t > 0 ? B.prefix[t - 1] : 0; hi = B.prefix[t]; }
    else { lo = B.prefix[t]; hi = B.prefix[t + 1]; }
    double s[S];
    add_tiles<S>(B, lo, hi, s);
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < S; k++) B.tred[3 * t + k] = s[k];
}
template <int S, class BT>
void launch_tensor_sums(const BT& B, hipStream_t st) {
    if (!B.folded) hipLaunchKernelGGL((k_sum_tiles<S, BT>), dim3(B.n), dim3(THREADS), 0, st, B);
}
// the sums of tensor ti (start: offset of the caller's tile), for every lane of the block
template <int S, class BT>
__device__ __forceinline__ void tensor_sums(const BT& B, const Rec& R, int ti, int start, double (&out)[S]) {
    if (B.folded) {
        const int lo = (int)blockIdx.x - start / B.tile;
        add_tiles<S>(B, lo, lo + (R.numel + B.tile - 1) / B.tile, out);
    } else {
#pragma unroll
        for (int s = 0; s < S; s++) out[s] = B.tred[3 * ti + s];
    }
}

inline int check_dtype(int i, int dtype) {
    if (dtype != SG_F32 && dtype != SG_F16 && dtype != SG_BF16) return sg::fail("tensor %d: bad dtype %d", i, dtype);
    return 0;
}
inline int check_numel(int i, int64_t n) {
    if (n < 0 || n > 0x7fffffff) return sg::fail("tensor %d: bad numel %lld", i, (long long)n);
    return 0;
}
// typed: pointers in the tensor's type OR-ed together; f32: fp32 pointers
inline int8_t vec4_ok(int dtype, uintptr_t typed, uintptr_t f32) {
    return (f32 & 15u) == 0 && (typed & (dtype == SG_F32 ? 15u : 7u)) == 0 ? 1 : 0;
}
inline uintptr_t bits(const void* p) { return (uintptr_t)p; }

// clipped gradient, written back in place when clipping is active (clip_grad_norms_device_side, csrc/ops.cpp:23-55)
template <int V>
__device__ __forceinline__ void clipped_grad(const Rec& R, int i, const Clip& clip, float (&g)[V]) {
    ldt<V>(R.grad, R.dtype, i, g);
    if (clip.on) {
#pragma unroll
        for (int c = 0; c < V; c++) g[c] = sg::round_to(R.dtype, g[c] * clip.coef);
        stt<V>(R.grad, R.dtype, i, g);
    }
}
// decoupled decay, then the Adam step: p*(1 - lr*wd) - step_size * ea / (sqrt(easq/bc2) + eps)
template <int V>
__device__ __forceinline__ void adam_update(const Rec& R, int i, const float (&fg)[V], float beta1, float om_beta1, float beta2,
                                            float om_beta2, float eps, float decay) {
    float ea[V], easq[V], p[V];
    ldf<V>(R.ea, i, ea);
    ldf<V>(R.easq, i, easq);
    ldt<V>(R.param, R.dtype, i, p);
#pragma unroll
    for (int c = 0; c < V; c++) {
        ea[c] = sg_fma(beta1, ea[c], om_beta1 * fg[c]);
        easq[c] = sg_fma(beta2, easq[c], (om_beta2 * fg[c]) * fg[c]);
        const float denom = __builtin_sqrtf(easq[c] / R.bc2) + eps;
        p[c] = sg_fma(p[c], decay, -((R.step_size * ea[c]) / denom));
    }
    stf<V>(R.ea, i, ea);
    stf<V>(R.easq, i, easq);
    stt<V>(R.param, R.dtype, i, p);
}

// ---- the 2 -> H -> 1 GELU net of SuperGrok v1.5 / v1.1 ---------------------------
// Every element evaluates H units of  w2 gelu(u + b1),  u = a g + c s: at H = 32 with the exact-erf form about 1100
// vector instructions, 0.6 ms for 25 M elements against 0.2 ms for their memory traffic.  But u is small for
// gradients of a model in training, and gelu(b1 + u) is then its Taylor polynomial: to fourth order in u the whole net is
// one polynomial of 15 terms in (g, s), whose coefficients are summed over the units once per call.  Bound of the
// remainder: |gelu^(5)| / 120 <= 0.023, so at |u| <= 1/36 it is 0.023 u^5 <= 3.8e-10, below 3e-8 of the unit's own
// value near b1 = 0 (u / 2) and below the rounding of the direct form elsewhere.  An element with a larger
// max|a| |g| + max|c| |s| (or a net with non-finite weights) takes the direct form.
constexpr float POLY_REACH = 1.0f / 36.0f;
struct MetaPoly {
    float c[15];           // 1 | g s | g2 gs s2 | g3 g2s gs2 s3 | g4 g3s g2s2 gs3 s4
    float amax, cmax;
};
struct PrepMetaPoly {
    static constexpr bool any = true;
    const float *W1, *b1, *W2, *b2;
    int H;
    template <class BT>
    __device__ void operator()(const BT& B) const {
        __shared__ double red[4][15];
        __shared__ float mx[4][2];
        double c[15] = {};
        float a0 = 0.0f, c0 = 0.0f;
        const int h = threadIdx.x;
        if (h < H) {
            a0 = W1[2 * h];
            c0 = W1[2 * h + 1];
            const double a = a0, s = c0, b = b1[h], w = W2[h];
            const double phi = 0.3989422804014326779 * exp(-0.5 * b * b), Phi = 0.5 * erfc(-0.70710678118654752440 * b);
            // gelu^(k)(b) / k!
            const double d0 = b * Phi, d1 = Phi + b * phi, d2 = phi * (2.0 - b * b) / 2.0, d3 = phi * (b * b * b - 4.0 * b) / 6.0,
                         d4 = phi * (-b * b * b * b + 7.0 * b * b - 4.0) / 24.0;
            c[0] = w * d0;
            c[1] = w * d1 * a; c[2] = w * d1 * s;
            c[3] = w * d2 * a * a; c[4] = 2.0 * w * d2 * a * s; c[5] = w * d2 * s * s;
            c[6] = w * d3 * a * a * a; c[7] = 3.0 * w * d3 * a * a * s; c[8] = 3.0 * w * d3 * a * s * s; c[9] = w * d3 * s * s * s;
            c[10] = w * d4 * a * a * a * a; c[11] = 4.0 * w * d4 * a * a * a * s; c[12] = 6.0 * w * d4 * a * a * s * s;
            c[13] = 4.0 * w * d4 * a * s * s * s; c[14] = w * d4 * s * s * s * s;
            a0 = sg_abs(a0);
            c0 = sg_abs(c0);
        }
        bool bad = false;
#pragma unroll
        for (int k = 0; k < 15; k++) {
            bad = bad || !(c[k] == c[k]) || !(fabs(c[k]) < 1e30);
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) c[k] += __shfl_down(c[k], d, 64);
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            a0 = sg_max(a0, __shfl_down(a0, d, 64));
            c0 = sg_max(c0, __shfl_down(c0, d, 64));
        }
        if ((h & 63) == 0) {
#pragma unroll
            for (int k = 0; k < 15; k++) red[h >> 6][k] = c[k];
            mx[h >> 6][0] = a0;
            mx[h >> 6][1] = c0;
        }
        bad = __syncthreads_or(bad ? 1 : 0) != 0;
        MetaPoly* out = static_cast<MetaPoly*>(B.table);
        if (h < 15) out->c[h] = (float)((red[0][h] + red[1][h]) + (red[2][h] + red[3][h]) + (h == 0 ? (double)b2[0] : 0.0));
        if (h < 2) {
            const float m = sg_max(sg_max(mx[0][h], mx[1][h]), sg_max(mx[2][h], mx[3][h]));
            (h == 0 ? out->amax : out->cmax) = bad ? __builtin_inff() : m;
        }
    }
};

// The net's output for one element.  GELU 0: exact erf, with the polynomial where it holds; 1: sigmoid form.
template <int GELU>
struct MetaNet {
    const float *sW1, *sb1, *sW2;
    float bias2;
    int H;
    const __attribute__((address_space(4))) MetaPoly* P;
    __device__ __forceinline__ float direct(float g, float s) const {
        float acc = 0.0f;
        for (int h = 0; h < H; h++) {
            const float z = sg_fma(sW1[2 * h + 1], s, sW1[2 * h] * g) + sb1[h];
            const float a = (GELU == 0) ? sg_gelu_erf(z) : sg_gelu_sigmoid(z);
            acc = sg_fma(sW2[h], a, acc);
        }
        return acc + bias2;
    }
    __device__ __forceinline__ float operator()(float g, float s) const {
        if (GELU == 0 && sg_fma(P->amax, sg_abs(g), P->cmax * sg_abs(s)) <= POLY_REACH) {
            // Horner in g, each coefficient a polynomial in s
            const float k4 = P->c[10];
            const float k3 = sg_fma(s, P->c[11], P->c[6]);
            const float k2 = sg_fma(s, sg_fma(s, P->c[12], P->c[7]), P->c[3]);
            const float k1 = sg_fma(s, sg_fma(s, sg_fma(s, P->c[13], P->c[8]), P->c[4]), P->c[1]);
            const float k0 = sg_fma(s, sg_fma(s, sg_fma(s, sg_fma(s, P->c[14], P->c[9]), P->c[5]), P->c[2]), P->c[0]);
            return sg_fma(g, sg_fma(g, sg_fma(g, sg_fma(g, k4, k3), k2), k1), k0);
        }
        return direct(g, s);
    }
};
// loads the weights into the block's LDS (no barrier)
__device__ __forceinline__ void load_net(const float* W1, const float* b1, const float* W2, int H, float* sW1, float* sb1, float* sW2) {
    for (int k = threadIdx.x; k < 2 * H; k += THREADS) sW1[k] = W1[k];
    for (int k = threadIdx.x; k < H; k += THREADS) { sb1[k] = b1[k]; sW2[k] = W2[k]; }
}

}  // namespace
}  // namespace sgew
#endif
