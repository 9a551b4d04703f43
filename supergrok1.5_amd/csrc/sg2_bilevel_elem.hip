// Per-element part of the bilevel meta-net update of SuperGrok v2, forward and backward in one pass: GRU, soft
// top-4 product-key routing (softmax of 10 x the four best scores of each sub-key, 16 experts per head), expert
// MLPs and the skip connection, followed at once by the gradients of  sum_i cot_i * smart_i  with respect to the
// two scan contexts of every element and to every weight of this part.
//
// Stands in for the per-element kernels of launch_mamba3_peer_backward[_batched]
// (csrc/supergrok2_mamba_peer_backward_kernels.cu of the reference, driven from
// grokking_optimizers/supergrok2.py:516-1330); the arithmetic is that of Mamba3PEERMetaNet.forward_for_bilevel
// (grokking_optimizers/mamba3_peer_metanet.py:395-436) and its autograd derivative.
//
// One wave per tile of 64 elements, one lane per element, every wave on its own: its tiles are a contiguous range, its
// staging rows are its own part of LDS, and nothing in the tile loop waits for another wave.  20 KB of LDS and at most
// 256 registers per wave: eight waves, two per SIMD, share a CU.  Nothing is kept between forward and backward: a
// lane holds its element's activations in registers, and the routing of a head is differentiated before the next head
// is evaluated.  Weight gradients are sums over elements, formed by fp32 matrix instructions from rows that the lanes
// leave in LDS (64 elements are the contraction):
//   * experts (16 per element and head, chosen per element).  An expert's hidden unit m is active where
//     W1[m] g + b1[m] > 0, i.e. on one side of the threshold -b1[m] / W1[m], so between two neighbouring thresholds of
//     its 16 units the expert is a straight line  out = A g + B.  k_expert_tables sorts the thresholds of every expert
//     and tabulates (A, B) for the 17 intervals.  The gradients of expert e need, per unit, S0 = sum w [unit active] and
//     S1 = sum w g [unit active] over the elements routed to e (w: routing weight times d loss / d head), i.e. sums of
//     (w, w g) per interval.  A wave holds, for +x and for -x of a reference magnitude x, the line of every expert and
//     the borders of the interval it holds on: an element whose g lies there for all of its experts costs one 16-byte
//     LDS read and a fma per expert, and the sums over such elements are outer products (first sub-key weights) (x)
//     (second sub-key weights), 16 x 16 x 4 instructions, separately for g > 0 and g <= 0.  The positive elements of a
//     tile take the first rows and the others the rows after them, so that each step is of one sign.
//     The bilevel pass hands the elements over in the order of the scan, by |g|: x is then the |g| of the tile's middle
//     element and almost every element of a large tensor lies in the interval of x for every expert.  When x moves past a
//     threshold of an expert, the lane that holds that expert's sums adds them to the interval's bin (a row of this
//     workgroup in memory) and starts again.  In element order x stays next to zero.  The exceptions - elements in
//     another interval of one of their experts - look the interval up in the tables and move their (w, w g) to its bin
//     with atomics.  They are the largest of a tensor and come together, sixteen a lane and head, so a head's exceptions
//     are dealt to all lanes of the wave.  (A lane going through its own one by one waited twice for
//     memory each time: 370 us instead of 310 in a call of 0.42 M elements whose small tensors lay with few waves.  Two jobs a lane
//     at a time took 280 there, but the registers they need are missed by every tile: 1.3 % of a pass over 25 M.  With all of a trained net's exceptions taken by LDS atomics, in element
//     order, they were half of the pass.)
//     (An element exactly on a threshold counts the unit as inactive on both sides; forward value and gradient use
//     the same interval, so they stay consistent.)
//   * GRU and query matrices: d (x) x, 16 x 16 x 4 steps over 27 columns of x;
//   * product keys (rows chosen per element): d score as two 12-vectors with four non-zeros each (x) the query's halves,
//     in 4 x 4 x 1 blocks, two elements a step.
// Each workgroup writes its sums to its own row of a partials buffer and k_elem_finish adds the rows in a fixed order
// and turns the bins into the experts' gradients.  The dense and key sums are formed in a fixed order; the bins are
// filled by atomics of four waves, so the last bits of the expert gradients can differ from run to run (as with the
// reference's atomicAdd).
//
// The net's products and their transposes are chains of 4 x 4 x 1 matrix instructions (product4), the same multiply-adds in the
// same order as scalar code: 550 of them for 2200 multiply-adds with scalar operands, whose loads were waited for in some
// hundred places and spilled into vector-register lanes.  A head's nine registers of weights are requested a phase ahead.
// (7.65 -> 7.2 ms, 0.227 -> 0.218.)
// Bound by the vector ALU and the waits between its phases (about 3000 vector and 900 matrix instructions per wave and tile;
// a tile takes 80 000 clocks beside the other wave of its SIMD, of which the experts' 64 lines 8500, the sums of routing
// weights 17 000).  Measured on 25 M elements with module-initialised experts
// after some meta steps: 7.2 ms (9.2 with the experts' lines read pick by pick, the sums' operands not ahead of
// them, a tile's indexes not before the tile and the products in scalar form), 47 ms as one lane per element of a 256-lane workgroup that summed the
// outer products lane by lane from LDS; on 0.42 M elements 0.22 ms, 0.29 before those and with a small tensor's tiles side by
// side, 1.1 at first.  (Products with their weights spread over all lanes' registers, from LDS or memory, took as
// long as the scalar form, with the bins in LDS longer on large calls: registers are what there is least of.)
#include "sg2_internal.hpp"

namespace sg2 {
namespace {

constexpr int BE_WAVES = 4;
constexpr int BE_THREADS = 64 * BE_WAVES;
constexpr int TOPK = 4;
typedef float be_f32x4 __attribute__((ext_vector_type(4)));
constexpr int NBIN = EH + 1;            // intervals between an expert's sorted unit thresholds
static_assert(EH == 16 && PK == 12 && NE == PK * PK && NH == 4 && DM == 8 && GH == 4, "row layouts and lane roles below");
// x row: h_new[4] (r * h_old[4] once the heads are done), fwd ctx[8], bwd ctx[8], g, s, 1, h_old[4]; the first 22 are the query's input
constexpr int X_HN = 0, X_CF = 4, X_CB = 12, X_G = 20, X_S = 21, X_ONE = 22, X_H = 23;
constexpr int XW = 27;
// rows of the second staging area, by turns:
constexpr int CW = 25;                  // routing weights of a head: first sub-key[12], second sub-key[12], g
constexpr int C_ROWS = 80;              // 64 elements, those of either sign padded to whole pairs of steps
constexpr int KW = 33;                  // d score of a head: first[12], second[12], query[8]
constexpr int EW = 13;                  // of a head's picks whose interval is another one: weights [4][4], indexes (two words), g, d loss / d head; then up to 1024 jobs
constexpr int DW = 17;                  // d query of two heads [16], or d pre_z[4], d pre_r[4], d pre_h[4] of the GRU
constexpr int R_FLOATS = 64 * KW;
static_assert(C_ROWS * CW <= R_FLOATS && 64 * EW + 64 * TOPK * TOPK <= R_FLOATS && EW % 2 == 1 && XW % 2 == 1 && CW % 2 == 1 && KW % 2 == 1 && DW % 2 == 1, "odd strides: lane-consecutive rows hit all banks");
constexpr int WAVE_FLOATS = 64 * XW + R_FLOATS + 2 * NE * 4;       // ... and the lines (A, B, low border, high border) of every expert at +x and -x
constexpr int KEY_FLOATS = 2 * NH * PK * (DM / 2);
constexpr int BE_LDS_BYTES = 4 * (KEY_FLOATS + BE_WAVES * WAVE_FLOATS);
static_assert(2 * BE_LDS_BYTES <= 160 * 1024 && (64 * XW + R_FLOATS) % 4 == 0 && WAVE_FLOATS % 4 == 0 && KEY_FLOATS % 4 == 0, "two workgroups per CU, aligned tables");

constexpr int N_GRU = 3 * (GH * GRL + GH), N_QHEAD = DM * PIN;     // 276 GRU entries, 176 query entries per head
constexpr int N_DENSE = N_GRU + NH * N_QHEAD + KEY_FLOATS;         // 276 + 704 + 384
constexpr int N_BINS = NE * NBIN * 2;                              // sums of w and w g over the elements of each interval
constexpr int ROW_FLOATS = (N_BINS + N_DENSE + 31) / 32 * 32;      // a workgroup's row: bins, then the dense sums
constexpr int TABLE_FLOATS = NE * EH + NE * NBIN * 2;              // thresholds ascending [NE][EH], lines [NE][NBIN][2]
static_assert(TABLE_FLOATS % 32 == 0 && N_DENSE + 3 * NE * EH + NE == SG2_ELEM_GRAD_FLOATS, "gradient layout, aligned rows");
constexpr int BE_MAX_GROUPS = 512;       // two resident workgroups on each of the 256 CUs: one round, every wave walks the same number of tiles (+-1)

// (row of d, column of x) whose product sums make up GRU gradient entry o, in the order
// W_z[4][22] b_z[4] W_r[4][22] b_r[4] W_h[4][22] b_h[4]
__device__ __forceinline__ void gru_entry(int o, int* drow, int* xcol) {
    const int gate = o / (GH * GRL + GH), q = o % (GH * GRL + GH);
    if (q >= GH * GRL) { *drow = gate * GH + (q - GH * GRL); *xcol = X_ONE; return; }
    const int j = q / GRL, c = q % GRL;
    *drow = gate * GH + j;
    *xcol = c < 2 ? X_G + c : c < 2 + 2 * DM ? X_CF + (c - 2) : (gate == 2 ? X_HN : X_H) + (c - 2 - 2 * DM);     // the candidate sees r*h in place of h
}

// Is the hidden unit (w1, b1), whose threshold is the rank-th lowest of its expert, active on interval k (the k lowest
// thresholds lie below g)?  W1 > 0: above its threshold; W1 < 0: below it; W1 = 0: wherever b1 > 0.
__device__ __forceinline__ bool unit_active(float w1, float b1, int rank, int k) {
    return w1 > 0.0f ? rank < k : (w1 < 0.0f ? rank >= k : b1 > 0.0f);
}
// Threshold of unit m of an expert of width eh and its rank among the 16 (ties by unit index); a unit with W1 = 0, or beyond
// eh, has none (+inf, never passed): it is active or not by the sign of b1 alone.  Called by 16 lanes, one per unit.
struct Unit { float w1, b1, thr; int rank; };
__device__ __forceinline__ Unit unit_of(const float* __restrict__ W1, const float* __restrict__ B1, int e, int eh, int m) {
    Unit u;
    u.w1 = m < eh ? W1[e * eh + m] : 0.0f;
    u.b1 = m < eh ? B1[e * eh + m] : 0.0f;
    u.thr = u.w1 != 0.0f ? -u.b1 / u.w1 : __builtin_inff();
    u.rank = 0;
#pragma unroll
    for (int j = 0; j < EH; j++) {
        const float tj = __shfl(u.thr, j, EH);
        u.rank += (tj < u.thr || (tj == u.thr && j < m)) ? 1 : 0;
    }
    return u;
}

// One expert per wave; clears *all_zero where a threshold is not 0.
__global__ __launch_bounds__(64) void k_expert_tables(Sg2Weights W, int eh, float* __restrict__ tables, int* all_zero) {
    const int e = blockIdx.x, lane = threadIdx.x, m = lane & (EH - 1);
    const Unit u = unit_of(W.w[W_EXP_W1], W.w[W_EXP_B1], e, eh, m);
    const float w2 = m < eh ? W.w[W_EXP_W2][e * eh + m] : 0.0f;
    if (lane < EH) tables[e * EH + u.rank] = u.thr;
    // (plain store: every writer stores the same value)
    if (all_zero != nullptr && __builtin_amdgcn_ballot_w64(u.w1 != 0.0f ? u.thr != 0.0f : u.b1 > 0.0f) != 0 && lane == 0) *all_zero = 0;
    float A = 0.0f, B = W.w[W_EXP_B2][e];
#pragma unroll
    for (int j = 0; j < EH; j++) {
        const float w1j = __shfl(u.w1, j, EH), b1j = __shfl(u.b1, j, EH), w2j = __shfl(w2, j, EH);
        const int rj = __shfl(u.rank, j, EH);
        if (unit_active(w1j, b1j, rj, lane)) {        // interval = lane
            A = sg_fma(w2j, w1j, A);
            B = sg_fma(w2j, b1j, B);
        }
    }
    if (lane < NBIN) {
        tables[NE * EH + (e * NBIN + lane) * 2] = A;
        tables[NE * EH + (e * NBIN + lane) * 2 + 1] = B;
    }
}

// Where the elements come from: flat arrays in element order, or (FLAT false) the tensors of a bilevel pass, in the sorted
// order that its forward scan left in the workspace (ctx and d_ctx in sorted order too; gradients and sharpness from the
// sort's arrays, GRU state and cotangent gathered).
// While every unit threshold is 0 - the state a meta-net is made in - the pass goes through the elements as they lie, and
// the experts' sums are formed in one order that depends on nothing but the number of elements: PLAIN_GROUPS workgroups take
// tiles of 256 elements in turns, the four elements of a step of either sign.  No element is an exception then, and the
// first step of an optimizer that divides a gradient by its own size (Adam) makes the thresholds of these sums: of one that
// nearly cancels, the order it was added up in decides a good part, and with it what every later pass computes.
constexpr int PLAIN_GROUPS = 256, PLAIN_TILE = 256;
__device__ __forceinline__ int plain_groups(int total) { return min(PLAIN_GROUPS, (total + PLAIN_TILE - 1) / PLAIN_TILE); }
struct ElemArgs {
    const float *g, *s, *gru, *cot;       // flat only
    const float* ctx;
    float *smart, *d_ctx, *partials, *gru_out;
    const float* tables;
    int total;
    const float* norms;                   // not flat, or NULL: the cotangent is -v / norms[tensor] (-v where that is <= 1e-12)
    float rescale;
    Sg2Weights W;
};

// LDS accesses of a wave execute in order; this keeps the compiler from moving them across each other where lanes
// exchange data.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// (the row belongs to this workgroup alone: workgroup scope lets the add run in the L2 next to it)
__device__ __forceinline__ void bin_add(float* p, float v) { __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }

// The thresholds of an expert, read together.
struct Thresholds {
    float t[EH];
    __device__ __forceinline__ Thresholds(const float* __restrict__ ths, int e) {
        const float4* t4 = reinterpret_cast<const float4*>(ths + e * EH);
#pragma unroll
        for (int q = 0; q < EH / 4; q++) { const float4 v = t4[q]; t[4 * q] = v.x; t[4 * q + 1] = v.y; t[4 * q + 2] = v.z; t[4 * q + 3] = v.w; }
    }
    __device__ __forceinline__ int below(float g) const {      // how many lie below g
        int k = 0;
#pragma unroll
        for (int q = 0; q < EH; q++) k += t[q] < g ? 1 : 0;
        return k;
    }
    __device__ __forceinline__ float low(float g) const {      // the last below g, the first not below it
        float v = -__builtin_inff();
#pragma unroll
        for (int q = 0; q < EH; q++) v = t[q] < g ? t[q] : v;
        return v;
    }
    __device__ __forceinline__ float high(float g) const {
        float v = __builtin_inff();
#pragma unroll
        for (int q = EH - 1; q >= 0; q--) v = t[q] < g ? v : t[q];
        return v;
    }
};
__device__ __forceinline__ void order(float& a, float& b) {
    const float hi = __builtin_fmaxf(a, b), lo = __builtin_fminf(a, b);
    a = hi;
    b = lo;
}
// The four best of twelve scores, ties to the lower index, in index order, with the softmax of 10 x score over them.  A
// selection network gives the fourth best value and with it the set; scratch (12 floats of the lane's own) turns an index
// into its score.
__device__ __forceinline__ void best_four(const float (&sc)[PK], float* scratch, int (&idx)[TOPK], float (&wgt)[TOPK]) {
    float v[PK];
#pragma unroll
    for (int q = 0; q < PK; q++) { v[q] = sc[q]; scratch[q] = sc[q]; }
#pragma unroll
    for (int b = 0; b < PK; b += 4) {
        order(v[b], v[b + 1]); order(v[b + 2], v[b + 3]);
        order(v[b], v[b + 2]); order(v[b + 1], v[b + 3]);
        order(v[b + 1], v[b + 2]);
    }
    const float best = __builtin_fmaxf(__builtin_fmaxf(v[0], v[4]), v[8]);
    float c[4];
#pragma unroll
    for (int k = 0; k < 4; k++) c[k] = __builtin_fmaxf(v[k], v[7 - k]);
    order(c[0], c[2]); order(c[1], c[3]); order(c[0], c[1]); order(c[2], c[3]);
    float fourth = __builtin_fmaxf(c[0], v[11]);
#pragma unroll
    for (int k = 1; k < 4; k++) fourth = __builtin_fminf(fourth, __builtin_fmaxf(c[k], v[11 - k]));
    unsigned set = 0u;                       // bit PK-1-q: score q is among them
#pragma unroll
    for (int q = 0; q < PK; q++) set = set + set + (sc[q] >= fourth ? 1u : 0u);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(__popc(set) != TOPK) != 0, 0)) {
        // ties at the border go to the lower indices; scores that do not compare (NaN) leave the set short
        for (int q = PK - 1; q >= 0 && __popc(set) > TOPK; q--)
            if (scratch[q] == fourth) set &= ~(1u << (PK - 1 - q));
        for (int q = 0; q < PK && __popc(set) < TOPK; q++) set |= 1u << (PK - 1 - q);
    }
    float ex[TOPK];
#pragma unroll
    for (int k = 0; k < TOPK; k++) {
        const int lead = __builtin_clz(set);          // set is never empty here
        idx[k] = lead - (32 - PK);
        set &= ~(0x80000000u >> lead);
        ex[k] = wgt[k] = sg_exp(10.0f * (scratch[idx[k]] - best));
    }
    // added from the best score down
    order(ex[0], ex[1]); order(ex[2], ex[3]); order(ex[0], ex[2]); order(ex[1], ex[3]); order(ex[1], ex[2]);
    const float inv = 1.0f / (((ex[0] + ex[1]) + ex[2]) + ex[3]);
#pragma unroll
    for (int k = 0; k < TOPK; k++) wgt[k] *= inv;
}

template <bool FLAT>
__global__ __launch_bounds__(BE_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_bilevel_elem(ElemArgs a, Plan pl) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float* const s_keys = lds;                                        // [2][NH][PK][DM/2]
    float* const s_x = lds + KEY_FLOATS + wave * WAVE_FLOATS;         // [64][XW]
    float* const s_r = s_x + 64 * XW;
    float4* const s_tab = reinterpret_cast<float4*>(s_r + R_FLOATS);  // [2][NE]: g > 0, g <= 0
    float* const bins = a.partials + (size_t)blockIdx.x * ROW_FLOATS;
    const float* __restrict__ ths = a.tables;
    const float* __restrict__ lines = a.tables + NE * EH;

    for (int i = tid; i < N_BINS; i += BE_THREADS) bins[i] = 0.0f;
    for (int i = tid; i < KEY_FLOATS; i += BE_THREADS) s_keys[i] = i < KEY_FLOATS / 2 ? a.W.w[W_KEYS_A][i] : a.W.w[W_KEYS_B][i - KEY_FLOATS / 2];
    for (int i = lane; i < (64 * XW + R_FLOATS) / 4; i += 64) reinterpret_cast<be_f32x4*>(s_x)[i] = be_f32x4{0.0f, 0.0f, 0.0f, 0.0f};     // rows are read whole: no NaN may lie in what was never written
    __syncthreads();

    const sg::cfloat_p bz = sg::as_const(a.W.w[W_GRU_BZ]), br = sg::as_const(a.W.w[W_GRU_BR]), bh = sg::as_const(a.W.w[W_GRU_BH]);

    const int li = lane & 15, lk = lane >> 4;             // operand roles of the 16 x 16 x 4 instructions: row / column, element of the step
    // accumulators.  Register v of a 16 x 16 one: row 4 (lane / 16) + v, column lane % 16; of a 4 x 4 x 16 one: block lane / 4, row v, column lane % 4
    const be_f32x4 zero4 = be_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    be_f32x4 cen[4] = {zero4, zero4, zero4, zero4};       // outer products of the routing weights: w for g > 0, w for g <= 0, w g for g > 0, for g <= 0
    be_f32x4 qacc[2][2] = {{zero4, zero4}, {zero4, zero4}};       // d query of two heads (x) x: columns 0..15, 16..31
    be_f32x4 gacc[2] = {zero4, zero4};
    be_f32x4 kacc[NH] = {zero4, zero4, zero4, zero4};     // blocks 0..5 (even elements) and 6..11 (odd): first sub-key rows 0-3, 4-7, 8-11, second
    const int kb = (lane >> 2) % 12, kb6 = kb % 6;
    const int key_a = (kb / 6) * KW + kb6 * 4 + (lane & 3), key_b = (kb / 6) * KW + 24 + (kb6 / 3) * 4 + (lane & 3);

    // sums over the tile's elements of (rows of d, DW floats each) (x) (rows of x), four elements a step, operands two steps ahead
    auto outer_sums = [&](be_f32x4 (&acc)[2]) {
        const float* d = s_r + lk * DW + li;
        const float* x = s_x + lk * XW + li;
        float dv[2][2], x0[2][2], x1[2][2];
        auto fetch = [&](int t0, int q) {
#pragma unroll
            for (int t = 0; t < 2; t++) {
                dv[q][t] = d[4 * (t0 + t) * DW];
                x0[q][t] = x[4 * (t0 + t) * XW];
                x1[q][t] = x[4 * (t0 + t) * XW + 16];
            }
            asm volatile("" ::: "memory");
        };
        auto sum = [&](int q) {
#pragma unroll
            for (int t = 0; t < 2; t++) {
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(dv[q][t], x0[q][t], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(dv[q][t], x1[q][t], acc[1], 0, 0, 0);
            }
        };
        fetch(0, 0);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            if (q < 7) fetch(2 * q + 2, (q + 1) & 1);
            sum(q & 1);
        }
    };

    // the four experts whose sums this lane holds in cen: first index 4 lk + v, second index li
    const bool owner = lane < 48 && li < PK;
    float x_held = -1.0f;                                 // reference magnitude of the lines in s_tab (< 0: none yet)
    auto reference = [](float x, int neg) { return neg ? -x : __builtin_fmaxf(x, 1.40129846e-45f); };      // (+0 stands for the interval just above zero)
    auto line_at = [&](const Thresholds& th, int e, float r) {       // the expert's line at r and the borders of its interval
        const float2 ab = reinterpret_cast<const float2*>(lines)[e * NBIN + th.below(r)];
        const float high = th.high(r);
        return make_float4(ab.x, ab.y, th.low(r), high == high ? high : -__builtin_inff());      // (a NaN border holds nothing: minima would drop it)
    };
    auto move_reference = [&](float x) {
        if (!FLAT) {
            unsigned stale = 0u;             // bit 2 v + neg: x lies in another interval of expert v on that side
            if (owner) {
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const float4 t = s_tab[(q & 1) * NE + (4 * lk + (q >> 1)) * PK + li];
                    const float r = reference(x, q & 1);
                    stale |= t.z < r && r <= t.w ? 0u : 1u << q;
                }
            }
            while (__builtin_amdgcn_ballot_w64(stale != 0u) != 0) {       // one per lane at a time: a tile passes a few thresholds
                if (stale != 0u) {
                    const int q = __builtin_ctz(stale), v = q >> 1, neg = q & 1, e = (4 * lk + v) * PK + li;
                    stale &= stale - 1u;
                    const Thresholds th(ths, e);
                    float w = 0.0f, wg = 0.0f;
#pragma unroll
                    for (int k = 0; k < 8; k++) {      // (selects: a dynamic index would send the sums to scratch)
                        const bool it = k == q;
                        w = it ? cen[k & 1][k >> 1] : w;
                        wg = it ? cen[2 + (k & 1)][k >> 1] : wg;
                        cen[k & 1][k >> 1] = it ? 0.0f : cen[k & 1][k >> 1];
                        cen[2 + (k & 1)][k >> 1] = it ? 0.0f : cen[2 + (k & 1)][k >> 1];
                    }
                    s_tab[neg * NE + e] = line_at(th, e, reference(x, neg));
                    float* b = bins + 2 * (e * NBIN + th.below(reference(x_held, neg)));
                    bin_add(b, w);
                    bin_add(b + 1, wg);
                }
            }
        }
        x_held = x;
        wave_sync();
    };
    // the first lines of a wave, everything requested at once
    auto first_reference = [&](float x) {
        constexpr int ROUNDS = (2 * NE + 63) / 64;
        float4 line[ROUNDS];
#pragma unroll
        for (int r = 0; r < ROUNDS; r++) {
            const int t = min(r * 64 + lane, 2 * NE - 1), neg = t >= NE ? 1 : 0, e = t - neg * NE;
            line[r] = line_at(Thresholds(ths, e), e, reference(x, neg));
        }
#pragma unroll
        for (int r = 0; r < ROUNDS; r++)
            if (r * 64 + lane < 2 * NE) s_tab[r * 64 + lane] = line[r];
        x_held = x;
        wave_sync();
    };

    const int ntiles = FLAT ? (a.total + 63) / 64 : pl.elem_tiles * (ELEM_TILE / 64);
    const int nwaves = (int)gridDim.x * BE_WAVES, wv = (int)blockIdx.x * BE_WAVES + wave;
    int tile0 = (int)((int64_t)ntiles * wv / nwaves), tile1 = (int)((int64_t)ntiles * (wv + 1) / nwaves), step = 1;
    if ((int)gridDim.x == BE_MAX_GROUPS && ntiles < 16 * nwaves) {
        // Few tiles a wave: two waves share a SIMD, in the order of dispatch wv and wv + nwaves / 2, so an equal part is dealt to
        // every such pair and halved between its waves.  (Dealt wave by wave, both had one tile more than the others or neither:
        // 0.42 M elements are 3.2 tiles a wave, and the launch, 233 us, waited for a SIMD with eight; 226 now.  Where a wave
        // has many the odd tile is nothing, and neighbours on one SIMD cost: 25 M elements, 191 a wave, 7.8 ms -> 8.7.)
        const int half = nwaves / 2, pair = wv % half, second = wv / half;
        const int p0 = (int)((int64_t)ntiles * pair / half), p1 = (int)((int64_t)ntiles * (pair + 1) / half), mid = p0 + (p1 - p0 + 1) / 2;
        tile0 = second ? mid : p0;
        tile1 = second ? p1 : mid;
    }
    const bool plain = !FLAT && !sorted_rows(pl);
    if (plain) {
        static_assert(PLAIN_TILE == 64 * BE_WAVES, "a tile of 64 per wave");
        tile0 = wv;
        tile1 = (int)blockIdx.x < plain_groups(a.total) ? (a.total + 63) / 64 : 0;
        step = plain_groups(a.total) * BE_WAVES;
    }
    const float kscale = a.rescale / (float)NH;
    sg::Seg seg = {-1, 0, 0};
    float cot_norm = 0.0f;
    // The tensor at a tile index, the tile's first element there and how many it holds; 0 where the index has no tile.  A tensor's
    // last ELEM_TILE elements are 16 indexes whatever there is of them, their tiles spread evenly over these: the tiles of a
    // small tensor, whose elements are mostly exceptions (99 of them two or three times a tile's usual time), then fall to
    // waves with little else.
    auto place = [&](int tile, int& start) {
        constexpr int PER = ELEM_TILE / 64;
        const int et = tile / PER, at = tile % PER;
        if (et >= seg.end) {
            seg = sg::find_seg(sg::as_const(pl.elem_tile_prefix), pl.P, et);
            cot_norm = a.norms ? a.norms[seg.i] : 0.0f;
        }
        const int first = (et - seg.first) * ELEM_TILE, left = pl.tensors[seg.i].numel - first, tiles = min(PER, (left + 63) / 64);
        const int here = at * tiles / PER;
        start = first + here * 64;
        return at > 0 && (at - 1) * tiles / PER == here ? 0 : left - here * 64;
    };
    if (FLAT || plain) {
        if (tile0 < tile1) first_reference(0.0f);
    } else {
        for (int start; tile0 < tile1; tile0++) {
            const int cnt = place(tile0, start);
            if (cnt <= 0) continue;
            first_reference(sg_i2f((int32_t)pl.keys[0][pl.tensors[seg.i].off + start + min(cnt - 1, 32)]));
            break;
        }
    }
    int32_t next_val = 0;                 // of the lane's element in the next tile, requested a tile ahead (the gathers wait for it)
    uint32_t next_key = 0u;
    bool have_next = false;
    for (int tile = tile0; tile < tile1; tile += step) {
        // every lane runs the element code (the wave works on whole tiles): lanes past the end redo the last element with a
        // zero cotangent, which zeroes everything they add, and store nothing
        bool valid;
        int at;                              // where ctx and d_ctx rows lie
        int out_at;                          // where smart goes
        float g, s, cot;
        float4 h4;
        if (FLAT) {
            valid = tile * 64 + lane < a.total;
            at = out_at = valid ? tile * 64 + lane : a.total - 1;
            g = a.g[at]; s = a.s[at]; cot = valid ? a.cot[at] : 0.0f;
            h4 = reinterpret_cast<const float4*>(a.gru)[at];
        } else if (plain) {
            valid = tile * 64 + lane < a.total;
            at = out_at = valid ? tile * 64 + lane : a.total - 1;
            int ti = 0;                      // the lane's tensor: the last one that starts no later
            for (int n = pl.P; n > 1;) {
                const int half = n / 2;
                if (pl.tensors[ti + half].off <= at) ti += half;
                n -= half;
            }
            const TensorDev& T = pl.tensors[ti];
            const int orig = at - T.off;
            g = sg::load_elem(T.grad, T.dtype, orig);
            s = sharp_rounded(T, orig);
            cot = sg::load_elem(T.param, T.dtype, orig);
            if (a.norms) { const float norm = a.norms[ti]; cot = -(norm > 1e-12f ? cot / norm : cot); }
            cot = valid ? cot : 0.0f;
            const be_f32x4 hv = ((const SG_GLOBAL be_f32x4*)T.gru)[orig];
            h4 = make_float4(hv[0], hv[1], hv[2], hv[3]);
        } else {
            int start;
            const int cnt = place(tile, start);
            if (cnt <= 0) continue;
            const TensorDev& T = pl.tensors[seg.i];
            valid = lane < cnt;
            at = T.off + start + (valid ? lane : cnt - 1);
            int32_t val = next_val;
            uint32_t key = next_key;
            if (!have_next) { val = pl.vals[0][at]; key = pl.keys[0][at]; }
            const int orig = min(val & 0x7fffffff, T.numel - 1);
            out_at = T.off + orig;
            // the sort's values, except where it put 0 for an entry that is not finite: those stay what they are
            g = sg_i2f((int32_t)key | (val & (int32_t)0x80000000));
            if (key == 0u) g = sg::load_elem(T.grad, T.dtype, orig);
            s = 0.0f;
            if (pl.sharp_nonzero[seg.i] != 0) {
                s = pl.ssorted[at];
                if (s == 0.0f) s = sharp_rounded(T, orig);
            }
            cot = sg::load_elem(T.param, T.dtype, orig);
            if (a.norms) cot = -(cot_norm > 1e-12f ? cot / cot_norm : cot);
            cot = valid ? cot : 0.0f;
            const be_f32x4 hv = ((const SG_GLOBAL be_f32x4*)T.gru)[orig];
            h4 = make_float4(hv[0], hv[1], hv[2], hv[3]);
            have_next = cnt > 64 && tile + 1 < tile1;
            if (have_next) {
                const int then = T.off + start + 64 + min(lane, cnt - 65);
                next_val = pl.vals[0][then];
                next_key = pl.keys[0][then];
            }
            move_reference(__shfl(sg_abs(g), min(cnt - 1, 32), 64));
        }
        float* const xrow = s_x + lane * XW;
        // rows of the routing weights: positive elements first, padded to whole pairs of steps (eight rows), then the others
        const unsigned long long pos = __builtin_amdgcn_ballot_w64(g > 0.0f);
        const int npos = __popcll(pos), npos8 = (npos + 7) >> 3, nneg8 = (64 - npos + 7) >> 3;
        const int before = __builtin_amdgcn_mbcnt_hi((unsigned)(pos >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)pos, 0u));      // positive elements in lower lanes
        const int slot = plain ? lane : g > 0.0f ? before : 8 * npos8 + (lane - before);
        // ... of which lane 0..7 / 8..15 clears one
        const int pad = (lane < 8 ? npos : 8 * npos8 + (64 - npos) - 8) + lane, pad_end = plain ? 0 : lane < 8 ? 8 * npos8 : lane < 16 ? 8 * (npos8 + nneg8) : 0;

        float cf[DM], cb[DM], h[GH] = {h4.x, h4.y, h4.z, h4.w};
        {
            const float4* pf = reinterpret_cast<const float4*>(a.ctx + (size_t)at * DM);
            const float4* pb = reinterpret_cast<const float4*>(a.ctx + ((size_t)a.total + at) * DM);
            const float4 a0 = pf[0], a1 = pf[1], b0 = pb[0], b1 = pb[1];
            cf[0] = a0.x; cf[1] = a0.y; cf[2] = a0.z; cf[3] = a0.w; cf[4] = a1.x; cf[5] = a1.y; cf[6] = a1.z; cf[7] = a1.w;
            cb[0] = b0.x; cb[1] = b0.y; cb[2] = b0.z; cb[3] = b0.w; cb[4] = b1.x; cb[5] = b1.y; cb[6] = b1.z; cb[7] = b1.w;
        }
        // Weights of the products (product4), requested where they are used: lane 4 block + row holds row `row` of four.  (The lane
        // is opaque to the compiler, or they would be held, and spilled, from one tile to the next.)
        auto opaque_lane = [&]() { int ln = lane; asm volatile("" : "+v"(ln)); return ln; };
        // of a head's products: inputs 0 .. 7, 8 .. 15, 14 .. 21 of the query's two halves; the keys' entries
        struct HeadWeights { float w[3], k[2]; };
        auto head_weights = [&](int hh) {
            const int ln = opaque_lane(), row = ln & 3, block = ln >> 2;
            const float* const wq = a.W.w[W_PEER_Q] + hh * DM * PIN + (4 * (block >> 3) + row) * PIN + (block & 7);
            const int at_k = hh * PK * (DM / 2) + (4 * min(block >> 2, PK / 4 - 1) + row) * (DM / 2) + (block & 3);
            return HeadWeights{{wq[0], wq[8], wq[14]}, {a.W.w[W_KEYS_A][at_k], a.W.w[W_KEYS_B][at_k]}};
        };
        HeadWeights ahead;
        // ---- GRU forward
        float zg[GH], rg[GH], cand[GH], hn[GH];
        {
            const int ln = opaque_lane(), at_w = (ln & 3) * GRL + (ln >> 2);
            float wz[2], wr[2], wh[2];       // inputs 0 .. 15 and 6 .. 21
#pragma unroll
            for (int r = 0; r < 2; r++) { wz[r] = a.W.w[W_GRU_WZ][at_w + 6 * r]; wr[r] = a.W.w[W_GRU_WR][at_w + 6 * r]; wh[r] = a.W.w[W_GRU_WH][at_w + 6 * r]; }
            float x[GRL];
            x[0] = g; x[1] = s;
#pragma unroll
            for (int q = 0; q < DM; q++) { x[2 + q] = cf[q]; x[2 + DM + q] = cb[q]; }
#pragma unroll
            for (int q = 0; q < GH; q++) x[2 + 2 * DM + q] = h[q];
            static_assert(GRL == 22 && GH == 4, "two registers of sixteen inputs");
            const int zo = sg::opaque_zero();
            be_f32x4 vz = {bz[zo], bz[zo + 1], bz[zo + 2], bz[zo + 3]}, vr = {br[zo], br[zo + 1], br[zo + 2], br[zo + 3]}, vh = {bh[zo], bh[zo + 1], bh[zo + 2], bh[zo + 3]};
            each<GRL>([&](auto c) {
                constexpr int R = c < 16 ? 0 : 1, B = c - 6 * R;
                vz = product4<B>(wz[R], x[c], vz);
                vr = product4<B>(wr[R], x[c], vr);
                if constexpr (c < GRL - GH) vh = product4<B>(wh[R], x[c], vh);
            });
#pragma unroll
            for (int j = 0; j < GH; j++) { zg[j] = sg_sigmoid(vz[j]); rg[j] = sg_sigmoid(vr[j]); }
            ahead = head_weights(0);
            each<GH>([&](auto q) { vh = product4<GRL - GH + q - 6>(wh[1], rg[q] * h[q], vh); });
#pragma unroll
            for (int j = 0; j < GH; j++) {
                cand[j] = sg_tanh(vh[j]);
                hn[j] = sg_fma(zg[j], cand[j], (1.0f - zg[j]) * h[j]);
            }
        }
        if (FLAT && valid && a.gru_out != nullptr) reinterpret_cast<float4*>(a.gru_out)[at] = make_float4(hn[0], hn[1], hn[2], hn[3]);
        xrow[X_G] = g; xrow[X_S] = s; xrow[X_ONE] = 1.0f;
#pragma unroll
        for (int q = 0; q < DM; q++) { xrow[X_CF + q] = cf[q]; xrow[X_CB + q] = cb[q]; }
#pragma unroll
        for (int q = 0; q < GH; q++) { xrow[X_H + q] = h[q]; xrow[X_HN + q] = hn[q]; }

        // ---- heads: forward, then at once the head's backward
        float total = 0.0f;
        // d loss / d h_new and the contexts, [0] and four at a time in [1] .. [4]
        be_f32x4 dx[1 + 2 * DM / 4];
        float dq_even[DM];
#pragma unroll
        for (int q = 0; q < 1 + 2 * DM / 4; q++) dx[q] = be_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < DM; q++) dq_even[q] = 0.0f;
        const float kk = cot * kscale;                 // d loss / d head output
        const int side = g > 0.0f ? 0 : NE;
#pragma unroll 1
        for (int hh = 0; hh < NH; hh++) {
            float query[DM];
            int idx[2][TOPK];
            float wgt[2][TOPK];
            {
                const float (&w)[3] = ahead.w;
                const float (&wk)[2] = ahead.k;
                static_assert(PIN == 22 && DM == 8 && PK == 12, "blocks of the weights' registers");
                float x[PIN];
#pragma unroll
                for (int q = 0; q < GH; q++) x[q] = hn[q];
#pragma unroll
                for (int q = 0; q < DM; q++) { x[GH + q] = cf[q]; x[GH + DM + q] = cb[q]; }
                x[GH + 2 * DM] = g; x[GH + 2 * DM + 1] = s;
                be_f32x4 q4[2] = {be_f32x4{0.0f, 0.0f, 0.0f, 0.0f}, be_f32x4{0.0f, 0.0f, 0.0f, 0.0f}};
                each<PIN>([&](auto c) {
                    constexpr int R = c / 8, B = R < 2 ? c % 8 : c - 14;
                    q4[0] = product4<B>(w[R], x[c], q4[0]);
                    q4[1] = product4<8 + B>(w[R], x[c], q4[1]);
                });
#pragma unroll
                for (int dd = 0; dd < DM; dd++) query[dd] = q4[dd / 4][dd % 4];
                be_f32x4 sc4[2][PK / 4];
#pragma unroll
                for (int hf = 0; hf < 2; hf++)
#pragma unroll
                    for (int t = 0; t < PK / 4; t++) sc4[hf][t] = be_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                each<DM / 2>([&](auto dd) {
                    each<2>([&](auto hf) { each<PK / 4>([&](auto t) { sc4[hf][t] = product4<4 * t + dd>(wk[hf], q4[hf][int(dd)], sc4[hf][t]); }); });
                });
#pragma unroll
                for (int hf = 0; hf < 2; hf++) {
                    float sc[PK];
#pragma unroll
                    for (int q = 0; q < PK; q++) sc[q] = sc4[hf][q / 4][q % 4];
                    best_four(sc, s_r + lane * CW + hf * PK, idx[hf], wgt[hf]);
                }
            }
            wave_sync();
            // ---- experts: the line of each at this element's side of zero, where its interval holds g
            // (The sixteen records of a lane are requested four at a time, whole and one row ahead of their use, and the borders are
            // compared together: chosen pick by pick, they became sixteen branches with two waits for LDS each.)
            float ra[TOPK] = {0.f, 0.f, 0.f, 0.f}, rb[TOPK] = {0.f, 0.f, 0.f, 0.f};
            unsigned other = 0u;                     // picks whose interval is another one
            {
                const be_f32x4* const ta = reinterpret_cast<const be_f32x4*>(s_tab) + side;
                be_f32x4 t[2][TOPK];
                auto fetch = [&](int ia) {
                    const be_f32x4* const row = ta + idx[0][ia] * PK;
#pragma unroll
                    for (int ib = 0; ib < TOPK; ib++) t[ia & 1][ib] = row[idx[1][ib]];
                };
                fetch(0);
#pragma unroll
                for (int ia = 0; ia < TOPK; ia++) {
                    if (ia + 1 < TOPK) fetch(ia + 1);
                    be_f32x4 (&u)[TOPK] = t[ia & 1];
                    asm volatile("" : "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]));
                    float out[TOPK];
#pragma unroll
                    for (int ib = 0; ib < TOPK; ib++) out[ib] = sg_fma(u[ib][0], g, u[ib][1]);
                    const float low = __builtin_fmaxf(__builtin_fmaxf(u[0][2], u[1][2]), __builtin_fmaxf(u[2][2], u[3][2]));
                    const float high = __builtin_fminf(__builtin_fminf(u[0][3], u[1][3]), __builtin_fminf(u[2][3], u[3][3]));
                    if (__builtin_amdgcn_ballot_w64(!(low < g && g <= high)) != 0) {
#pragma unroll
                        for (int ib = 0; ib < TOPK; ib++) {
                            const bool in = u[ib][2] < g && g <= u[ib][3];
                            out[ib] = in ? out[ib] : 0.0f;
                            other |= in ? 0u : 1u << (ia * TOPK + ib);
                        }
                    }
#pragma unroll
                    for (int ib = 0; ib < TOPK; ib++) {
                        ra[ia] = sg_fma(wgt[1][ib], out[ib], ra[ia]);
                        rb[ib] = sg_fma(wgt[0][ia], out[ib], rb[ib]);
                    }
                }
            }
            if (!valid) other = 0u;
            if (__builtin_amdgcn_ballot_w64(other != 0u) != 0) {
                // some lanes have all sixteen of them (the largest elements of a tensor), others none: they are dealt to all lanes
                float* const mine = s_r + lane * EW;
                int ia4 = 0, ib4 = 0;
#pragma unroll
                for (int k = 0; k < TOPK; k++) {
                    ia4 |= idx[0][k] << (8 * k); ib4 |= idx[1][k] << (8 * k);
                    mine[k] = wgt[0][k]; mine[TOPK + k] = wgt[1][k];
                }
                mine[2 * TOPK] = __int_as_float(ia4); mine[2 * TOPK + 1] = __int_as_float(ib4);
                mine[2 * TOPK + 2] = g; mine[2 * TOPK + 3] = kk;
                float* const jobs = s_r + 64 * EW;           // (lane, pick) of each, then its output in the same place
                const int picks = __popc(other);
                int rank = 0, all = 0;                       // picks of the lanes below, of all
#pragma unroll
                for (int b = 0; b < 5; b++) {
                    const unsigned long long has = __builtin_amdgcn_ballot_w64((picks >> b) & 1);
                    rank += (int)__builtin_amdgcn_mbcnt_hi((unsigned)(has >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)has, 0u)) << b;
                    all += __popcll(has) << b;
                }
#pragma unroll
                for (int ia = 0; ia < TOPK; ia++)
                    if (__builtin_amdgcn_ballot_w64((other >> (TOPK * ia)) & 15u) != 0)
#pragma unroll
                        for (int p = TOPK * ia; p < TOPK * ia + TOPK; p++)
                            if ((other >> p) & 1u) jobs[rank + __popc(other & ((1u << p) - 1u))] = __int_as_float(16 * lane + p);
                wave_sync();
#pragma unroll 1
                for (int n = lane; n < all; n += 64) {
                    const int job = __float_as_int(jobs[n]), ia = (job >> 2) & 3, ib = job & 3;
                    const float* row = s_r + (job >> 4) * EW;
                    const int e = ((__float_as_int(row[2 * TOPK]) >> (8 * ia)) & 255) * PK + ((__float_as_int(row[2 * TOPK + 1]) >> (8 * ib)) & 255);
                    const float wa = row[ia], wb = row[TOPK + ib], eg = row[2 * TOPK + 2];
                    const Thresholds th(ths, e);
                    const int k = th.below(eg), kr = th.below(reference(x_held, !(eg > 0.0f)));
                    const float2 ab = reinterpret_cast<const float2*>(lines)[e * NBIN + k];
                    jobs[n] = sg_fma(ab.x, eg, ab.y);
                    const float w = (row[2 * TOPK + 3] * wa) * wb;
                    float* b = bins + 2 * e * NBIN;
                    bin_add(b + 2 * k, w);
                    bin_add(b + 2 * k + 1, w * eg);
                    bin_add(b + 2 * kr, -w);
                    bin_add(b + 2 * kr + 1, -(w * eg));
                }
                wave_sync();
#pragma unroll
                for (int ia = 0; ia < TOPK; ia++)
                    if (__builtin_amdgcn_ballot_w64((other >> (TOPK * ia)) & 15u) != 0)
#pragma unroll
                        for (int ib = 0; ib < TOPK; ib++) {
                            const int p = TOPK * ia + ib;
                            const float out = (other >> p) & 1u ? jobs[rank + __popc(other & ((1u << p) - 1u))] : 0.0f;
                            ra[ia] += wgt[1][ib] * out;
                            rb[ib] += wgt[0][ia] * out;
                        }
                wave_sync();
            }
            float head_out = 0.0f;
#pragma unroll
            for (int ia = 0; ia < TOPK; ia++) head_out = sg_fma(wgt[0][ia], ra[ia], head_out);
            total += head_out;
            float w_back[4];       // of the query's derivative, two of its entries each
            {
                const int ln = opaque_lane(), row = ln & 3, block = ln >> 2;
                const float* const wq = a.W.w[W_PEER_Q] + hh * DM * PIN + (block >> 3) * PIN + 4 * min(block & 7, 4) + row;
#pragma unroll
                for (int r = 0; r < 4; r++) w_back[r] = wq[2 * r * PIN];
            }
            // ---- sums of the routing weights over this tile's elements, four a step
            {
                float* const crow = s_r + slot * CW;
#pragma unroll
                for (int k = 0; k < 2 * PK; k++) crow[k] = 0.0f;
                crow[2 * PK] = g;
                if (pad < pad_end) {
#pragma unroll
                    for (int k = 0; k < CW; k++) s_r[pad * CW + k] = 0.0f;
                }
#pragma unroll
                for (int k = 0; k < TOPK; k++) {
                    crow[idx[0][k]] = kk * wgt[0][k];
                    crow[PK + idx[1][k]] = wgt[1][k];
                }
                wave_sync();
                // two steps at a time, the next two on their way
                const float* row = s_r + lk * CW;
                float av[2], bv[2], gv[2];
                auto fetch = [&]() {
#pragma unroll
                    for (int u = 0; u < 2; u++) { av[u] = row[4 * u * CW + li]; bv[u] = row[4 * u * CW + PK + li]; gv[u] = row[4 * u * CW + 2 * PK]; }
                    row += 8 * CW;
                };
                auto sums = [&](int steps, be_f32x4& acc, be_f32x4& acc_g) {
                    for (int t = 0; t < steps; t++) {
                        const float a0 = av[0], b0 = bv[0], g0 = gv[0], a1 = av[1], b1 = bv[1], g1 = gv[1];
                        fetch();
                        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b0, acc, 0, 0, 0);
                        acc_g = __builtin_amdgcn_mfma_f32_16x16x4f32(a0 * g0, b0, acc_g, 0, 0, 0);
                        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b1, acc, 0, 0, 0);
                        acc_g = __builtin_amdgcn_mfma_f32_16x16x4f32(a1 * g1, b1, acc_g, 0, 0, 0);
                    }
                };
                if (!plain) {
                    fetch();
                    sums(npos8, cen[0], cen[2]);
                    sums(nneg8, cen[1], cen[3]);
                } else {
#pragma unroll 1
                    for (int t = 0; t < 16; t++, row += 4 * CW) {
                        const float a4 = row[li], b4 = row[PK + li], g4 = row[2 * PK];
                        const float ap = g4 > 0.0f ? a4 : 0.0f, an = g4 > 0.0f ? 0.0f : a4;
                        cen[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(ap, b4, cen[0], 0, 0, 0);
                        cen[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(an, b4, cen[1], 0, 0, 0);
                        cen[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(ap * g4, b4, cen[2], 0, 0, 0);
                        cen[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(an * g4, b4, cen[3], 0, 0, 0);
                    }
                }
                wave_sync();
            }
            // ---- routing backward: softmax, scores, query
            float dq[DM], dv[2][TOPK];
#pragma unroll
            for (int hf = 0; hf < 2; hf++) {
                const float4* keys = reinterpret_cast<const float4*>(s_keys) + (hf * NH + hh) * PK;
                float mean = 0.0f;
#pragma unroll
                for (int k = 0; k < TOPK; k++) mean = sg_fma(wgt[hf][k], kk * (hf ? rb[k] : ra[k]), mean);
                float d0 = 0.0f, d1 = 0.0f, d2 = 0.0f, d3 = 0.0f;
#pragma unroll
                for (int k = 0; k < TOPK; k++) {
                    const float4 key = keys[idx[hf][k]];
                    dv[hf][k] = 10.0f * wgt[hf][k] * (kk * (hf ? rb[k] : ra[k]) - mean);
                    d0 = sg_fma(dv[hf][k], key.x, d0);
                    d1 = sg_fma(dv[hf][k], key.y, d1);
                    d2 = sg_fma(dv[hf][k], key.z, d2);
                    d3 = sg_fma(dv[hf][k], key.w, d3);
                }
                dq[4 * hf] = d0; dq[4 * hf + 1] = d1; dq[4 * hf + 2] = d2; dq[4 * hf + 3] = d3;
            }
            {
                each<DM>([&](auto dd) { each<5>([&](auto q) { dx[q] = product4<8 * (dd % 2) + q>(w_back[dd / 2], dq[dd], dx[q]); }); });
            }
            // ---- product-key gradients, d score (x) query half, two elements a step
            {
                float* const krow = s_r + lane * KW;
#pragma unroll
                for (int k = 0; k < 2 * PK; k++) krow[k] = 0.0f;
#pragma unroll
                for (int k = 0; k < TOPK; k++) {
                    krow[idx[0][k]] = dv[0][k];
                    krow[PK + idx[1][k]] = dv[1][k];
                }
#pragma unroll
                for (int dd = 0; dd < DM; dd++) krow[2 * PK + dd] = query[dd];
                wave_sync();
                // (operands eight steps ahead of the instructions that take them)
                auto key_sums = [&](be_f32x4& acc) {
                    float ka[2][8], kv[2][8];
                    auto fetch = [&](int t0, int q) {
#pragma unroll
                        for (int t = 0; t < 8; t++) { ka[q][t] = s_r[2 * (t0 + t) * KW + key_a]; kv[q][t] = s_r[2 * (t0 + t) * KW + key_b]; }
                        asm volatile("" ::: "memory");
                    };
                    auto sum = [&](int q) {
#pragma unroll
                        for (int t = 0; t < 8; t++) acc = __builtin_amdgcn_mfma_f32_4x4x1f32(ka[q][t], kv[q][t], acc, 0, 0, 0);
                    };
                    fetch(0, 0);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        if (q < 3) fetch(8 * q + 8, (q + 1) & 1);
                        sum(q & 1);
                    }
                };
                if (hh + 1 < NH) ahead = head_weights(hh + 1);
                if (hh == 0) key_sums(kacc[0]);
                else if (hh == 1) key_sums(kacc[1]);
                else if (hh == 2) key_sums(kacc[2]);
                else key_sums(kacc[3]);
                wave_sync();
            }
            // ---- query-matrix gradients, d query (x) query input, two heads at a time
            if ((hh & 1) == 0) {
#pragma unroll
                for (int dd = 0; dd < DM; dd++) dq_even[dd] = dq[dd];
            } else {
                float* const drow = s_r + lane * DW;
#pragma unroll
                for (int dd = 0; dd < DM; dd++) { drow[dd] = dq_even[dd]; drow[DM + dd] = dq[dd]; }
                wave_sync();
                if (hh == 1) outer_sums(qacc[0]);
                else outer_sums(qacc[1]);
                wave_sync();
            }
        }
        if (valid && a.smart != nullptr) a.smart[out_at] = sg_fma(a.rescale, total / (float)NH, g);

        // ---- GRU backward
        float dpz[GH], dpr[GH], dph[GH];
#pragma unroll
        for (int j = 0; j < GH; j++) {
            dpz[j] = (dx[0][j] * (cand[j] - h[j])) * (zg[j] * (1.0f - zg[j]));
            dph[j] = (dx[0][j] * zg[j]) * (1.0f - cand[j] * cand[j]);
        }
        {
            const int ln = opaque_lane(), row = ln & 3, block = ln >> 2, at_w = (block >> 2) * GRL + 2 + 4 * (block & 3) + row;
            const float wz = a.W.w[W_GRU_WZ][at_w], wr = a.W.w[W_GRU_WR][at_w], wh = a.W.w[W_GRU_WH][at_w];
            const float wh_h = a.W.w[W_GRU_WH][(block & 3) * GRL + 2 + 2 * DM + row];
            be_f32x4 drh = {0.0f, 0.0f, 0.0f, 0.0f};
            each<GH>([&](auto j) {
                each<4>([&](auto q) { dx[1 + q] = product4<4 * j + q>(wh, dph[j], dx[1 + q]); });
                drh = product4<j>(wh_h, dph[j], drh);
            });
#pragma unroll
            for (int j = 0; j < GH; j++) dpr[j] = (drh[j] * h[j]) * (rg[j] * (1.0f - rg[j]));
            each<GH>([&](auto j) {
                each<4>([&](auto q) { dx[1 + q] = product4<4 * j + q>(wz, dpz[j], dx[1 + q]); });
                each<4>([&](auto q) { dx[1 + q] = product4<4 * j + q>(wr, dpr[j], dx[1 + q]); });
            });
        }
        if (valid) {
            float4* of = reinterpret_cast<float4*>(a.d_ctx + (size_t)at * DM);
            float4* ob = reinterpret_cast<float4*>(a.d_ctx + ((size_t)a.total + at) * DM);
            of[0] = make_float4(dx[1][0], dx[1][1], dx[1][2], dx[1][3]); of[1] = make_float4(dx[2][0], dx[2][1], dx[2][2], dx[2][3]);
            ob[0] = make_float4(dx[3][0], dx[3][1], dx[3][2], dx[3][3]); ob[1] = make_float4(dx[4][0], dx[4][1], dx[4][2], dx[4][3]);
        }
        // ---- GRU gradients
        {
            float* const drow = s_r + lane * DW;
#pragma unroll
            for (int j = 0; j < GH; j++) { drow[j] = dpz[j]; drow[GH + j] = dpr[j]; drow[2 * GH + j] = dph[j]; xrow[X_HN + j] = rg[j] * h[j]; }
            wave_sync();
            outer_sums(gacc);
            wave_sync();
        }
    }

    // ---- this workgroup's sums -> its row of the partials buffer, through LDS: the waves' held expert sums with the
    // intervals they belong to (wave after wave: a fixed order), then the dense sums
    static_assert(6 * NE <= 64 * XW + R_FLOATS, "the held sums fit the wave's staging rows");
    if (owner) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int e = (4 * lk + v) * PK + li;
            const Thresholds th(ths, e);
#pragma unroll
            for (int neg = 0; neg < 2; neg++) {
                float* t = s_x + (neg * NE + e) * 3;
                t[0] = cen[neg][v];
                t[1] = cen[2 + neg][v];
                t[2] = (float)(x_held < 0.0f ? 0 : th.below(reference(x_held, neg)));      // (a wave without a tile holds zeros)
            }
        }
    }
    __syncthreads();
    for (int t = tid; t < 2 * NE; t += BE_THREADS) {
        for (int w = 0; w < BE_WAVES; w++) {
            const float* held = lds + KEY_FLOATS + w * WAVE_FLOATS + t * 3;
            float* b = bins + 2 * ((t % NE) * NBIN + (int)held[2]);
            bin_add(b, held[0]);
            bin_add(b + 1, held[1]);
        }
    }
    __syncthreads();
    constexpr int M_Q = 16 * 32, M_K = M_Q + 32 * 32, M_FLOATS = M_K + NH * 256;       // GRU [16][32], query [32][32], keys [NH][16 blocks][4][4]
    static_assert(M_FLOATS <= 64 * XW + R_FLOATS, "the sums fit the wave's staging rows");
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int row = 4 * lk + v;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            s_x[row * 32 + 16 * c + li] = gacc[c][v];
#pragma unroll
            for (int p = 0; p < 2; p++) s_x[M_Q + (16 * p + row) * 32 + 16 * c + li] = qacc[p][c][v];
        }
#pragma unroll
        for (int hd = 0; hd < NH; hd++) s_x[M_K + hd * 256 + (lane >> 2) * 16 + v * 4 + (lane & 3)] = kacc[hd][v];
    }
    __syncthreads();
    const float* const m0 = lds + KEY_FLOATS;
    auto waves_sum = [&](int i) { return ((m0[i] + m0[i + WAVE_FLOATS]) + m0[i + 2 * WAVE_FLOATS]) + m0[i + 3 * WAVE_FLOATS]; };
    static_assert(BE_WAVES == 4, "waves_sum");
    float* const out = bins + N_BINS;
    for (int o = tid; o < N_DENSE; o += BE_THREADS) {
        float v;
        if (o < N_GRU) {
            int drow, xcol;
            gru_entry(o, &drow, &xcol);
            v = waves_sum(drow * 32 + xcol);
        } else if (o < N_GRU + NH * N_QHEAD) {
            const int q = o - N_GRU;
            v = waves_sum(M_Q + (q / PIN) * 32 + q % PIN);
        } else {        // [half][head][row][entry]
            const int q = o - N_GRU - NH * N_QHEAD, hf = q / (KEY_FLOATS / 2), hd = q / (PK * (DM / 2)) % NH, row = q / (DM / 2) % PK, dd = q % (DM / 2);
            const int i = M_K + hd * 256 + (hf * 3 + row / 4) * 16 + (row % 4) * 4 + dd;
            v = waves_sum(i) + waves_sum(i + 6 * 16);
        }
        out[o] = v;
    }
}

// Rows of the partials buffer added in a fixed order, eight slices of rows per column.  The first workgroups take 64 columns
// of the dense sums each; each of the others takes the bins of one expert and forms its gradients from them: with S0, S1 of
// a unit the sums of the bins on its active side, d b1 = W2 S0, d W1 = W2 S1, d W2 = sum w relu(pre) = W1 S1 + b1 S0,
// d b2 = sum w.
constexpr int FIN_SLICES = 8;
constexpr int FIN_DENSE = (N_DENSE + 63) / 64;
// (All thresholds 0 in the bilevel pass: the gradients are formed per row and then added, in four slices, for the one order of
// k_bilevel_elem's sums.)
__global__ __launch_bounds__(64 * FIN_SLICES) void k_elem_finish(const float* __restrict__ partials, int rows, Sg2Weights W, int eh,
                                                                 float* __restrict__ out, Plan pl) {
    __shared__ float s_part[FIN_SLICES][64];
    const int col = threadIdx.x & 63, slice = threadIdx.x >> 6;
    const bool dense = blockIdx.x < FIN_DENSE;
    const int e = (int)blockIdx.x - FIN_DENSE;
    const int o = dense ? (int)blockIdx.x * 64 + col : col;
    const bool live = dense ? o < N_DENSE : col < 2 * NBIN;
    const float* src = partials + (dense ? N_BINS + o : e * NBIN * 2 + o);
    float acc = 0.0f;
    if (!dense && pl.whole_pass && !sorted_rows(pl)) {
        // columns: d W1[16], d b1[16], d W2[16], d b2; of a unit's active side only the bin next to zero is not empty
        const int kind = col / EH, m = col % EH, mw = min(m, eh - 1);
        const float w1 = W.w[W_EXP_W1][e * eh + mw], b1 = W.w[W_EXP_B1][e * eh + mw], w2 = W.w[W_EXP_W2][e * eh + mw];
        int above = 0;
        for (int q = 0; q < eh; q++) above += W.w[W_EXP_W1][e * eh + q] != 0.0f ? 1 : 0;
        const float* bin = partials + e * NBIN * 2;
        rows = plain_groups(pl.total);
        if (slice < 4) {
#pragma unroll 4
            for (int r = slice; r < rows; r += 4) {
                const float* at = bin + (size_t)r * ROW_FLOATS + (w1 > 0.0f ? 2 * above : 0);
                const float S0 = w1 != 0.0f ? at[0] : 0.0f, S1 = w1 != 0.0f ? at[1] : 0.0f;
                acc += kind == 0 ? w2 * S1 : kind == 1 ? w2 * S0 : kind == 2 ? sg_fma(w1, S1, b1 * S0)
                                 : above > 0 ? bin[(size_t)r * ROW_FLOATS] + bin[(size_t)r * ROW_FLOATS + 2 * above] : bin[(size_t)r * ROW_FLOATS];
            }
        }
        s_part[slice][col] = acc;
        __syncthreads();
        if (slice != 0) return;
        acc = ((s_part[0][col] + s_part[1][col]) + s_part[2][col]) + s_part[3][col];
        float* const dst = out + N_DENSE;
        if (kind < 3 && m < eh) dst[kind * NE * eh + e * eh + m] = acc;
        if (col == 3 * EH) dst[3 * NE * eh + e] = acc;
        return;
    }
    if (live) {
#pragma unroll 8
        for (int r = slice; r < rows; r += FIN_SLICES) acc += src[(size_t)r * ROW_FLOATS];
    }
    s_part[slice][col] = acc;
    __syncthreads();
    if (slice != 0) return;
#pragma unroll
    for (int q = 1; q < FIN_SLICES; q++) acc += s_part[q][col];
    if (dense) {
        if (live) out[o] = acc;
        return;
    }
    s_part[0][col] = acc;
    wave_sync();
    const int m = col & (EH - 1);
    const Unit u = unit_of(W.w[W_EXP_W1], W.w[W_EXP_B1], e, eh, m);
    const float* bin = s_part[0];
    float S0 = 0.0f, S1 = 0.0f, sum = 0.0f;
#pragma unroll
    for (int k = 0; k < NBIN; k++) {
        sum += bin[2 * k];
        if (!unit_active(u.w1, u.b1, u.rank, k)) continue;
        S0 += bin[2 * k];
        S1 += bin[2 * k + 1];
    }
    float* const dst = out + N_DENSE;
    if (col < eh) {
        const float w2 = W.w[W_EXP_W2][e * eh + m];
        dst[e * eh + m] = w2 * S1;
        dst[NE * eh + e * eh + m] = w2 * S0;
        dst[2 * NE * eh + e * eh + m] = sg_fma(u.w1, S1, u.b1 * S0);
    }
    if (col == 0) dst[3 * NE * eh + e] = sum;
}

int elem_groups(int64_t tiles) {
    const int64_t groups = (tiles + BE_WAVES - 1) / BE_WAVES;
    return (int)(groups < BE_MAX_GROUPS ? (groups > 0 ? groups : 1) : BE_MAX_GROUPS);
}

size_t elem_workspace(int groups) { return sizeof(float) * (TABLE_FLOATS + (size_t)groups * ROW_FLOATS); }

int run_tables(const Sg2Weights& W, int eh, float* tables, int* all_zero, hipStream_t st) {
    hipLaunchKernelGGL(k_expert_tables, dim3(NE), dim3(64), 0, st, W, eh, tables, all_zero);
    SG_LAUNCH_CHECK("k_expert_tables");
    return 0;
}

// a.tables and a.partials are set here, from the workspace; the tables are there
template <bool FLAT>
int run_elem(ElemArgs& a, const Plan& pl, int groups, int eh, void* workspace, float* grads_out, hipStream_t st) {
    {
        static bool raised[64] = {};
        int dev = 0;
        SG_HIP_CHECK(hipGetDevice(&dev));
        if (dev < 0 || dev >= 64) return sg::fail("device index %d out of range", dev);
        if (!raised[dev]) {
            SG_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_bilevel_elem<FLAT>), hipFuncAttributeMaxDynamicSharedMemorySize, BE_LDS_BYTES));
            raised[dev] = true;
        }
    }
    float* tables = static_cast<float*>(workspace);
    a.tables = tables;
    a.partials = tables + TABLE_FLOATS;
    hipLaunchKernelGGL(k_bilevel_elem<FLAT>, dim3(groups), dim3(BE_THREADS), BE_LDS_BYTES, st, a, pl);
    SG_LAUNCH_CHECK("k_bilevel_elem");
    hipLaunchKernelGGL(k_elem_finish, dim3(FIN_DENSE + NE), dim3(64 * FIN_SLICES), 0, st, a.partials, groups, a.W, eh, grads_out, pl);
    SG_LAUNCH_CHECK("k_elem_finish");
    return 0;
}

}  // namespace

size_t bilevel_elem_workspace(int elem_tiles) { return elem_workspace(elem_groups((int64_t)elem_tiles * (ELEM_TILE / 64))); }
int launch_expert_tables(const Plan& pl, int eh, void* workspace, hipStream_t st) {
    return run_tables(pl.W, eh, static_cast<float*>(workspace), pl.contracted + 3, st);
}
int launch_bilevel_elem(const Plan& pl, const float* norms, int eh, float* smart_out, float* d_ctx, float* grads_out, void* workspace, hipStream_t st) {
    ElemArgs a = {};
    a.ctx = pl.ctx; a.smart = smart_out; a.d_ctx = d_ctx;
    a.total = pl.total; a.norms = norms; a.rescale = pl.rescale; a.W = pl.W;
    return run_elem<false>(a, pl, elem_groups((int64_t)pl.elem_tiles * (ELEM_TILE / 64)), eh, workspace, grads_out, st);
}
}  // namespace sg2

extern "C" {

size_t sg2_bilevel_elem_workspace_bytes(int64_t total) {
    if (total < 0) return 0;
    return sg2::elem_workspace(sg2::elem_groups((total + 63) / 64));
}

int sg2_bilevel_elem(const SgDims* dims, const Sg2Weights* weights, int64_t total, const float* grad, const float* sharpness,
                     const float* ctx, const float* gru_state, const float* cotangent, float rescale, float* smart_out,
                     float* d_ctx, float* grads_out, void* workspace, size_t workspace_bytes, void* stream) {
    return sg2_bilevel_elem_ex(dims, weights, total, grad, sharpness, ctx, gru_state, cotangent, rescale, smart_out, nullptr, d_ctx, grads_out,
                               workspace, workspace_bytes, stream);
}

int sg2_bilevel_elem_ex(const SgDims* dims, const Sg2Weights* weights, int64_t total, const float* grad, const float* sharpness,
                        const float* ctx, const float* gru_state, const float* cotangent, float rescale, float* smart_out,
                        float* gru_out, float* d_ctx, float* grads_out, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace sg2;
    hipStream_t st = (hipStream_t)stream;
    if (check_dims(dims, true)) return 1;
    if (!weights || !grads_out) return sg::fail("NULL argument");
    if (total < 0 || total > 0x7fffffffLL - BE_THREADS) return sg::fail("element count %lld out of range", (long long)total);
    for (int k = W_GRU_WZ; k < SG2_NUM_WEIGHTS; k++)
        if (!weights->w[k]) return sg::fail("weight pointer %d is NULL", k);
    const int groups = elem_groups((total + 63) / 64);
    if (!workspace || workspace_bytes < elem_workspace(groups))
        return sg::fail("workspace too small: need %zu bytes, got %zu", elem_workspace(groups), workspace_bytes);
    if (((uintptr_t)workspace & 127u) != 0) return sg::fail("workspace must be 128-byte aligned");
    if (total > 0) {
        if (!grad || !sharpness || !ctx || !gru_state || !cotangent || !d_ctx) return sg::fail("NULL argument");
        if ((((uintptr_t)ctx | (uintptr_t)gru_state | (uintptr_t)d_ctx | (uintptr_t)gru_out) & 15u) != 0)
            return sg::fail("ctx, gru_state, gru_out and d_ctx must be 16-byte aligned");
    }
    ElemArgs a = {};
    a.g = grad; a.s = sharpness; a.ctx = ctx; a.gru = gru_state; a.cot = cotangent;
    a.smart = smart_out; a.d_ctx = d_ctx; a.gru_out = gru_out;
    a.total = (int)total; a.rescale = rescale; a.W = *weights;
    if (run_tables(a.W, EH, static_cast<float*>(workspace), nullptr, st)) return 1;
    return run_elem<true>(a, Plan{}, groups, EH, workspace, grads_out, st);
}

}  // extern "C"
