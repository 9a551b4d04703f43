// Backward pass of the bidirectional Mamba-3 scan for the bilevel meta-net update of SuperGrok v2: given the
// gradient of the loss with respect to the two 8-float contexts of every element, the gradients with respect to
// the scan's weights.
//
// Stands in for the scan part of launch_mamba3_peer_backward[_batched]
// (csrc/supergrok2_mamba_peer_backward_kernels.cu:2512-3624 of the reference, called from
// grokking_optimizers/supergrok2.py:516-1330).  The forward pass is the production scan itself
// (sort + summaries + prefix + replay, carried states untouched), which additionally keeps the state entering every
// HT_STEP-th step; the per-element part of the meta-net (GRU, soft top-4 PEER routing, experts) is differentiated by
// sg2_bilevel_elem.hip (from torch operations for routing sizes that kernel is not built for).
//
// The adjoint state lambda obeys a linear recurrence over the scan steps in reverse.  Its transfer map contracts like
// the forward recurrence's, so it is not handed from chunk to chunk: k_adjoint gives every wave a range of steps of equal
// length, and the wave starts its walk behind the end of its range, at lambda = 0, as many steps as it takes for the
// map from there to fall below 2^-64 (the bound the forward summaries use; checked by the product of the steps' norms, and
// exact where the walk starts at the tensor's end).  Where the forward pass found a chunk whose map does not contract
// (Plan::contracted is 0) the ranges are the forward pass's chunks, and two more launches hand lambda over exactly:
//   k_adj_summary  per (chunk, direction): the affine map lambda_end-of-chunk -> lambda_start-of-chunk
//                  (a 2x2 matrix and an offset per lane), which needs only d y of every step, not the states;
//   k_adj_prefix   per (tensor, direction): composes the maps from the last chunk to the first, leaving the adjoint
//                  state that arrives at the end of every chunk.
// (They return at once in the usual case: handing lambda over that way cost 0.15 ms of the pass on 0.42 M elements.)
//
// A range is walked in tiles of 16 steps from the last to the first.  Per tile:
//   1  projections of the 16 steps from (g, s) and the composed coefficients, the incoming context gradients and
//      d out = out_proj^T d ctx, d y;
//   2  from the kept state at the tile's start, in blocks of four steps, last block first: the forward recurrence once more,
//      then the adjoint  lambda <- R(theta)^T diag(A_bar) (lambda + d y C)  with the gradients of dt, x-branch, B and C
//      per step (reduced over pairs / columns) and of A_log and the RoPE frequencies per lane;
//   3  per step and column: out, d z and the rest of d x-branch and d dt, and the sums over the tile's steps:
//      composed-coefficient gradients d v (x) (g, s, 1), d D, d out_proj.
// Gradients of the composed coefficients are carried back to input_proj / in_proj / dt_proj / B_proj / C_proj by a last
// one-workgroup kernel (k_compose_backward, the transpose of the composition).  Every wave keeps its sums in registers
// over the steps it handles and writes them to its own row of a partials buffer, which k_adj_sum_rows adds in a fixed
// order: the result is reproducible run to run.
// k_bilevel_backward is the form with the gradient of the input projection as a second output, chunk by chunk.
#include <algorithm>

#include "sg2_internal.hpp"
#include "../../include/sg2_compose.h"
#include "sg2_pair_sums.hpp"

namespace sg2 {
namespace {

constexpr int BST = SCAN_TT + 4;                 // row stride of the [16][64] LDS arrays
constexpr int ROWS = 16;
// LDS arrays of ROWS x BST floats
enum { A_DT, A_DSP, A_XB, A_B, A_C, A_GATE, A_DGATE, A_Y, A_DY, A_DZ, A_DXB, A_DDT, A_COUNT };
// k_bilevel_backward works on tiles of BT steps (half a forward tile), which keeps its LDS below half
// a CU's so that two workgroups share a CU.
constexpr int BT = 2 * HT_STEP;
constexpr int BBST = BT + 1;                     // row stride of its [16][BT] arrays (odd: the 16 rows a step reads hit 16 banks)
constexpr int LDS_ROWS_FLOATS = A_COUNT * ROWS * BBST;
constexpr int LDS_H_FLOATS = BT * SCAN_THREADS * 2;               // state after every step of the tile
constexpr int LDS_MISC_FLOATS = BT * DM + BT * 2 + DI;            // d ctx tile, (g, s) of the tile, per-column frequency bound
static_assert(SCAN_THREADS == 4 * BT && ROWS % 4 == 0 && (LDS_ROWS_FLOATS + LDS_H_FLOATS) % 4 == 0, "projection roles, float4 alignment");
constexpr int BILEVEL_LDS_BYTES = 4 * (LDS_ROWS_FLOATS + LDS_H_FLOATS + LDS_MISC_FLOATS);
// with the gradient of the input projection as an output: per-step sums over the columns of the B / C shares of each
// wave ([2 waves][BT][d B even, d B odd, d C even, d C odd][8 pairs]) and d(pre-activation row)/d x ([80][DM])
constexpr int LDS_DX_FLOATS = 2 * BT * 4 * HP + SG2_COMP_GROUPS * 16 * DM;
constexpr int BILEVEL_DX_LDS_BYTES = BILEVEL_LDS_BYTES + 4 * LDS_DX_FLOATS;

// What comes in and goes out besides the weight gradients.  Exactly one of d_ctx / d_scan is given.
struct AdjIO {
    const float* d_ctx;     // [2][total][DM]  gradient w.r.t. the two contexts, element order
    const float* d_scan[2]; // per direction [total][DI]  gradient w.r.t. the gated scan output (before out_proj), scan order
    const float* rx;        // [2][SG2_COMP_GROUPS*16][DM]  d(pre-activation row)/d x of each direction (only with dx)
    float* dx;              // [2][total][DM]  out, optional: each direction's gradient w.r.t. the input projection x, sorted order
};

// value of the lane whose index differs in one bit, by DPP where the pattern stays inside a row of 16 lanes
template <int CTRL>
__device__ __forceinline__ float dpp_get(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float xor_sum_columns(float v) {      // sum over the 8 columns of a wave (lanes 8 apart)
    v += dpp_get<0x128>(v);              // row_ror:8 = lane ^ 8
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    return v;
}
__device__ __forceinline__ float pair_sum(float v) {             // sum over the 8 pairs of a column (adjacent lanes)
    v += dpp_get<0xB1>(v);               // quad_perm [1,0,3,2] = lane ^ 1
    v += dpp_get<0x4E>(v);               // quad_perm [2,3,0,1] = lane ^ 2
    v += dpp_get<0x141>(v);              // row_half_mirror: lane 7-i of the 8; every quad already holds its sum
    return v;
}

// What a (chunk, direction) needs to find its steps.
struct ChunkRef {
    int ti, N, off, ustart, uend;
    bool has_s;
    const uint32_t* skey;
    const int32_t* sval;
    const float* ssrt;
    const float* dctx;
    const float* dscan;      // this tensor's rows of d_scan for this direction, indexed by scan step
};
__device__ __forceinline__ ChunkRef chunk_ref(const Plan& pl, int chunk, int dir, const AdjIO& io) {
    ChunkRef c;
    c.ti = sg::upper_seg(sg::as_const(pl.chunk_prefix), pl.P, chunk);
    const TensorDev& T = pl.tensors[c.ti];
    c.N = T.numel;
    c.off = T.off;
    c.ustart = (chunk - pl.chunk_prefix[c.ti]) * pl.chunk_len;
    c.uend = min(c.N, c.ustart + pl.chunk_len);
    c.has_s = pl.sharp_nonzero[c.ti] != 0;        // all-zero sharpness is never gathered into sorted order
    c.skey = pl.keys[0] + c.off;
    c.sval = pl.vals[0] + c.off;
    c.ssrt = pl.ssorted + c.off;
    c.dctx = io.d_ctx ? io.d_ctx + ((size_t)dir * pl.total + c.off) * DM : nullptr;
    c.dscan = io.d_scan[dir] ? io.d_scan[dir] + (size_t)c.off * DI : nullptr;
    return c;
}
// (g, s) and the element index of scan step u of a chunk's tensor; zeros past the end
__device__ __forceinline__ void load_step(const ChunkRef& c, int dir, int u, bool valid, float* g, float* s, int* orig) {
    *g = 0.0f; *s = 0.0f; *orig = 0;
    if (valid) {
        const int t = dir ? (c.N - 1 - u) : u;
        const int32_t v = c.sval[t];
        int o = v & 0x7fffffff;
        *orig = ((unsigned)o < (unsigned)c.N) ? o : 0;
        *g = sg_i2f((int32_t)c.skey[t] | (v & (int32_t)0x80000000));
        *s = c.has_s ? c.ssrt[t] : 0.0f;
    }
}

// sin/cos of a rotation angle; `tiny` (uniform over the workgroup) says that every angle of the tile is below the limit
// of the short polynomial pair, which the forward pass uses for such blocks as well
__device__ __forceinline__ void rot_sincos(bool tiny, float th, float* sn, float* cs) {
    if (tiny) sg_sincos_tiny(th, sn, cs); else sg_sincos(th, sn, cs);
}
// per column, the largest |rope frequency| of its 8 pairs (dt >= 0: dt*fmax bounds every angle of the column)
__device__ __forceinline__ void fill_fmax(float* s_fmax, const float* __restrict__ rope) {
    if (threadIdx.x < DI) {
        float m = 0.0f;
        for (int p = 0; p < HP; p++) m = sg_max(m, sg_abs(rope[threadIdx.x * HP + p]));
        s_fmax[threadIdx.x] = m;
    }
    __syncthreads();
}

// lambda -> R(theta)^T diag(A_bar) lambda for one lane's pair
__device__ __forceinline__ void adj_apply(float ae, float ao, float sn, float cs, float* xe, float* xo) {
    const float dre = *xe * ae, dro = *xo * ao;
    *xe = sg_fma(dre, cs, dro * sn);
    *xo = sg_fma(dro, cs, -(dre * sn));
}

// ---- affine map of the adjoint state across every chunk
constexpr int SUMM_ROWS = 4;                     // LDS arrays of the summary kernel: dt, C, gate, d y
__global__ __launch_bounds__(SCAN_THREADS) void k_adj_summary(Plan pl, AdjIO io, bool use_flag) {
    __shared__ float rows[SUMM_ROWS * ROWS * BST];
    __shared__ __attribute__((aligned(16))) float s_dctx[SCAN_TT * DM];
    __shared__ float s_fmax[DI];
    auto arr = [&](int a) { return rows + a * ROWS * BST; };
    const int chunk = blockIdx.x, dir = blockIdx.y;
    const ChunkRef c = chunk_ref(pl, chunk, dir, io);
    const int b = dir ? W_B_INPROJ : W_F_INPROJ;
    const float* __restrict__ Alog = pl.W.w[b + 5];
    const float* __restrict__ rope = pl.W.w[b + 7];
    const float* __restrict__ Wout = pl.W.w[b + 8];
    const float* __restrict__ comp = pl.comp + dir * (SG2_COMP_GROUPS * 16 * 3);
    const int tid = threadIdx.x;
    const int tu = tid & (SCAN_TT - 1), half = tid >> 6;
    const int j = tid >> 3, p = tid & 7;
    const float a_e = 0.5f * sg_exp(Alog[j * DS + 2 * p]), a_o = 0.5f * sg_exp(Alog[j * DS + 2 * p + 1]);
    const float freq = rope[j * HP + p];
    if (use_flag && *pl.contracted != 0) return;   // nobody reads the maps
    const bool in_order = sorted_rows(pl);
    if (chunk == pl.chunk_prefix[c.ti]) return;    // nothing lies before a tensor's first chunk: its map is never applied
    fill_fmax(s_fmax, rope);
    float u1e, u1o, u2e, u2o, ve, vo;
    const int ntiles = (c.uend - c.ustart + SCAN_TT - 1) / SCAN_TT;
    // The map contracts like the forward recurrence, so - as in the forward summary pass - the chunk is walked in blocks
    // of `window` steps, here from its start (the end of this reverse sweep): each block's map is taken from the identity
    // and applied after the map of everything before it ((U, v) <- (U_early U_block, U_early v_block + v_early)).  As soon as
    // every entry of the running matrix, in all 128 lanes, is below 2^-100, whatever arrives from later steps is multiplied
    // by less than that: the chunk's map is (0, v) and the walk stops.
    const int wtiles = (pl.window > 0 && pl.window < pl.chunk_len) ? max(1, pl.window / SCAN_TT) : ntiles;
    float e1e = 1.0f, e1o = 0.0f, e2e = 0.0f, e2o = 1.0f, eve = 0.0f, evo = 0.0f;     // map of the blocks before the current one
    bool have_early = false;
    for (int blk_tile0 = 0; blk_tile0 < ntiles; blk_tile0 += wtiles) {
      const int blk_last = min(ntiles, blk_tile0 + wtiles) - 1;
      u1e = 1.0f; u1o = 0.0f; u2e = 0.0f; u2o = 1.0f; ve = 0.0f; vo = 0.0f;
      for (int tile = blk_last; tile >= blk_tile0; tile--) {
        const int u0 = c.ustart + tile * SCAN_TT, cnt = min(SCAN_TT, c.uend - u0);
        bool small = true;
        {
            const bool valid = tu < cnt;
            float g, s;
            int orig;
            load_step(c, dir, u0 + tu, valid, &g, &s, &orig);
            if (c.dctx != nullptr) {
                const int at = in_order ? (dir ? c.N - 1 - (u0 + tu) : u0 + tu) : orig;
                const float4 dv = valid ? reinterpret_cast<const float4*>(c.dctx + (size_t)at * DM)[half] : make_float4(0.f, 0.f, 0.f, 0.f);
                reinterpret_cast<float4*>(s_dctx + tu * DM)[half] = dv;
            }
            for (int q = 0; q < ROWS / 2; q++) {
                const int r = half * (ROWS / 2) + q;
                const float dtv = valid ? sg_softplus(sg2_comp_eval(comp + (SG2_COMP_DT * 16 + r) * 3, g, s)) : 0.0f;
                small = small && (dtv * s_fmax[r] < SG_SINCOS_TINY_LIMIT);
                arr(0)[r * BST + tu] = dtv;
                arr(1)[r * BST + tu] = sg2_comp_eval(comp + (SG2_COMP_C * 16 + r) * 3, g, s);
                const float z = sg2_comp_eval(comp + (SG2_COMP_Z * 16 + r) * 3, g, s);
                arr(2)[r * BST + tu] = z * sg_sigmoid(z);
            }
        }
        const bool tiny = __syncthreads_and(small);
        for (int q = 0; q < ROWS / 2; q++) {
            const int r = half * (ROWS / 2) + q;
            float dout = 0.0f;
            if (c.dscan != nullptr) {
                if (tu < cnt) dout = c.dscan[(size_t)(u0 + tu) * DI + r];
            } else {
#pragma unroll
                for (int d = 0; d < DM; d++) dout = sg_fma(Wout[d * DI + r], s_dctx[tu * DM + d], dout);
            }
            arr(3)[r * BST + tu] = (tu < cnt) ? dout * arr(2)[r * BST + tu] : 0.0f;
        }
        __syncthreads();
        for (int k = cnt - 1; k >= 0; k--) {
            const float dt = arr(0)[j * BST + k], dy = arr(3)[j * BST + k];
            float ae, ao, sn, cs;
            sg_abar_pair(dt, a_e, a_o, &ae, &ao);
            rot_sincos(tiny, dt * freq, &sn, &cs);
            ve = sg_fma(dy, arr(1)[(2 * p) * BST + k], ve);
            vo = sg_fma(dy, arr(1)[(2 * p + 1) * BST + k], vo);
            adj_apply(ae, ao, sn, cs, &u1e, &u1o);
            adj_apply(ae, ao, sn, cs, &u2e, &u2o);
            adj_apply(ae, ao, sn, cs, &ve, &vo);
        }
        __syncthreads();
    }
      if (have_early) {     // (U, v) of this block after (E, ev) of the earlier ones: E U, E v + ev
          const float n1e = sg_fma(e1e, u1e, e2e * u1o), n1o = sg_fma(e1o, u1e, e2o * u1o);
          const float n2e = sg_fma(e1e, u2e, e2e * u2o), n2o = sg_fma(e1o, u2e, e2o * u2o);
          const float nve = sg_fma(e1e, ve, sg_fma(e2e, vo, eve)), nvo = sg_fma(e1o, ve, sg_fma(e2o, vo, evo));
          u1e = n1e; u1o = n1o; u2e = n2e; u2o = n2o; ve = nve; vo = nvo;
      }
      if (blk_last == ntiles - 1) break;      // the whole chunk is covered
      const float big = sg_max(sg_max(sg_abs(u1e), sg_abs(u1o)), sg_max(sg_abs(u2e), sg_abs(u2o)));
      if (__syncthreads_and(big < 0x1p-100f)) { u1e = u1o = u2e = u2o = 0.0f; break; }
      e1e = u1e; e1o = u1o; e2e = u2e; e2o = u2o; eve = ve; evo = vo;
      have_early = true;
    }
    float* out = pl.adj_summ + (((size_t)dir * pl.chunks + chunk) * SCAN_THREADS + tid) * 6;
    out[0] = u1e; out[1] = u1o; out[2] = u2e; out[3] = u2o; out[4] = ve; out[5] = vo;
}

// ---- adjoint state arriving at the end of every chunk, last chunk of a tensor first
__global__ __launch_bounds__(SCAN_THREADS) void k_adj_prefix(Plan pl, bool use_flag) {
    if (use_flag && *pl.contracted != 0) return;
    const int ti = blockIdx.x, dir = blockIdx.y, tid = threadIdx.x;
    const int base = pl.chunk_prefix[ti], nc = pl.chunk_prefix[ti + 1] - base;
    float le = 0.0f, lo = 0.0f;
    for (int c = nc - 1; c >= 0; c--) {
        const size_t at = ((size_t)dir * pl.chunks + base + c) * SCAN_THREADS + tid;
        pl.adj_lam[at * 2] = le;
        pl.adj_lam[at * 2 + 1] = lo;
        if (c == 0) break;
        const float* m = pl.adj_summ + at * 6;
        const float ne = sg_fma(m[0], le, sg_fma(m[2], lo, m[4]));
        const float no = sg_fma(m[1], le, sg_fma(m[3], lo, m[5]));
        le = ne;
        lo = no;
    }
}

// ---- the gradients, range by range
// One wave per (range, direction); eight per CU.  Lane roles within a tile: step st = lane % 16 with rows 4 (lane / 16) .. + 3
// of every 16-row group (projections, part 3), and column jl = lane / 8 and jl + 8 with RoPE pair p = lane % 8 (recurrence):
// the two columns share their B and C, the gradients of B and C add up over both before they go anywhere, and their
// sums against (g, s, 1) are 4 x 4 x 1 matrix instructions, one per step and entry.
// A tile of 16 whole steps whose inputs are small enough takes polynomials: softplus, SiLU and their derivatives as cubics
// around the constant of their row (sg2_taylor_ok), A_bar as a cubic, sin and cos as quadratics in d = dt - dt0 (remainders
// below 5e-8 while a d < 1/80, f d < 1/256; limits from compose_block).  Other tiles, and the ragged last one of a tensor, take the functions
// themselves.
// Bound by the vector ALU: 156 instructions per step (for its 256 states).  15.5 ms on 25 M
// elements, 0.33 ms on 0.42 M; 53.5 and 1.14 as one 128-lane workgroup per chunk with one wave per SIMD, the exact functions
// at every step and all states of a tile in LDS.
constexpr int AT = HT_STEP;             // steps per tile
constexpr int AB = 4;                   // steps per block
constexpr int FLUSH_TILES = 64;         // tiles between two writes of the sums
constexpr int ADJ_STRIDE = 4 * DI + 4;  // per step: (dt, dt - dt0, dt * x-branch, d y) of the 16 columns; later (d x-branch, d dt, d z, out)
constexpr int BC_STRIDE = 4 * HP + 4;   // per step: (B even, B odd, C even, C odd) of the 8 pairs
constexpr int SUM_STRIDE = AT + 4;      // per input: its values at the steps
constexpr int BLK_STRIDE = 64 * 4 + 4;  // per block of steps (the four blocks' reads of a column's step fall on different banks)
constexpr int IN_STRIDE = 13;           // per step: g, s, 1, d ctx[8]
typedef float adj_f32x4 __attribute__((ext_vector_type(4)));

// sigmoid and the derivative of SiLU as cubics around c (as sg2_softplus_taylor, sg2_silu_taylor)
__device__ __forceinline__ void sigmoid_taylor(float c, float t[4]) {
    const float s = sg_sigmoid(c), q = s * (1.0f - s), r = 1.0f - (s + s);
    t[0] = s;
    t[1] = q;
    t[2] = 0.5f * (q * r);
    t[3] = (q * sg_fma(r, r, -(q + q))) * 0.166666672f;
}
__device__ __forceinline__ void dsilu_taylor(float c, float t[4]) {
    const float s = sg_sigmoid(c), q = s * (1.0f - s), r = 1.0f - (s + s);
    const float a = sg_fma(r, sg_fma(c, r, 3.0f), -((c + c) * q));          // third derivative of SiLU over q
    t[0] = sg_fma(c, q, s);
    t[1] = q * sg_fma(c, r, 2.0f);
    t[2] = 0.5f * (q * a);
    t[3] = (q * (sg_fma(r, a, sg_fma(r, r, -8.0f * q)) - 6.0f * (c * q) * r)) * 0.166666672f;
}
__device__ __forceinline__ float cubic(const adj_f32x4 t, float d) { return sg_fma(sg_fma(sg_fma(t[3], d, t[2]), d, t[1]), d, t[0]); }

// Bound by the vector ALU: about 2500 instructions a tile of 16 steps at 4.1 clocks each and SIMD (two waves), of 20 600 clocks a
// tile blocks 12 900, states at their starts 2950, part 3 2700, projections 1650.  So that nothing of the tile loop spills at 256
// registers, what only part 3 needs lies in LDS (matrix accumulators; the pair sums where the states of their block were) and
// addresses are formed where they are used: a reload, or the spill of a prefetched value, waits for every load before it, and
// that was four memory latencies a tile (25 M elements 18.4 -> 16.2 ms).
template <bool SCAN_GRADS>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_adjoint(Plan pl, AdjIO io) {      // SCAN_GRADS: the gradient of the gated outputs comes in instead of that of the contexts
    static_assert(AT == 16 && DI == 16 && DS == 16 && HP == 8 && DM == 8 && AB == 4, "lane roles");
    __shared__ __attribute__((aligned(16))) float s_a[AT * ADJ_STRIDE];
    __shared__ __attribute__((aligned(16))) float s_b[AT * BC_STRIDE];
    __shared__ __attribute__((aligned(16))) float s_in[AT * IN_STRIDE + 4], s_gt[4 * SUM_STRIDE];      // inputs per step; g, s, 1 per row
    // per block of steps the lanes' states at its start; once these are read, the sums over the pairs of its steps: y,
    // d / d (dt * x-branch), d dt but for that, [16 columns][4 steps] each
    __shared__ __attribute__((aligned(16))) float s_h[(AT / AB) * BLK_STRIDE];
    // sums of part 3 (rows x (g, s, 1, d ctx): d x-branch, d dt, d z, out), a lane's matrix accumulators
    __shared__ __attribute__((aligned(16))) float s_acc[4 * 64 * 4];
    __shared__ __attribute__((aligned(16))) float s_k[2 * 64 * 4];                // gate and d out of the lanes' steps and rows, for part 3
    __shared__ __attribute__((aligned(16))) float s_coef[SG2_COMP_GROUPS * DI * 4];   // composed triples, D beside the x-branch's
    __shared__ __attribute__((aligned(16))) float s_tay[4 * DI * 4];              // dt, its derivative, gate, its derivative
    // (together 20 432 bytes: eight workgroups share a CU's 160 KB)

    const int lane = threadIdx.x, dir = blockIdx.y;
    const int st = lane & 15, rg = lane >> 4;
    const int jl = lane >> 3, p = lane & 7;
    const int b = dir ? W_B_INPROJ : W_F_INPROJ;
    const float* __restrict__ Wout = pl.W.w[b + 8];

    // ---- tables and the lane's constants
    {
        const float* comp = pl.comp + dir * (SG2_COMP_GROUPS * DI * 3);
        const float* tay = pl.comp + 2 * SG2_COMP_GROUPS * DI * 3 + dir * 2 * DI * 4;
        const float* Dw = pl.W.w[b + 6];
        for (int i = lane; i < SG2_COMP_GROUPS * DI; i += 64) {
            const float* t = comp + i * 3;
            *reinterpret_cast<adj_f32x4*>(s_coef + i * 4) = adj_f32x4{t[0], t[1], t[2], i / DI == SG2_COMP_XB ? Dw[i % DI] : 0.0f};
        }
        // (the forward pass's own polynomials for dt and gate)
        s_tay[lane] = tay[lane];
        s_tay[2 * DI * 4 + lane] = tay[DI * 4 + lane];
        if (lane < DI) {
            float t[4];
            sigmoid_taylor(comp[(SG2_COMP_DT * DI + lane) * 3 + 2], t);
            *reinterpret_cast<adj_f32x4*>(s_tay + (DI + lane) * 4) = adj_f32x4{t[0], t[1], t[2], t[3]};
            dsilu_taylor(comp[(SG2_COMP_Z * DI + lane) * 3 + 2], t);
            *reinterpret_cast<adj_f32x4*>(s_tay + (3 * DI + lane) * 4) = adj_f32x4{t[0], t[1], t[2], t[3]};
        }
        for (int i = lane; i < AT * IN_STRIDE + 4; i += 64) s_in[i] = 0.0f;
        for (int i = lane; i < 4 * SUM_STRIDE; i += 64) s_gt[i] = 0.0f;
        __syncthreads();
    }
    float pe[2][4], po[2][4], qs[2][3], qc[2][3];       // A_bar even / odd, sin, cos of the lane's two pairs as polynomials in dt - dt0
    float se[2], so[2], freq[2];                        // -a/2 of the two poles (a = -A/2), rotation frequency
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int j = jl + 8 * h;
        const float dt0 = s_tay[j * 4];
        const float a_e = 0.5f * sg_exp(pl.W.w[b + 5][j * DS + 2 * p]), a_o = 0.5f * sg_exp(pl.W.w[b + 5][j * DS + 2 * p + 1]);
        freq[h] = pl.W.w[b + 7][j * HP + p];
        se[h] = -0.5f * a_e;
        so[h] = -0.5f * a_o;
        sg2_abar_poly(dt0, a_e, pe[h]);
        sg2_abar_poly(dt0, a_o, po[h]);
        sg2_sincos_poly(dt0, freq[h], qs[h], qc[h]);
    }
    const float wo0 = Wout[rg * DI + st], wo1 = Wout[(4 + rg) * DI + st];      // operand of d out = out_proj^T d ctx
    const sg::cfloat_p lim = sg::as_const(pl.comp) + 2 * SG2_COMP_GROUPS * DI * 3 + 2 * 2 * DI * 4;
    const float cmax_g = lim[2 * dir], cmax_s = lim[2 * dir + 1], kcub_g = lim[12 + 2 * dir], kcub_s = lim[13 + 2 * dir];

    // ---- sums
    const adj_f32x4 zero4 = adj_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float al_e[2] = {0.0f, 0.0f}, al_o[2] = {0.0f, 0.0f}, rope[2] = {0.0f, 0.0f};
    adj_f32x4 aBe = zero4, aBo = zero4, aCe = zero4, aCo = zero4;
    adj_f32x4* const acc16 = reinterpret_cast<adj_f32x4*>(s_acc) + lane;
#pragma unroll
    for (int q = 0; q < 4; q++) acc16[64 * q] = zero4;
    float accD[4] = {0.0f, 0.0f, 0.0f, 0.0f};

    // this wave's sums -> its row of the partials buffer, every FLUSH_TILES tiles: one chain of additions over all of a
    // wave's steps would lose two digits of the sums of B and C where these nearly cancel (an entry is always the same lane's)
    float* const row = pl.adj_part + ((size_t)dir * gridDim.x + blockIdx.x) * SG2_BWD_STRIDE;
    for (int i = lane; i < SG2_BWD_STRIDE; i += 64) row[i] = 0.0f;
    __syncthreads();
    int unflushed = 0;
    auto flush = [&]() {
        float* const g_comp = row;
        float* const g_alog = g_comp + SG2_COMP_GROUPS * DI * 3;
        float* const g_rope = g_alog + DI * DS;
        float* const g_D = g_rope + DI * HP;
        float* const g_wout = g_D + DI;
        adj_f32x4 a16[4];
#pragma unroll
        for (int q = 0; q < 4; q++) { a16[q] = acc16[64 * q]; acc16[64 * q] = zero4; }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int j = jl + 8 * h;
            g_alog[j * DS + 2 * p] += al_e[h] * se[h];
            g_alog[j * DS + 2 * p + 1] += al_o[h] * so[h];
            g_rope[j * HP + p] += rope[h];
            al_e[h] = al_o[h] = rope[h] = 0.0f;
        }
#pragma unroll
        for (int v = 0; v < 4; v++) {
            // 16 x 16: rows 4 rg + v, column st
            if (st < 3) {
                g_comp[(SG2_COMP_XB * DI + 4 * rg + v) * 3 + st] += a16[0][v];
                g_comp[(SG2_COMP_DT * DI + 4 * rg + v) * 3 + st] += a16[1][v];
                g_comp[(SG2_COMP_Z * DI + 4 * rg + v) * 3 + st] += a16[2][v];
            } else if (st < 3 + DM) {
                g_wout[(st - 3) * DI + 4 * rg + v] += a16[3][v];
            }
            // 4 x 4: the pair of lane 4 (lane / 4) + v against column lane % 4; added over the columns jl
            auto over_columns = [](float x) {
                x += __shfl_xor(x, 8, 64);
                x += __shfl_xor(x, 16, 64);
                return x + __shfl_xor(x, 32, 64);
            };
            const float sums[4] = {over_columns(aBe[v]), over_columns(aBo[v]), over_columns(aCe[v]), over_columns(aCo[v])};
            if (lane < 8 && (lane & 3) < 3) {
                const int pr = (lane & 4) + v;
#pragma unroll
                for (int q = 0; q < 4; q++) g_comp[((q < 2 ? SG2_COMP_B : SG2_COMP_C) * DI + 2 * pr + (q & 1)) * 3 + (lane & 3)] += sums[q];
            }
            float d = accD[v];
#pragma unroll
            for (int m = 8; m >= 1; m >>= 1) d += __shfl_xor(d, m, 64);
            if (st == 0) g_D[4 * rg + v] += d;
        }
        aBe = aBo = aCe = aCo = zero4;
#pragma unroll
        for (int q = 0; q < 4; q++) accD[q] = 0.0f;
        unflushed = 0;
    };

    // ---- the tensor at hand
    int ti = 0, N = 0, off = 0;
    bool has_s = false;
    float le[2] = {0.0f, 0.0f}, lo[2] = {0.0f, 0.0f};
    const float* dctx = nullptr;
    const float* dscan = nullptr;

    const bool in_order = sorted_rows(pl);
    // what a tile reads from memory, requested one tile ahead
    struct Inputs { uint32_t key; int32_t val; float s, d0, d1; adj_f32x4 ds, h; };
    auto request = [&](int u0, bool with_state) {
        Inputs in = {0, 0, 0.0f, 0.0f, 0.0f, zero4, zero4};
        // (opaque: a lane's addresses, formed ahead of the loop, would spill, and their reload waits for every load before it)
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int st = ln & 15, rg = ln >> 4, u = min(u0 + st, N - 1);      // (steps past the end: unpack and project leave them out)
        const int t = dir ? N - 1 - u : u;
        in.key = pl.keys[0][off + t];
        in.val = pl.vals[0][off + t];
        if (has_s) in.s = pl.ssorted[off + t];
        if (SCAN_GRADS) {
            in.ds = *reinterpret_cast<const adj_f32x4*>(dscan + (size_t)u * DI + 4 * rg);
        } else {
            int at = t;
            if (!in_order) {      // (kept a branch: a choice would wait for the index here)
                asm volatile("");
                at = min(in.val & 0x7fffffff, N - 1);
            }
            in.d0 = dctx[(size_t)at * DM + rg];
            in.d1 = dctx[(size_t)at * DM + 4 + rg];
        }
        if (with_state) {
            const float* ht = pl.htile + ((size_t)dir * htile_count(pl.total, pl.P) + htile_index(off, ti, u0)) * 2 * SCAN_THREADS;
            in.h = adj_f32x4{ht[ln], ht[SCAN_THREADS + ln], ht[64 + ln], ht[SCAN_THREADS + 64 + ln]};
        }
        return in;
    };

    // A_bar, sin, cos of the lane's pair h
    auto coefficients = [&](auto fast_c, int h, float dt, float d, float& ae, float& ao, float& sn, float& cs) {
        if (decltype(fast_c)::value) {
            ae = sg2_poly3(pe[h], d);
            ao = sg2_poly3(po[h], d);
            sn = sg2_poly2(qs[h], d);
            cs = sg2_poly2(qc[h], d);
        } else {
            sg_abar_pair(dt, -2.0f * se[h], -2.0f * so[h], &ae, &ao);
            sg_sincos(dt * freq[h], &sn, &cs);
        }
    };

    // operands of a step of the recurrence: its two columns, its B and C.  They are fetched one step ahead, and fetched_here()
    // keeps the compiler from moving a fetch down to where it is used (with registers scarce it does, and waits each time).
    struct Step { adj_f32x4 a[2], bc; };
    auto step_at = [&](int k) {
        Step o;
        o.a[0] = *reinterpret_cast<const adj_f32x4*>(s_a + k * ADJ_STRIDE + 4 * jl);
        o.a[1] = *reinterpret_cast<const adj_f32x4*>(s_a + k * ADJ_STRIDE + 4 * jl + 32);
        o.bc = *reinterpret_cast<const adj_f32x4*>(s_b + k * BC_STRIDE + 4 * p);
        return o;
    };
    auto fetched_here = []() { asm volatile("" ::: "memory"); };

    // part 1 -> s_a, s_b, s_in, s_gt; gate and d out of the lane's step and rows -> s_k
    struct Rows { float g, s; bool valid; };
    auto project = [&](auto fast_c, const Inputs& in, int cnt, float g, float s) {
        constexpr bool FAST = decltype(fast_c)::value;
        Rows R;
        R.g = g; R.s = s; R.valid = st < cnt;
        adj_f32x4 dout = in.ds;
        if (!SCAN_GRADS) {
            dout = __builtin_amdgcn_mfma_f32_16x16x4f32(wo0, in.d0, zero4, 0, 0, 0);
            dout = __builtin_amdgcn_mfma_f32_16x16x4f32(wo1, in.d1, dout, 0, 0, 0);
        }
        if (rg == 0) {
            s_gt[st] = g; s_gt[SUM_STRIDE + st] = s; s_gt[2 * SUM_STRIDE + st] = R.valid ? 1.0f : 0.0f;
            s_in[st * IN_STRIDE] = g; s_in[st * IN_STRIDE + 1] = s; s_in[st * IN_STRIDE + 2] = R.valid ? 1.0f : 0.0f;
        }
        s_in[st * IN_STRIDE + 3 + rg] = in.d0;
        s_in[st * IN_STRIDE + 7 + rg] = in.d1;
        float B[4], C[4];
        adj_f32x4 gate;
        auto eval = [&](const adj_f32x4 c) { return sg_fma(c[0], g, sg_fma(c[1], s, c[2])); };
#pragma unroll
        for (int v0 = 0; v0 < 4; v0 += 2) {
            adj_f32x4 c[2][SG2_COMP_GROUPS], td[2], tg[2];
#pragma unroll
            for (int v = 0; v < 2; v++) {
                const int row = 4 * rg + v0 + v;
#pragma unroll
                for (int q = 0; q < SG2_COMP_GROUPS; q++) c[v][q] = *reinterpret_cast<const adj_f32x4*>(s_coef + (q * DI + row) * 4);
                td[v] = *reinterpret_cast<const adj_f32x4*>(s_tay + row * 4);
                tg[v] = *reinterpret_cast<const adj_f32x4*>(s_tay + (2 * DI + row) * 4);
            }
            fetched_here();
#pragma unroll
            for (int v = v0; v < v0 + 2; v++) {
                const adj_f32x4 (&cv)[SG2_COMP_GROUPS] = c[v - v0];
                const adj_f32x4 cd = cv[SG2_COMP_DT], cz = cv[SG2_COMP_Z];
                float dt;
                if (FAST) {
                    dt = cubic(td[v - v0], sg_fma(cd[0], g, cd[1] * s));
                    gate[v] = cubic(tg[v - v0], sg_fma(cz[0], g, cz[1] * s));
                } else {
                    dt = R.valid ? sg_softplus(eval(cd)) : 0.0f;
                    const float z = eval(cz);
                    gate[v] = z * sg_sigmoid(z);
                    if (!R.valid) dout[v] = 0.0f;
                }
                const float xb = FAST || R.valid ? eval(cv[SG2_COMP_XB]) : 0.0f;
                B[v] = eval(cv[SG2_COMP_B]);
                C[v] = eval(cv[SG2_COMP_C]);
                *reinterpret_cast<adj_f32x4*>(s_a + st * ADJ_STRIDE + 4 * (4 * rg + v)) = adj_f32x4{dt, FAST ? dt - td[v - v0][0] : dt, dt * xb, dout[v] * gate[v]};
            }
        }
        reinterpret_cast<adj_f32x4*>(s_k)[lane] = gate;
        reinterpret_cast<adj_f32x4*>(s_k)[64 + lane] = dout;
        *reinterpret_cast<adj_f32x4*>(s_b + st * BC_STRIDE + 8 * rg) = adj_f32x4{B[0], B[1], C[0], C[1]};
        *reinterpret_cast<adj_f32x4*>(s_b + st * BC_STRIDE + 8 * rg + 4) = adj_f32x4{B[2], B[3], C[2], C[3]};
        __syncthreads();       // one wave: no s_barrier is issued, the LDS writes above are ordered before the reads below
        return R;
    };
    // (g, s) of the lane's step, and whether the whole tile may take the polynomials
    auto unpack = [&](const Inputs& in, int cnt, float& g, float& s) {
        const bool valid = st < cnt;
        g = valid ? sg_i2f((int32_t)in.key | (in.val & (int32_t)0x80000000)) : 0.0f;
        s = valid ? in.s : 0.0f;
        return cnt == AT && __builtin_amdgcn_ballot_w64(!(sg2_taylor_ok(cmax_g, cmax_s, g, s) && sg2_poly_ok(kcub_g, kcub_s, g, s))) == 0;
    };

    // lambda alone, from step v_end (0 there) to u_end; bound: product of the norms of the steps' maps
    auto approach = [&](int v_end, int u_end, float& bound) {
        float bd[2] = {1.0f, 1.0f};
        le[0] = le[1] = lo[0] = lo[1] = 0.0f;
        const int first = u_end, last = first + ((v_end - first - 1) / AT) * AT;
        Inputs next = request(last, false);
        for (int u0 = last; u0 >= first; u0 -= AT) {
            const Inputs in = next;
            if (u0 > first) next = request(u0 - AT, false);
            const int cnt = min(AT, v_end - u0);
            float g, s;
            const bool fast = unpack(in, cnt, g, s);
            auto walk = [&](auto fast_c) {
                project(fast_c, in, cnt, g, s);
                Step o = step_at(cnt - 1);
#pragma unroll 2
                for (int k = cnt - 1; k >= 0; k--) {
                    const Step now = o;
                    o = step_at(max(k - 1, 0));
                    fetched_here();
                    const adj_f32x4 bc = now.bc;
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const adj_f32x4 a = now.a[h];
                        float ae, ao, sn, cs;
                        coefficients(fast_c, h, a[0], a[1], ae, ao, sn, cs);
                        const float dre = sg_fma(a[3], bc[2], le[h]) * ae, dro = sg_fma(a[3], bc[3], lo[h]) * ao;
                        le[h] = sg_fma(dre, cs, dro * sn);
                        lo[h] = sg_fma(dro, cs, -(dre * sn));
                        bd[h] *= sg_max(sg_abs(ae), sg_abs(ao));
                    }
                }
            };
            if (fast) walk(std::true_type{});
            else walk(std::false_type{});
            __syncthreads();
        }
        bound = sg_max(bd[0], bd[1]);
    };

    // the gradients of steps [u_lo, u_hi), lambda behind them given; u_lo is a multiple of AT
    auto range = [&](int u_lo, int u_hi) {
        const int last = u_lo + ((u_hi - u_lo - 1) / AT) * AT;
        Inputs next = request(last, true);
        for (int u0 = last; u0 >= u_lo; u0 -= AT) {
            const Inputs in = next;
            if (u0 > u_lo) next = request(u0 - AT, true);
            const int cnt = min(AT, u_hi - u0);
            float g, s;
            const bool fast = unpack(in, cnt, g, s);
            auto walk = [&](auto fast_c) {
                constexpr bool FAST = decltype(fast_c)::value;
                const Rows R = project(fast_c, in, cnt, g, s);
                // ---- 2: states at the starts of the blocks
                adj_f32x4* const sh = reinterpret_cast<adj_f32x4*>(s_h) + lane;
                {
                    adj_f32x4 hh = in.h;
                    sh[0] = hh;
                    Step o = step_at(0);
#pragma unroll 1
                    for (int k0 = 0; k0 < AT - AB; k0 += AB) {
#pragma unroll
                        for (int u = 0; u < AB; u++) {
                            const Step now = o;
                            o = step_at(k0 + u + 1);
                            fetched_here();
                            const adj_f32x4 bc = now.bc;
#pragma unroll
                            for (int h = 0; h < 2; h++) {
                                const adj_f32x4 a = now.a[h];
                                float ae, ao, sn, cs;
                                coefficients(fast_c, h, a[0], a[1], ae, ao, sn, cs);
                                const float re = sg_fma(hh[2 * h], cs, -(hh[2 * h + 1] * sn)), ro = sg_fma(hh[2 * h + 1], cs, hh[2 * h] * sn);
                                hh[2 * h] = sg_fma(ae, re, a[2] * bc[0]);
                                hh[2 * h + 1] = sg_fma(ao, ro, a[2] * bc[1]);
                            }
                        }
                        sh[(k0 / AB + 1) * (BLK_STRIDE / 4)] = hh;
                    }
                }
                // ---- the blocks, last first (a ragged tile: its steps past the end leave lambda alone and add nothing, their
                // dt, x-branch and d y being 0)
                Step o = step_at(AT - AB);
                adj_f32x4 h_next = sh[(AT / AB - 1) * (BLK_STRIDE / 4)];
#pragma unroll 1
                for (int k0 = AT - AB; k0 >= 0; k0 -= AB) {
                    const adj_f32x4 h0 = h_next;
                    float ae[2][AB], ao[2][AB], sn[2][AB], cs[2][AB], re[2][AB], ro[2][AB], he[2][AB + 1], ho[2][AB + 1];
                    float y[8];
                    he[0][0] = h0[0]; ho[0][0] = h0[1]; he[1][0] = h0[2]; ho[1][0] = h0[3];
#pragma unroll
                    for (int u = 0; u < AB; u++) {
                        const Step now = o;
                        if (u < AB - 1) {
                            o = step_at(k0 + u + 1);
                            fetched_here();
                        }
                        const adj_f32x4 bc = now.bc;
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const adj_f32x4 a = now.a[h];
                            coefficients(fast_c, h, a[0], a[1], ae[h][u], ao[h][u], sn[h][u], cs[h][u]);
                            re[h][u] = sg_fma(he[h][u], cs[h][u], -(ho[h][u] * sn[h][u]));
                            ro[h][u] = sg_fma(ho[h][u], cs[h][u], he[h][u] * sn[h][u]);
                            he[h][u + 1] = sg_fma(ae[h][u], re[h][u], a[2] * bc[0]);
                            ho[h][u + 1] = sg_fma(ao[h][u], ro[h][u], a[2] * bc[1]);
                            y[4 * h + u] = sg_fma(ho[h][u + 1], bc[3], he[h][u + 1] * bc[2]);
                        }
                    }
                    // (the operands of the four steps are fetched again below, from the last, still at hand, down: held they would spill)
                    const adj_f32x4 gt = *reinterpret_cast<const adj_f32x4*>(s_gt + (lane & 3) * SUM_STRIDE + k0);
                    fetched_here();
                    block_pair_sums<HP>(y);
                    // lanes p = 0 hold the sums of column jl, p = 4 those of column jl + 8 (the block's state has been read)
                    adj_f32x4* const sums = reinterpret_cast<adj_f32x4*>(s_h + k0 / AB * BLK_STRIDE) + jl + 2 * p;
                    if ((p & 3) == 0) sums[0] = adj_f32x4{y[0], y[1], y[2], y[3]};
                    float q[8], dd[8];
#pragma unroll
                    for (int u = AB - 1; u >= 0; u--) {
                        float tBe = 0.0f, tBo = 0.0f, tCe = 0.0f, tCo = 0.0f;
                        const Step now = o;
                        o = step_at(max(u > 0 ? k0 + u - 1 : k0 - AB, 0));
                        if (u == 0) h_next = sh[max(k0 / AB - 1, 0) * (BLK_STRIDE / 4)];
                        fetched_here();
                        const adj_f32x4 bc = now.bc;
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const adj_f32x4 a = now.a[h];
                            const float dt = a[0], ux = a[2], dy = a[3];
                            // y = sum h C
                            const float l_e = sg_fma(dy, bc[2], le[h]), l_o = sg_fma(dy, bc[3], lo[h]);
                            tCe = sg_fma(dy, he[h][u + 1], tCe);
                            tCo = sg_fma(dy, ho[h][u + 1], tCo);
                            // h' = A_bar * rot(h) + dt * xb * B
                            tBe = sg_fma(l_e, ux, tBe);
                            tBo = sg_fma(l_o, ux, tBo);
                            q[4 * h + u] = sg_fma(l_e, bc[0], l_o * bc[1]);
                            // A_bar = 2/(1 + a dt) - 1: dA_bar/d dt = -a/2 (A_bar + 1)^2 (x + x A_bar, twice, each one rounding)
                            const float xe = l_e * re[h][u], xo = l_o * ro[h][u];
                            const float we = sg_fma(xe, ae[h][u], xe), wo = sg_fma(xo, ao[h][u], xo);
                            const float te = sg_fma(we, ae[h][u], we), to = sg_fma(wo, ao[h][u], wo);
                            al_e[h] = sg_fma(te, dt, al_e[h]);
                            al_o[h] = sg_fma(to, dt, al_o[h]);
                            // lambda for the previous step; d theta = d ro * re - d re * ro
                            const float dre = l_e * ae[h][u], dro = l_o * ao[h][u];
                            const float dth = sg_fma(dro, re[h][u], -(dre * ro[h][u]));
                            rope[h] = sg_fma(dth, dt, rope[h]);
                            dd[4 * h + u] = sg_fma(dth, freq[h], sg_fma(te, se[h], to * so[h]));
                            const float n_e = sg_fma(dre, cs[h][u], dro * sn[h][u]), n_o = sg_fma(dro, cs[h][u], -(dre * sn[h][u]));
                            le[h] = FAST || k0 + u < cnt ? n_e : le[h];
                            lo[h] = FAST || k0 + u < cnt ? n_o : lo[h];
                        }
                        aBe = __builtin_amdgcn_mfma_f32_4x4x1f32(tBe, gt[u], aBe, 0, 0, 0);
                        aBo = __builtin_amdgcn_mfma_f32_4x4x1f32(tBo, gt[u], aBo, 0, 0, 0);
                        aCe = __builtin_amdgcn_mfma_f32_4x4x1f32(tCe, gt[u], aCe, 0, 0, 0);
                        aCo = __builtin_amdgcn_mfma_f32_4x4x1f32(tCo, gt[u], aCo, 0, 0, 0);
                    }
                    block_pair_sums<HP>(q);
                    block_pair_sums<HP>(dd);
                    if ((p & 3) == 0) {
                        sums[DI] = adj_f32x4{q[0], q[1], q[2], q[3]};
                        sums[2 * DI] = adj_f32x4{dd[0], dd[1], dd[2], dd[3]};
                    }
                }
                __syncthreads();
                // ---- 3
                int ln = lane;         // (opaque, as in request)
                asm volatile("" : "+v"(ln));
                const int st = ln & 15, rg = ln >> 4;
                const float* const sums = s_h + (st >> 2) * BLK_STRIDE + (st & 3);
                const adj_f32x4 gate = reinterpret_cast<adj_f32x4*>(s_k)[ln], dout = reinterpret_cast<adj_f32x4*>(s_k)[64 + ln];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int row = 4 * rg + v;
                    const float yv = sums[AB * row], qb = sums[AB * (DI + row)], ddr = sums[AB * (2 * DI + row)];
                    const float dt = s_a[st * ADJ_STRIDE + 4 * row];
                    const adj_f32x4 cd = *reinterpret_cast<const adj_f32x4*>(s_coef + (SG2_COMP_DT * DI + row) * 4);
                    const adj_f32x4 cz = *reinterpret_cast<const adj_f32x4*>(s_coef + (SG2_COMP_Z * DI + row) * 4);
                    const adj_f32x4 cx = *reinterpret_cast<const adj_f32x4*>(s_coef + (SG2_COMP_XB * DI + row) * 4);
                    const adj_f32x4 td = *reinterpret_cast<const adj_f32x4*>(s_tay + (DI + row) * 4);
                    const adj_f32x4 tg = *reinterpret_cast<const adj_f32x4*>(s_tay + (3 * DI + row) * 4);
                    fetched_here();
                    const float D = cx[3], xb = FAST || R.valid ? sg_fma(cx[0], R.g, sg_fma(cx[1], R.s, cx[2])) : 0.0f;
                    float dsp, dgate;
                    if (FAST) {
                        dsp = cubic(td, sg_fma(cd[0], R.g, cd[1] * R.s));
                        dgate = cubic(tg, sg_fma(cz[0], R.g, cz[1] * R.s));
                    } else {
                        const float raw = sg_fma(cd[0], R.g, sg_fma(cd[1], R.s, cd[2])), z = sg_fma(cz[0], R.g, sg_fma(cz[1], R.s, cz[2]));
                        const float sz = sg_sigmoid(z);
                        dsp = raw > 20.0f ? 1.0f : sg_sigmoid(raw);
                        dgate = sz * sg_fma(z, 1.0f - sz, 1.0f);
                    }
                    accD[v] = sg_fma(dout[v], xb, accD[v]);
                    adj_f32x4 out = adj_f32x4{sg_fma(qb, dt, dout[v] * D), sg_fma(qb, xb, ddr) * dsp, (dout[v] * yv) * dgate,
                                              sg_fma(yv, gate[v], D * xb)};
                    if (!FAST && !R.valid) out = zero4;
                    *reinterpret_cast<adj_f32x4*>(s_a + st * ADJ_STRIDE + 4 * row) = out;
                }
                __syncthreads();
                adj_f32x4 a16[4];
#pragma unroll
                for (int q = 0; q < 4; q++) a16[q] = acc16[64 * q];
#pragma unroll
                for (int t = 0; t < AT / 4; t++) {
                    const adj_f32x4 d = *reinterpret_cast<const adj_f32x4*>(s_a + (4 * t + rg) * ADJ_STRIDE + 4 * st);      // step 4 t + rg, row st
                    const float in16 = s_in[(4 * t + rg) * IN_STRIDE + st];
#pragma unroll
                    for (int q4 = 0; q4 < 4; q4++) a16[q4] = __builtin_amdgcn_mfma_f32_16x16x4f32(d[q4], in16, a16[q4], 0, 0, 0);
                }
#pragma unroll
                for (int q = 0; q < 4; q++) acc16[64 * q] = a16[q];
                __syncthreads();
            };
            if (fast) walk(std::true_type{});
            else walk(std::false_type{});
            if (++unflushed == FLUSH_TILES) flush();
        }
    };

    auto set_tensor = [&](int i) {
        ti = i;
        const TensorDev& T = pl.tensors[i];
        N = __builtin_amdgcn_readfirstlane(T.numel);
        off = __builtin_amdgcn_readfirstlane(T.off);
        has_s = __builtin_amdgcn_readfirstlane(pl.sharp_nonzero[i]) != 0;
        dctx = io.d_ctx ? io.d_ctx + ((size_t)dir * pl.total + off) * DM : nullptr;
        dscan = io.d_scan[dir] ? io.d_scan[dir] + (size_t)off * DI : nullptr;
    };
    // Usual case: the tiles of all tensors in one row (a tensor takes whole elementwise tiles of it), an equal part to every
    // wave.  Else the chunks of the forward pass, every gridDim.x-th.
    constexpr int PER = ELEM_TILE / AT;
    const bool parts = __builtin_amdgcn_readfirstlane(pl.contracted[0]) != 0;
    const int first_block = __builtin_amdgcn_readfirstlane(pl.contracted[1]);
    const int64_t tiles = (int64_t)pl.elem_tiles * PER;
    int at = parts ? (int)(tiles * blockIdx.x / gridDim.x) : (int)blockIdx.x;
    const int end = parts ? (int)(tiles * (blockIdx.x + 1) / gridDim.x) : pl.chunks;
    while (at < end) {
        int u_lo, u_hi;
        const sg::Seg seg = sg::find_seg(sg::as_const(parts ? pl.elem_tile_prefix : pl.chunk_prefix), pl.P, parts ? at / PER : at);
        set_tensor(seg.i);
        le[0] = le[1] = lo[0] = lo[1] = 0.0f;
        int from, far;                     // where the walk to u_hi starts, and where it starts if that was not far enough
        if (parts) {
            const int stop = min(end, seg.end * PER);
            u_lo = (at - seg.first * PER) * AT;
            u_hi = min((stop - seg.first * PER) * AT, N);
            at = stop;
            // two chunk lengths hold a whole chunk of the forward pass, whose map is known to contract
            far = min(N, u_hi + 2 * pl.chunk_len);
            from = first_block > 0 ? min(far, u_hi + (first_block + AT - 1) / AT * AT) : far;
        } else {
            u_lo = (at - seg.first) * pl.chunk_len;
            u_hi = min(N, u_lo + pl.chunk_len);
            from = far = u_hi;
            const float* lam = pl.adj_lam + ((size_t)dir * pl.chunks + at) * SCAN_THREADS * 2;
            if (u_hi < N) {
#pragma unroll
                for (int h = 0; h < 2; h++) { le[h] = lam[(lane + 64 * h) * 2]; lo[h] = lam[(lane + 64 * h) * 2 + 1]; }
            }
            at += (int)gridDim.x;
        }
        if (u_lo >= u_hi) continue;        // an empty rest of a tensor's last elementwise tile
        while (from > u_hi) {
            float bound;
            approach(from, u_hi, bound);
            if (from == far || __builtin_amdgcn_ballot_w64(!(bound < SG2_FORGOTTEN)) == 0) break;
            from = far;
        }
        range(u_lo, u_hi);
    }

    flush();
}

// ---- the gradients with the gradient of the input projection, chunk by chunk: one 128-lane workgroup per (chunk,
// direction), lane (j,p) owning column j and RoPE pair p
__global__ __launch_bounds__(SCAN_THREADS) void k_bilevel_backward(Plan pl, AdjIO io) {
    constexpr bool DX = true;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float* rows = lds;
    float* sH = lds + LDS_ROWS_FLOATS;
    float* s_dctx = sH + LDS_H_FLOATS;
    float* s_gs = s_dctx + BT * DM;
    float* s_fmax = s_gs + BT * 2;
    float* s_bc = s_fmax + DI;                       // DX only
    float* s_rx = s_bc + 2 * BT * 4 * HP;            // DX only
    auto arr = [&](int a) { return rows + a * ROWS * BBST; };

    const int dir = blockIdx.y;
    const int b = dir ? W_B_INPROJ : W_F_INPROJ;
    const float* __restrict__ Alog = pl.W.w[b + 5];
    const float* __restrict__ Dw = pl.W.w[b + 6];
    const float* __restrict__ rope = pl.W.w[b + 7];
    const float* __restrict__ Wout = pl.W.w[b + 8];
    const float* __restrict__ comp = pl.comp + dir * (SG2_COMP_GROUPS * 16 * 3);

    const int tid = threadIdx.x;
    const int tu = tid & (BT - 1), part = tid >> 5;               // projection role: step tu, rows 4*part .. 4*part+3
    const int j = tid >> 3, p = tid & 7, w = tid >> 6;             // recurrence role
    const float a_e = 0.5f * sg_exp(Alog[j * DS + 2 * p]), a_o = 0.5f * sg_exp(Alog[j * DS + 2 * p + 1]);
    const float freq = rope[j * HP + p];

    if (DX) {
        for (int i = threadIdx.x; i < SG2_COMP_GROUPS * 16 * DM; i += SCAN_THREADS) s_rx[i] = io.rx[(size_t)dir * SG2_COMP_GROUPS * 16 * DM + i];
    }
    fill_fmax(s_fmax, rope);
    // this lane's rows of the composed coefficients, of out_proj^T and of D, kept in registers: the barriers inside
    // the tile loop would otherwise make every tile fetch them again
    float cw[SG2_COMP_GROUPS][ROWS / 4][3], wo[ROWS / 4][DM], dwr[ROWS / 4];
#pragma unroll
    for (int q = 0; q < ROWS / 4; q++) {
        const int r = part * (ROWS / 4) + q;
#pragma unroll
        for (int gq = 0; gq < SG2_COMP_GROUPS; gq++)
#pragma unroll
            for (int e = 0; e < 3; e++) cw[gq][q][e] = comp[(gq * 16 + r) * 3 + e];
#pragma unroll
        for (int d = 0; d < DM; d++) wo[q][d] = Wout[d * DI + r];
        dwr[q] = Dw[r];
    }
    float acc_alog_e = 0.0f, acc_alog_o = 0.0f, acc_rope = 0.0f;
    float acc_c0 = 0.0f, acc_c1 = 0.0f, acc_c2 = 0.0f, acc_D = 0.0f, acc_wout = 0.0f;
    float acc_bc[12];                 // this lane's column share of d B[2p], d B[2p+1], d C[2p], d C[2p+1] against (g, s, 1)
#pragma unroll
    for (int q = 0; q < 12; q++) acc_bc[q] = 0.0f;

  for (int chunk = blockIdx.x; chunk < pl.chunks; chunk += gridDim.x) {
    const ChunkRef c = chunk_ref(pl, chunk, dir, io);
    const int ti = c.ti, off = c.off;
    float le, lo;                                    // adjoint of the state after the current step
    {
        const float* lam = pl.adj_lam + (((size_t)dir * pl.chunks + chunk) * SCAN_THREADS + tid) * 2;
        le = lam[0];
        lo = lam[1];
    }
    const int ntiles = (c.uend - c.ustart + BT - 1) / BT;
    for (int tile = ntiles - 1; tile >= 0; tile--) {
        const int u0 = c.ustart + tile * BT, cnt = min(BT, c.uend - u0);
        // ---- 1: projections, activation derivatives, incoming gradients
        bool small = true;
        {
            const bool valid = tu < cnt;
            float g, s;
            int orig;
            load_step(c, dir, u0 + tu, valid, &g, &s, &orig);
            if (part == 0) { s_gs[2 * tu] = g; s_gs[2 * tu + 1] = s; }
            if (part < DM / 4 && c.dctx != nullptr) {
                const float4 dv = valid ? reinterpret_cast<const float4*>(c.dctx + (size_t)orig * DM)[part] : make_float4(0.f, 0.f, 0.f, 0.f);
                reinterpret_cast<float4*>(s_dctx + tu * DM)[part] = dv;
            }
#pragma unroll
            for (int q = 0; q < ROWS / 4; q++) {
                const int r = part * (ROWS / 4) + q;
                const float raw = sg2_comp_eval(cw[SG2_COMP_DT][q], g, s);
                const float dtv = valid ? sg_softplus(raw) : 0.0f;
                small = small && (dtv * s_fmax[r] < SG_SINCOS_TINY_LIMIT);
                arr(A_DT)[r * BBST + tu] = dtv;
                arr(A_DSP)[r * BBST + tu] = (raw > 20.0f) ? 1.0f : sg_sigmoid(raw);
                arr(A_XB)[r * BBST + tu] = valid ? sg2_comp_eval(cw[SG2_COMP_XB][q], g, s) : 0.0f;
                arr(A_B)[r * BBST + tu] = sg2_comp_eval(cw[SG2_COMP_B][q], g, s);
                arr(A_C)[r * BBST + tu] = sg2_comp_eval(cw[SG2_COMP_C][q], g, s);
                const float z = sg2_comp_eval(cw[SG2_COMP_Z][q], g, s);
                const float sz = sg_sigmoid(z);
                arr(A_GATE)[r * BBST + tu] = z * sz;
                arr(A_DGATE)[r * BBST + tu] = sz * sg_fma(z, 1.0f - sz, 1.0f);
            }
        }
        const bool tiny = __syncthreads_and(small);

        // ---- 2: forward recurrence over the tile, states kept
        const float* ht = pl.htile + ((size_t)dir * htile_count(pl.total, pl.P) + htile_index(off, ti, u0)) * 2 * SCAN_THREADS;
        const float hs_e = ht[tid], hs_o = ht[SCAN_THREADS + tid];
        {
            // in blocks of FB steps: operands and the state-independent coefficients of the whole block first (independent
            // instruction streams), then the short serial state update.  Steps past the end of the chunk are
            // identities (dt = 0, x-branch = 0) whose results nobody reads.
            constexpr int FB = 8;
            static_assert(BT % FB == 0, "whole blocks");
            float he = hs_e, ho = hs_o;
            for (int k0 = 0; k0 < cnt; k0 += FB) {
                float dtv[FB], uxv[FB], Bev[FB], Bov[FB], Cev[FB], Cov[FB], aev[FB], aov[FB], snv[FB], csv[FB], yv[FB];
#pragma unroll
                for (int q = 0; q < FB; q++) {
                    const int k = k0 + q;
                    dtv[q] = arr(A_DT)[j * BBST + k];
                    uxv[q] = dtv[q] * arr(A_XB)[j * BBST + k];
                    Bev[q] = arr(A_B)[(2 * p) * BBST + k]; Bov[q] = arr(A_B)[(2 * p + 1) * BBST + k];
                    Cev[q] = arr(A_C)[(2 * p) * BBST + k]; Cov[q] = arr(A_C)[(2 * p + 1) * BBST + k];
                }
#pragma unroll
                for (int q = 0; q < FB; q++) {
                    sg_abar_pair(dtv[q], a_e, a_o, &aev[q], &aov[q]);
                    rot_sincos(tiny, dtv[q] * freq, &snv[q], &csv[q]);
                }
#pragma unroll
                for (int q = 0; q < FB; q++) {
                    const float re = sg_fma(he, csv[q], -(ho * snv[q])), ro = sg_fma(ho, csv[q], he * snv[q]);
                    he = sg_fma(aev[q], re, uxv[q] * Bev[q]);
                    ho = sg_fma(aov[q], ro, uxv[q] * Bov[q]);
                    sH[((k0 + q) * SCAN_THREADS + tid) * 2] = he;
                    sH[((k0 + q) * SCAN_THREADS + tid) * 2 + 1] = ho;
                    yv[q] = sg_fma(ho, Cov[q], he * Cev[q]);
                }
#pragma unroll
                for (int q = 0; q < FB; q++) yv[q] = pair_sum(yv[q]);
                if (p == 0) {
#pragma unroll
                    for (int q = 0; q < FB; q++) arr(A_Y)[j * BBST + k0 + q] = yv[q];
                }
            }
        }
        __syncthreads();

        // ---- 3: per step and column: out, d out, d y, d z, D-skip part of d x-branch
        float4 dscan4 = make_float4(0.f, 0.f, 0.f, 0.f);          // d out of this lane's four rows when it comes in directly
        if (c.dscan != nullptr && tu < cnt) dscan4 = reinterpret_cast<const float4*>(c.dscan + (size_t)(u0 + tu) * DI)[part];
#pragma unroll
        for (int q = 0; q < ROWS / 4; q++) {
            const int r = part * (ROWS / 4) + q;
            float dout = 0.0f;
            if (c.dscan != nullptr) {
                dout = q == 0 ? dscan4.x : q == 1 ? dscan4.y : q == 2 ? dscan4.z : dscan4.w;
            } else {
#pragma unroll
                for (int d = 0; d < DM; d++) dout = sg_fma(wo[q][d], s_dctx[tu * DM + d], dout);
            }
            const float y = arr(A_Y)[r * BBST + tu], gate = arr(A_GATE)[r * BBST + tu], xb = arr(A_XB)[r * BBST + tu];
            const bool valid = tu < cnt;
            arr(A_DY)[r * BBST + tu] = valid ? dout * gate : 0.0f;
            arr(A_DZ)[r * BBST + tu] = valid ? (dout * y) * arr(A_DGATE)[r * BBST + tu] : 0.0f;
            arr(A_DXB)[r * BBST + tu] = valid ? dout * dwr[q] : 0.0f;
            arr(A_GATE)[r * BBST + tu] = valid ? sg_fma(y, gate, dwr[q] * xb) : 0.0f;     // out, for d out_proj
            arr(A_DGATE)[r * BBST + tu] = valid ? dout : 0.0f;                           // d out, for d D
            arr(A_DDT)[r * BBST + tu] = 0.0f;
        }
        __syncthreads();

        // ---- 4: adjoint recurrence, last step of the tile first
        // (blocks of RB steps, operands and coefficients of the block first, as in step 2)
        constexpr int RB = 8;
        static_assert(BT % RB == 0, "whole blocks");
        for (int k0 = ((cnt - 1) / RB) * RB; k0 >= 0; k0 -= RB) {
            float dtv[RB], xbv[RB], dyv[RB], Bev[RB], Bov[RB], Cev[RB], Cov[RB], gkv[RB], skv[RB], hev[RB + 1], hov[RB + 1];
            float aev[RB], aov[RB], snv[RB], csv[RB];
#pragma unroll
            for (int q = 0; q < RB; q++) {
                const int k = k0 + q;
                dtv[q] = arr(A_DT)[j * BBST + k]; xbv[q] = arr(A_XB)[j * BBST + k]; dyv[q] = arr(A_DY)[j * BBST + k];
                Bev[q] = arr(A_B)[(2 * p) * BBST + k]; Bov[q] = arr(A_B)[(2 * p + 1) * BBST + k];
                Cev[q] = arr(A_C)[(2 * p) * BBST + k]; Cov[q] = arr(A_C)[(2 * p + 1) * BBST + k];
                gkv[q] = s_gs[2 * k]; skv[q] = s_gs[2 * k + 1];
                hev[q + 1] = sH[(k * SCAN_THREADS + tid) * 2]; hov[q + 1] = sH[(k * SCAN_THREADS + tid) * 2 + 1];
            }
            hev[0] = (k0 > 0) ? sH[((k0 - 1) * SCAN_THREADS + tid) * 2] : hs_e;
            hov[0] = (k0 > 0) ? sH[((k0 - 1) * SCAN_THREADS + tid) * 2 + 1] : hs_o;
#pragma unroll
            for (int q = 0; q < RB; q++) {
                sg_abar_pair(dtv[q], a_e, a_o, &aev[q], &aov[q]);
                rot_sincos(tiny, dtv[q] * freq, &snv[q], &csv[q]);
            }
            float ddtv[RB], dxbv[RB];
            float shBe[DX ? RB : 1], shBo[DX ? RB : 1], shCe[DX ? RB : 1], shCo[DX ? RB : 1];     // this column's share of d B / d C per step
#pragma unroll
            for (int q = RB - 1; q >= 0; q--) {
                const bool live = k0 + q < cnt;                  // steps past the end of the chunk leave lambda alone
                const float dt = dtv[q], xb = xbv[q], dy = dyv[q], ae = aev[q], ao = aov[q], sn = snv[q], cs = csv[q];
                const float he = hev[q + 1], ho = hov[q + 1], pe = hev[q], po = hov[q], gk = gkv[q], sk = skv[q];
                // y = sum h C
                le = sg_fma(dy, Cev[q], le);
                lo = sg_fma(dy, Cov[q], lo);
                // d C[2p], d C[2p+1] of this step are sums over the columns of dy*h, d B of lambda*dt*xb; what is wanted
                // is their sum over steps against (g, s, 1), so each lane sums its own column's share over the steps
                // and the columns are added once, when the workgroup is done
                {
                    const float te = dy * he, to = dy * ho;
                    acc_bc[6] = sg_fma(te, gk, acc_bc[6]); acc_bc[7] = sg_fma(te, sk, acc_bc[7]); acc_bc[8] += te;
                    acc_bc[9] = sg_fma(to, gk, acc_bc[9]); acc_bc[10] = sg_fma(to, sk, acc_bc[10]); acc_bc[11] += to;
                    if (DX) { shCe[q] = te; shCo[q] = to; }
                }
                // h' = A_bar * rot(h) + dt * xb * B
                const float re = sg_fma(pe, cs, -(po * sn)), ro = sg_fma(po, cs, pe * sn);
                // A_bar = 2/d - 1, d = 1 + dt*a: dA_bar/dd = -2/d^2 = -(A_bar+1)^2/2
                const float dd_e = (le * re) * (-0.5f * (ae + 1.0f) * (ae + 1.0f));
                const float dd_o = (lo * ro) * (-0.5f * (ao + 1.0f) * (ao + 1.0f));
                float ddt = sg_fma(dd_e, a_e, dd_o * a_o);
                acc_alog_e = sg_fma(dd_e * dt, a_e, acc_alog_e);
                acc_alog_o = sg_fma(dd_o * dt, a_o, acc_alog_o);
                const float dre = le * ae, dro = lo * ao;
                const float dth = sg_fma(dro, re, -(dre * ro));        // d re/d theta = -ro, d ro/d theta = re
                ddt = sg_fma(dth, freq, ddt);
                acc_rope = sg_fma(dth, dt, acc_rope);
                const float qb = sg_fma(le, Bev[q], lo * Bov[q]);
                ddt = sg_fma(qb, xb, ddt);
                const float ux = dt * xb;
                {
                    const float te = le * ux, to = lo * ux;
                    acc_bc[0] = sg_fma(te, gk, acc_bc[0]); acc_bc[1] = sg_fma(te, sk, acc_bc[1]); acc_bc[2] += te;
                    acc_bc[3] = sg_fma(to, gk, acc_bc[3]); acc_bc[4] = sg_fma(to, sk, acc_bc[4]); acc_bc[5] += to;
                    if (DX) { shBe[q] = te; shBo[q] = to; }
                }
                ddtv[q] = ddt;
                dxbv[q] = qb * dt;
                // lambda for the previous step
                const float nle = sg_fma(dre, cs, dro * sn), nlo = sg_fma(dro, cs, -(dre * sn));
                le = live ? nle : le;
                lo = live ? nlo : lo;
            }
#pragma unroll
            for (int q = 0; q < RB; q++) { ddtv[q] = pair_sum(ddtv[q]); dxbv[q] = pair_sum(dxbv[q]); }
            if (DX) {
                // d B[2p], d B[2p+1], d C[2p], d C[2p+1] of every step: columns of the wave added here, the two waves in step 6
#pragma unroll
                for (int q = 0; q < RB; q++) {
                    const float s0 = xor_sum_columns(shBe[q]), s1 = xor_sum_columns(shBo[q]);
                    const float s2 = xor_sum_columns(shCe[q]), s3 = xor_sum_columns(shCo[q]);
                    if ((tid & 63) < HP) {
                        float* dst = s_bc + ((w * BT + k0 + q) * 4) * HP + p;
                        dst[0] = s0; dst[HP] = s1; dst[2 * HP] = s2; dst[3 * HP] = s3;
                    }
                }
            }
            if (p == 0) {
#pragma unroll
                for (int q = 0; q < RB; q++) {
                    if (k0 + q < cnt) {
                        arr(A_DDT)[j * BBST + k0 + q] = ddtv[q] * arr(A_DSP)[j * BBST + k0 + q];
                        arr(A_DXB)[j * BBST + k0 + q] += dxbv[q];
                    }
                }
            }
        }
        __syncthreads();

        // ---- 5: sums over the tile's steps (steps past the end of the chunk hold zeros in every array read here)
        if (tid < 3 * 16) {              // x-branch, z, dt (the first three coefficient groups)
            const int group = tid / 16, r = tid % 16;
#pragma unroll 8
            for (int k = 0; k < BT; k++) {
                float dv;
                if (group == SG2_COMP_XB) dv = arr(A_DXB)[r * BBST + k];
                else if (group == SG2_COMP_Z) dv = arr(A_DZ)[r * BBST + k];
                else dv = arr(A_DDT)[r * BBST + k];
                acc_c0 = sg_fma(dv, s_gs[2 * k], acc_c0);
                acc_c1 = sg_fma(dv, s_gs[2 * k + 1], acc_c1);
                acc_c2 += dv;
            }
        } else if (tid < SG2_COMP_GROUPS * 16 + DI) {
            const int r = tid - SG2_COMP_GROUPS * 16;
#pragma unroll 8
            for (int k = 0; k < BT; k++) acc_D = sg_fma(arr(A_DGATE)[r * BBST + k], arr(A_XB)[r * BBST + k], acc_D);
        }
        if (c.dscan == nullptr) {
            const int d = tid >> 4, r = tid & 15;       // out_proj[d][r]
#pragma unroll 8
            for (int k = 0; k < BT; k++) acc_wout = sg_fma(s_dctx[k * DM + d], arr(A_GATE)[r * BBST + k], acc_wout);
        }
        // ---- 6 (optional): gradient w.r.t. the input projection x of every step of the tile,
        //      d x = sum over the 80 pre-activation rows of (d row) * d row/d x; lane (tu, part) forms entries 2*part, 2*part+1
        if (DX) {
            if (tu < cnt) {
                float a0 = 0.0f, a1 = 0.0f;
                const float* rx = s_rx + 2 * part;
#pragma unroll 4
                for (int r = 0; r < 16; r++) {
                    const float dxb = arr(A_DXB)[r * BBST + tu], dz = arr(A_DZ)[r * BBST + tu], ddt = arr(A_DDT)[r * BBST + tu];
                    const int pr = r >> 1, odd = r & 1;
                    const float dB = s_bc[((0 * BT + tu) * 4 + odd) * HP + pr] + s_bc[((1 * BT + tu) * 4 + odd) * HP + pr];
                    const float dC = s_bc[((0 * BT + tu) * 4 + 2 + odd) * HP + pr] + s_bc[((1 * BT + tu) * 4 + 2 + odd) * HP + pr];
                    const float* r0 = rx + (SG2_COMP_XB * 16 + r) * DM;
                    const float* r1 = rx + (SG2_COMP_Z * 16 + r) * DM;
                    const float* r2 = rx + (SG2_COMP_DT * 16 + r) * DM;
                    const float* r3 = rx + (SG2_COMP_B * 16 + r) * DM;
                    const float* r4 = rx + (SG2_COMP_C * 16 + r) * DM;
                    a0 = sg_fma(dxb, r0[0], a0); a1 = sg_fma(dxb, r0[1], a1);
                    a0 = sg_fma(dz, r1[0], a0); a1 = sg_fma(dz, r1[1], a1);
                    a0 = sg_fma(ddt, r2[0], a0); a1 = sg_fma(ddt, r2[1], a1);
                    a0 = sg_fma(dB, r3[0], a0); a1 = sg_fma(dB, r3[1], a1);
                    a0 = sg_fma(dC, r4[0], a0); a1 = sg_fma(dC, r4[1], a1);
                }
                const int u = u0 + tu, t = dir ? (c.N - 1 - u) : u;
                float2* dst = reinterpret_cast<float2*>(io.dx + ((size_t)dir * pl.total + off + t) * DM) + part;
                *dst = make_float2(a0, a1);
            }
        }
        __syncthreads();
    }

  }
    // this workgroup's sums -> its row of the partials buffer (every entry of the row is written)
    float* g_comp = pl.adj_part + ((size_t)dir * gridDim.x + blockIdx.x) * SG2_BWD_STRIDE;
    float* g_alog = g_comp + SG2_COMP_GROUPS * 16 * 3;
    float* g_rope = g_alog + DI * DS;
    float* g_D = g_rope + DI * HP;
    float* g_wout = g_D + DI;
    g_alog[j * DS + 2 * p] = acc_alog_e;
    g_alog[j * DS + 2 * p + 1] = acc_alog_o;
    g_rope[j * HP + p] = acc_rope;
    // B and C coefficient gradients: columns added within the wave, then the two waves through LDS
#pragma unroll
    for (int q = 0; q < 12; q++) acc_bc[q] = xor_sum_columns(acc_bc[q]);
    __syncthreads();
    if ((tid & 63) < 8) {             // column 0 of each wave holds the wave's sums for pair p
#pragma unroll
        for (int q = 0; q < 12; q++) lds[(w * 8 + p) * 12 + q] = acc_bc[q];
    }
    __syncthreads();
    if (tid < 3 * 16) {
        g_comp[tid * 3 + 0] = acc_c0;
        g_comp[tid * 3 + 1] = acc_c1;
        g_comp[tid * 3 + 2] = acc_c2;
    } else if (tid < SG2_COMP_GROUPS * 16) {
        const int group = tid / 16, r = tid % 16;            // B: group 3, C: group 4; row r = 2*pair + (odd)
        const int q0 = (group == SG2_COMP_C ? 6 : 0) + (r & 1) * 3;
#pragma unroll
        for (int c = 0; c < 3; c++) g_comp[tid * 3 + c] = lds[(r >> 1) * 12 + q0 + c] + lds[(8 + (r >> 1)) * 12 + q0 + c];
    } else if (tid < SG2_COMP_GROUPS * 16 + DI) {
        g_D[tid - SG2_COMP_GROUPS * 16] = acc_D;
    }
    g_wout[tid] = acc_wout;
}

// ---- rows of the partials buffer added in a fixed order (64 entries per workgroup, ROW_SLICES lanes per entry each taking
// every ROW_SLICES-th row, then the partial sums in order)
constexpr int ROW_SLICES = 16;
__global__ __launch_bounds__(64 * ROW_SLICES) void k_adj_sum_rows(const float* __restrict__ part, int rows_per_dir, float* __restrict__ out) {
    __shared__ float s_part[ROW_SLICES][64];
    const int col = threadIdx.x & 63, slice = threadIdx.x >> 6;
    const int o = blockIdx.x * 64 + col;          // 2 * SG2_BWD_STRIDE is a multiple of 64
    const int dir = o / SG2_BWD_STRIDE, e = o % SG2_BWD_STRIDE;
    float acc = 0.0f;
#pragma unroll 8
    for (int r = slice; r < rows_per_dir; r += ROW_SLICES) acc += part[((size_t)dir * rows_per_dir + r) * SG2_BWD_STRIDE + e];
    s_part[slice][col] = acc;
    __syncthreads();
    if (slice != 0) return;
#pragma unroll
    for (int q = 1; q < ROW_SLICES; q++) acc += s_part[q][col];
    out[o] = acc;
}

// ---- from the gradients of the composed coefficients to those of the weights they were composed from
// (the transpose of sg2_compose_one), and the final layout: input_proj W [8][2], b [8]; then per direction in_proj
// [32][8], dt_proj W [16][16], b [16], B_proj [16][16], C_proj [16][16], A_log [16][16], D [16], rope_freq [16][8],
// out_proj [8][16].  One workgroup; blk is k_adj_sum_rows' output ([2][SG2_BWD_STRIDE]).
//   src = [W_in | b_in] (8x3);  xb = in_proj[:16] src;  z = in_proj[16:] src;  dt = dt_W xb + [0 0 dt_b];  B = B_proj xb;  C = C_proj xb
__global__ __launch_bounds__(256) void k_compose_backward(Plan pl, const float* __restrict__ blk, float* __restrict__ out) {
    static_assert(DM == 8 && DI == 16 && DS == 16 && SG2_COMP_GROUPS == 5, "k_compose_backward: fixed dimensions");
    __shared__ float s_src[DM][3], s_xb[DI][3], s_d[SG2_COMP_GROUPS][16][3], s_dxb[DI][3];
    const int tid = threadIdx.x;
    constexpr int PER_DIR = 2 * DI * DM + DI * DI + DI + 2 * DS * DI + DI * DS + DI + DI * HP + DM * DI;
    static_assert(2 * DM + DM + 2 * PER_DIR == SG2_SCAN_GRAD_FLOATS, "gradient layout");
    if (tid < DM * 3) s_src[tid / 3][tid % 3] = (tid % 3 < 2) ? pl.W.w[W_IN_W][(tid / 3) * 2 + tid % 3] : pl.W.w[W_IN_B][tid / 3];
    float dsrc = 0.0f;                              // thread (d, c) for tid < 24, summed over both directions
    for (int dir = 0; dir < 2; dir++) {
        const int b = dir ? W_B_INPROJ : W_F_INPROJ;
        const float* __restrict__ in_proj = pl.W.w[b];
        const float* __restrict__ dtW = pl.W.w[b + 1];
        const float* __restrict__ Bp = pl.W.w[b + 3];
        const float* __restrict__ Cp = pl.W.w[b + 4];
        const float* __restrict__ g = blk + dir * SG2_BWD_STRIDE;
        float* __restrict__ o = out + 3 * DM + dir * PER_DIR;
        __syncthreads();
        if (tid < SG2_COMP_GROUPS * 16 * 3) (&s_d[0][0][0])[tid] = g[tid];
        if (tid < DI * 3) (&s_xb[0][0])[tid] = pl.comp[dir * (SG2_COMP_GROUPS * 16 * 3) + SG2_COMP_XB * 16 * 3 + tid];
        __syncthreads();
        {   // dt_W, B_proj, C_proj: d W[r][k] = sum_c d v[r][c] * xb[k][c]
            const int r = tid >> 4, k = tid & 15;
            float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                a0 = sg_fma(s_d[SG2_COMP_DT][r][c], s_xb[k][c], a0);
                a1 = sg_fma(s_d[SG2_COMP_B][r][c], s_xb[k][c], a1);
                a2 = sg_fma(s_d[SG2_COMP_C][r][c], s_xb[k][c], a2);
            }
            o[2 * DI * DM + tid] = a0;
            o[2 * DI * DM + DI * DI + DI + tid] = a1;
            o[2 * DI * DM + DI * DI + DI + DS * DI + tid] = a2;
            if (tid < DI) o[2 * DI * DM + DI * DI + tid] = s_d[SG2_COMP_DT][tid][2];      // dt_b
        }
        if (tid < DI * 3) {   // d xb[k][c] = d xb-coefficients + dt_W^T d dt + B_proj^T d B + C_proj^T d C
            const int k = tid / 3, c = tid % 3;
            float a = s_d[SG2_COMP_XB][k][c];
            for (int r = 0; r < 16; r++) {
                a = sg_fma(dtW[r * DI + k], s_d[SG2_COMP_DT][r][c], a);
                a = sg_fma(Bp[r * DI + k], s_d[SG2_COMP_B][r][c], a);
                a = sg_fma(Cp[r * DI + k], s_d[SG2_COMP_C][r][c], a);
            }
            s_dxb[k][c] = a;
        }
        __syncthreads();
        {   // in_proj [32][8]: rows 0..15 from d xb, rows 16..31 from d z
            const int r = tid >> 3, d = tid & 7;
            float a = 0.0f;
#pragma unroll
            for (int c = 0; c < 3; c++) a = sg_fma(r < DI ? s_dxb[r][c] : s_d[SG2_COMP_Z][r - DI][c], s_src[d][c], a);
            o[tid] = a;
        }
        if (tid < DM * 3) {
            const int d = tid / 3, c = tid % 3;
            for (int r = 0; r < DI; r++) {
                dsrc = sg_fma(in_proj[r * DM + d], s_dxb[r][c], dsrc);
                dsrc = sg_fma(in_proj[(DI + r) * DM + d], s_d[SG2_COMP_Z][r][c], dsrc);
            }
        }
        // A_log, D, rope_freq, out_proj pass through (the block holds them as A_log, rope_freq, D, out_proj)
        const float* ga = g + SG2_COMP_GROUPS * 16 * 3;
        float* oa = o + 2 * DI * DM + DI * DI + DI + 2 * DS * DI;
        oa[tid] = ga[tid];                                                        // A_log [16][16]
        if (tid < DI) oa[DI * DS + tid] = ga[DI * DS + DI * HP + tid];            // D
        if (tid < DI * HP) oa[DI * DS + DI + tid] = ga[DI * DS + tid];            // rope_freq
        if (tid < DM * DI) oa[DI * DS + DI + DI * HP + tid] = ga[DI * DS + DI * HP + DI + tid];   // out_proj
    }
    if (tid < DM * 3) {
        const int d = tid / 3, c = tid % 3;
        if (c < 2) out[d * 2 + c] = dsrc; else out[2 * DM + d] = dsrc;
    }
}

__global__ void k_fill_zero(float* p, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0.0f;
}

// x = W_in [g, s] + b_in of every sorted position (the scan's 8-float input, which the forward kernels never
// materialise), for callers that keep the reference's interface.  One thread per element.
__global__ __launch_bounds__(256) void k_x_sorted(Plan pl, float* __restrict__ x_out) {
    const int tile = blockIdx.x;
    const int ti = sg::upper_seg(sg::as_const(pl.elem_tile_prefix), pl.P, tile);
    const TensorDev& T = pl.tensors[ti];
    const int start = (tile - pl.elem_tile_prefix[ti]) * ELEM_TILE;
    const int cnt = min(ELEM_TILE, T.numel - start);
    const bool has_s = pl.sharp_nonzero[ti] != 0;
    const float* __restrict__ Win = pl.W.w[W_IN_W];
    const float* __restrict__ bin = pl.W.w[W_IN_B];
    for (int k = threadIdx.x; k < cnt; k += 256) {
        const int t = T.off + start + k;
        const int32_t v = pl.vals[0][t];
        const float g = sg_i2f((int32_t)pl.keys[0][t] | (v & (int32_t)0x80000000));
        const float s = has_s ? pl.ssorted[t] : 0.0f;
        float4 lo, hi;
        float x[DM];
#pragma unroll
        for (int d = 0; d < DM; d++) x[d] = sg_fma(Win[2 * d + 1], s, Win[2 * d] * g) + bin[d];
        lo = make_float4(x[0], x[1], x[2], x[3]);
        hi = make_float4(x[4], x[5], x[6], x[7]);
        reinterpret_cast<float4*>(x_out + (size_t)t * DM)[0] = lo;
        reinterpret_cast<float4*>(x_out + (size_t)t * DM)[1] = hi;
    }
}

// The intermediates the reference's forward-save kernels leave behind (x-branch, z, dt of every scan step; the state
// after a step, every step or every `interval`-th; rows in the order of each direction's own scan, like scan_out:
// the reference runs its backward direction on a flipped copy of the input), rebuilt from what the forward pass kept: one workgroup per
// (chunk, direction) restarts every 32-step tile from its kept entry state and walks it with the plain forms of the
// recurrence (the forward pass may have taken a polynomial form for the same step: the values agree to rounding).
struct SavedOut {
    float* xb[2];
    float* z[2];
    float* dt[2];
    float* states[2];
    int interval;
};
__global__ __launch_bounds__(SCAN_THREADS) void k_saved_fill(Plan pl, SavedOut out) {
    constexpr int STEPS = 2 * HT_STEP, ST = STEPS + 1;
    __shared__ float s_dt[DI * ST], s_xb[DI * ST], s_B[DS * ST];
    static_assert(SCAN_THREADS == 4 * STEPS && DI == 16 && DS == 16, "four row groups of four rows per step");
    const int chunk = blockIdx.x, dir = blockIdx.y, tid = threadIdx.x;
    const AdjIO none = {nullptr, {nullptr, nullptr}, nullptr, nullptr};
    const ChunkRef c = chunk_ref(pl, chunk, dir, none);
    const int b = dir ? W_B_INPROJ : W_F_INPROJ;
    const float* __restrict__ Alog = pl.W.w[b + 5];
    const float* __restrict__ rope = pl.W.w[b + 7];
    const float* __restrict__ comp = pl.comp + dir * (SG2_COMP_GROUPS * 16 * 3);
    const int tu = tid & (STEPS - 1), quarter = tid >> 5;
    const int j = tid >> 3, p = tid & 7;
    const float a_e = 0.5f * sg_exp(Alog[j * DS + 2 * p]), a_o = 0.5f * sg_exp(Alog[j * DS + 2 * p + 1]);
    const float freq = rope[j * HP + p];
    int row0 = c.off;                 // first row of this tensor in saved_states
    if (out.interval > 1) {
        row0 = 0;
        for (int i = 0; i < c.ti; i++) row0 += (pl.tensors[i].numel + out.interval - 1) / out.interval;
    }
    for (int u0 = c.ustart; u0 < c.uend; u0 += STEPS) {
        const int cnt = min(STEPS, c.uend - u0);
        {
            const bool valid = tu < cnt;
            float g, s;
            int orig;
            load_step(c, dir, u0 + tu, valid, &g, &s, &orig);
            float xv[4], zv[4], dv[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = quarter * 4 + q;
                xv[q] = sg2_comp_eval(comp + (SG2_COMP_XB * 16 + r) * 3, g, s);
                zv[q] = sg2_comp_eval(comp + (SG2_COMP_Z * 16 + r) * 3, g, s);
                dv[q] = sg_softplus(sg2_comp_eval(comp + (SG2_COMP_DT * 16 + r) * 3, g, s));
                s_dt[r * ST + tu] = valid ? dv[q] : 0.0f;
                s_xb[r * ST + tu] = valid ? xv[q] : 0.0f;
                s_B[r * ST + tu] = sg2_comp_eval(comp + (SG2_COMP_B * 16 + r) * 3, g, s);
            }
            if (valid) {
                const size_t at = ((size_t)c.off + u0 + tu) * DI + quarter * 4;       // row = scan step, as for scan_out
                if (out.xb[dir]) *reinterpret_cast<float4*>(out.xb[dir] + at) = make_float4(xv[0], xv[1], xv[2], xv[3]);
                if (out.z[dir]) *reinterpret_cast<float4*>(out.z[dir] + at) = make_float4(zv[0], zv[1], zv[2], zv[3]);
                if (out.dt[dir]) *reinterpret_cast<float4*>(out.dt[dir] + at) = make_float4(dv[0], dv[1], dv[2], dv[3]);
            }
        }
        __syncthreads();
        if (out.states[dir] != nullptr) {
            const float* ht = pl.htile + ((size_t)dir * htile_count(pl.total, pl.P) + htile_index(c.off, c.ti, u0)) * 2 * SCAN_THREADS;
            float he = ht[tid], ho = ht[SCAN_THREADS + tid];
            for (int k = 0; k < cnt; k++) {
                const float dt = s_dt[j * ST + k], ux = dt * s_xb[j * ST + k];
                float ae, ao, sn, cs;
                sg_abar_pair(dt, a_e, a_o, &ae, &ao);
                sg_sincos(dt * freq, &sn, &cs);
                const float re = sg_fma(he, cs, -(ho * sn)), ro = sg_fma(ho, cs, he * sn);
                he = sg_fma(ae, re, ux * s_B[(2 * p) * ST + k]);
                ho = sg_fma(ao, ro, ux * s_B[(2 * p + 1) * ST + k]);
                const int u = u0 + k;
                int row = -1;
                if (out.interval <= 1) row = c.off + u;
                else if ((u + 1) % out.interval == 0 || u == c.N - 1) row = row0 + u / out.interval;
                if (row >= 0) *reinterpret_cast<float2*>(out.states[dir] + ((size_t)row * DI + j) * DS + 2 * p) = make_float2(he, ho);
            }
        }
        __syncthreads();
    }
}

}  // namespace

int launch_saved_intermediates(const Plan& pl, const Sg2BilevelExtra& ex, hipStream_t st) {
    if (pl.total == 0) return 0;
    SavedOut out;
    bool any = false;
    for (int d = 0; d < 2; d++) {
        out.xb[d] = ex.saved_x_branch[d]; out.z[d] = ex.saved_z[d]; out.dt[d] = ex.saved_dt[d]; out.states[d] = ex.saved_states[d];
        any = any || out.xb[d] || out.z[d] || out.dt[d] || out.states[d];
    }
    if (!any) return 0;
    out.interval = ex.checkpoint_interval;
    hipLaunchKernelGGL(k_saved_fill, dim3(pl.chunks, 2), dim3(SCAN_THREADS), 0, st, pl, out);
    SG_LAUNCH_CHECK("k_saved_fill");
    return 0;
}

int launch_x_sorted(const Plan& pl, float* x_out, hipStream_t st) {
    static_assert(DM == 8, "k_x_sorted: two float4 per element");
    if (pl.total == 0) return 0;
    hipLaunchKernelGGL(k_x_sorted, dim3(pl.elem_tiles), dim3(256), 0, st, pl, x_out);
    SG_LAUNCH_CHECK("k_x_sorted");
    return 0;
}

int launch_bilevel_backward(const Plan& pl, const float* d_ctx, const float* const d_scan[2], const float* rx, float* dx, float* grads_out,
                            hipStream_t st) {
    static_assert(DM * DI == SCAN_THREADS, "one thread per out_proj entry");
    static_assert(SG2_BWD_STRIDE == SG2_COMP_GROUPS * 16 * 3 + DI * DS + DI * HP + DI + DM * DI, "layout of the per-direction sums");
    if (pl.total == 0) {
        hipLaunchKernelGGL(k_fill_zero, dim3(8), dim3(256), 0, st, grads_out, SG2_SCAN_GRAD_FLOATS);
        SG_LAUNCH_CHECK("k_fill_zero");
        return 0;
    }
    const AdjIO io = {d_ctx, {d_scan ? d_scan[0] : nullptr, d_scan ? d_scan[1] : nullptr}, rx, dx};
    // at least four tiles per wave: below that the steps behind the range outweigh it
    const int64_t tiles = (int64_t)pl.elem_tiles * (ELEM_TILE / AT);
    const int64_t waves = std::max<int64_t>((tiles + 3) / 4, pl.chunks);
    const int groups = dx != nullptr ? std::min(pl.chunks, 512) : (int)std::min<int64_t>(waves, ADJ_GROUPS);
    if (pl.wchunks > 0) {
        hipLaunchKernelGGL(k_adj_summary, dim3(pl.chunks, 2), dim3(SCAN_THREADS), 0, st, pl, io, dx == nullptr);
        SG_LAUNCH_CHECK("k_adj_summary");
    }
    if (pl.wchunks > 0 || dx != nullptr) {
        hipLaunchKernelGGL(k_adj_prefix, dim3(pl.P, 2), dim3(SCAN_THREADS), 0, st, pl, dx == nullptr);
        SG_LAUNCH_CHECK("k_adj_prefix");
    }
    if (dx != nullptr) {
        static bool raised[64] = {};
        int dev = 0;
        SG_HIP_CHECK(hipGetDevice(&dev));
        if (dev < 0 || dev >= 64) return sg::fail("device index %d out of range", dev);
        if (!raised[dev]) {
            SG_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_bilevel_backward), hipFuncAttributeMaxDynamicSharedMemorySize,
                                             BILEVEL_DX_LDS_BYTES));
            raised[dev] = true;
        }
        hipLaunchKernelGGL(k_bilevel_backward, dim3(groups, 2), dim3(SCAN_THREADS), BILEVEL_DX_LDS_BYTES, st, pl, io);
        SG_LAUNCH_CHECK("k_bilevel_backward");
    } else {
        if (d_ctx != nullptr) hipLaunchKernelGGL(k_adjoint<false>, dim3(groups, 2), dim3(64), 0, st, pl, io);
        else hipLaunchKernelGGL(k_adjoint<true>, dim3(groups, 2), dim3(64), 0, st, pl, io);
        SG_LAUNCH_CHECK("k_adjoint");
    }
    static_assert((2 * SG2_BWD_STRIDE) % 64 == 0, "k_adj_sum_rows: whole workgroups");
    hipLaunchKernelGGL(k_adj_sum_rows, dim3(2 * SG2_BWD_STRIDE / 64), dim3(64 * ROW_SLICES), 0, st, pl.adj_part, groups, pl.adj_blk);
    SG_LAUNCH_CHECK("k_adj_sum_rows");
    hipLaunchKernelGGL(k_compose_backward, dim3(1), dim3(256), 0, st, pl, pl.adj_blk, grads_out);
    SG_LAUNCH_CHECK("k_compose_backward");
    return 0;
}

}  // namespace sg2
