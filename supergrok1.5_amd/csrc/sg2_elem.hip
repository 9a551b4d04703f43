// Per-element tail of the SuperGrok v2 step: GRU -> 4-head PEER product-key
// routing -> expert MLP -> skip connection -> mu EMA -> Adam + weight decay.
//
// Replaces fused_elem_step_kernel
// (csrc/supergrok2_mamba_peer_kernels.cu:793-1089 of the reference); the
// out_proj contraction that kernel starts with is done by the scan kernel,
// which hands over the two 8-float contexts per element in element order.
//
// One launch covers every tensor: a persistent grid walks tiles of 1024
// elements; the tile index is mapped to (tensor, offset) by a binary search
// over a P+1 entry prefix table.  The 144 expert MLPs live in LDS (records of
// 48 floats padded to 52 so that random per-lane experts spread over the
// banks); the net's dense products are chains of fp32 matrix instructions
// (step4).  expert_counts is accumulated in an LDS histogram and flushed
// once per workgroup (the reference issues one global atomic per element and
// head).
#include "sg2_internal.hpp"

namespace sg2 {
namespace {

constexpr int ELEM_THREADS = 256;
// floats per expert record in LDS: W1[EH] b1[EH] W2[EH] (+ pad for the 16-wide experts so that random per-lane
// experts spread over the banks)
template <int EHW>
constexpr int exp_stride() { return EHW == 16 ? 52 : 3 * EHW; }
typedef outputs4 vf4;

// The net's small matrix-vector products (GRU, queries, key scores) run on the matrix pipe (product4): step n's weights are
// block n % 16 of register n / 16, and a whole net of the default geometry takes 22.  As multiply-adds with scalar operands,
// GRU and scores were 650 of 1550 vector instructions an element and wave, with some forty scalar loads between them; the
// queries, as 32x32x1 products whose outputs had to be exchanged between lanes, are as fast in large calls, but a wave that
// evaluates one head needs only its quarter of them now.  The launch: 8 tensors below 256 elements 8.6 -> 6.6 us, 0.42 M
// elements 38.5 -> 34.6 (wide geometry 71 -> 61), 3.1 M bfloat16 174 -> 171, 25 M 1.21 -> 1.20 ms (there the part's power sets
// the rate: 4.65 ns a product and SIMD, 1.3 to 1.9 a multiply-add).
template <int N>
__device__ __forceinline__ vf4 step4(const float* w, float x, vf4 acc) { return product4<N % 16>(w[N / 16], x, acc); }

// Four waves per SIMD for the default geometry: told so, the compiler keeps the matrix results in ordinary registers
// instead of settling for three waves with accumulation registers to copy out of.
template <class G>
constexpr int elem_waves() { return G::DM == 8 ? 4 : 2; }
// FWD: the net's forward alone (sg2_meta_forward) -- smart gradient and new GRU state of every element go to the packed
// arrays fwd_smart / fwd_gru, nothing of the optimizer state is read or written.
// HEADS: small calls.  The four waves of a workgroup share 64 elements and evaluate one head each, so that an element's
// serial chain holds one head instead of four; wave 0 goes on with the sum, in the order of the heads as ever.
template <class G, int EH, bool DBG, bool FWD = false, bool HEADS = false>
__global__ __launch_bounds__(ELEM_THREADS) __attribute__((amdgpu_waves_per_eu(elem_waves<G>(), elem_waves<G>()))) void k_elem(Plan pl, int32_t* __restrict__ expert_counts,
                                                       int32_t* __restrict__ dbg_eidx, float* __restrict__ fwd_smart,
                                                       float* __restrict__ fwd_gru, int split) {
    constexpr int DM = G::DM, GRL = G::GRL, PIN = G::PIN, EXP_STRIDE = exp_stride<EH>();
    static_assert(!HEADS || ELEM_THREADS == 64 * NH, "a wave per head");
    constexpr int STEP = HEADS ? 64 : ELEM_THREADS;      // elements a workgroup works on at once
    static_assert(EH % 4 == 0, "expert records are read 16 bytes at a time");
    __shared__ float s_exp[NE * EXP_STRIDE];
    __shared__ float s_b2[NE];
    __shared__ int s_cnt[NE];
    // Weights of the products, four rows a block (see step4): GRU [z, r, h][input], queries [4 rows][input], keys [head][half][4 keys]
    // [dimension]; of the wave's own head only where it evaluates one.  Keys stay in registers, the others come from LDS, four
    // registers to a read.
    constexpr int HEADS_HERE = HEADS ? 1 : NH, HALF = DM / 2, KEY_GROUPS = PK / 4, Q_GROUPS = HEADS_HERE * DM / 4;
    static_assert(GH == 4 && PK % 4 == 0 && HALF % 4 == 0, "rows in groups of four");
    constexpr int N_GRU = 3 * GRL, N_QUERY = Q_GROUPS * PIN, N_KEYS = HEADS_HERE * 2 * KEY_GROUPS * HALF;
    constexpr int R_GRU = (N_GRU + 63) / 64 * 4, R_QUERY = (N_QUERY + 63) / 64 * 4, R_KEYS = (N_KEYS + 15) / 16;
    __shared__ __attribute__((aligned(16))) float s_w[(R_GRU + (HEADS ? NH : 1) * R_QUERY) * 64];
    __shared__ float s_head[HEADS ? 2 : 1][HEADS ? NH : 1][HEADS ? 64 : 1];
    const int own = HEADS ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0, member = threadIdx.x & (STEP - 1);
    int turn = 0;

    {
        const float* __restrict__ W[3] = {pl.W.w[W_EXP_W1], pl.W.w[W_EXP_B1], pl.W.w[W_EXP_W2]};
        constexpr int ROUNDS = (NE * EH + ELEM_THREADS - 1) / ELEM_THREADS;
        float v[3][ROUNDS];
#pragma unroll
        for (int r = 0; r < ROUNDS; r++)
#pragma unroll
            for (int m = 0; m < 3; m++) v[m][r] = W[m][min(r * ELEM_THREADS + (int)threadIdx.x, NE * EH - 1)];
        if (threadIdx.x < NE) {
            s_b2[threadIdx.x] = pl.W.w[W_EXP_B2][threadIdx.x];
            s_cnt[threadIdx.x] = 0;
        }
#pragma unroll
        for (int r = 0; r < ROUNDS; r++) {
            const int i = min(r * ELEM_THREADS + (int)threadIdx.x, NE * EH - 1), at = (i / EH) * EXP_STRIDE + i % EH;
#pragma unroll
            for (int m = 0; m < 3; m++) s_exp[at + m * EH] = v[m][r];
        }
    }
    float w_keys[R_KEYS];
    {
        const int lane = threadIdx.x & 63, row = lane & 3, block = lane >> 2;
        constexpr int WAVES = ELEM_THREADS / 64, QUERIES = (HEADS ? NH : 1) * R_QUERY;
        auto put = [&](int r, float v) { s_w[(r / 4) * 256 + lane * 4 + r % 4] = v; };
#pragma unroll
        for (int r0 = 0; r0 < R_GRU; r0 += WAVES) {
            const int r = r0 + (int)(threadIdx.x >> 6), n = min(16 * r + block, N_GRU - 1), m = n / GRL;
            put(r, (m == 0 ? pl.W.w[W_GRU_WZ] : m == 1 ? pl.W.w[W_GRU_WR] : pl.W.w[W_GRU_WH])[row * GRL + n % GRL]);
        }
#pragma unroll
        for (int r0 = 0; r0 < QUERIES; r0 += WAVES) {
            const int r = r0 + (int)(threadIdx.x >> 6), n = min(16 * (r % R_QUERY) + block, N_QUERY - 1);
            put(R_GRU + r, pl.W.w[W_PEER_Q][(r / R_QUERY * DM + 4 * (n / PIN) + row) * PIN + n % PIN]);
        }
#pragma unroll
        for (int r = 0; r < R_KEYS; r++) {
            const int n = min(16 * r + block, N_KEYS - 1), at = n / HALF, hh = own + at / (2 * KEY_GROUPS);
            w_keys[r] = (at / KEY_GROUPS % 2 ? pl.W.w[W_KEYS_B] : pl.W.w[W_KEYS_A])[(hh * PK + 4 * (at % KEY_GROUPS) + row) * HALF + n % HALF];
        }
    }
    __syncthreads();
    auto weights = [&](int first, auto& w) {
#pragma unroll
        for (int r = 0; r < (int)(sizeof(w) / 16); r++) {
            const vf4 v = *reinterpret_cast<const vf4*>(s_w + (first / 4 + r) * 256 + (threadIdx.x & 63) * 4);
#pragma unroll
            for (int q = 0; q < 4; q++) w[4 * r + q] = v[q];
        }
    };

    const sg::cfloat_p bz0 = sg::as_const(pl.W.w[W_GRU_BZ]), br0 = sg::as_const(pl.W.w[W_GRU_BR]), bh0 = sg::as_const(pl.W.w[W_GRU_BH]);

    // split: parts that a tile is cut into (1 or ELEM_TILE / STEP, see elem_grid)
    for (int part = blockIdx.x; part < pl.elem_tiles * split; part += gridDim.x) {
        const int tile = split == 1 ? part : part / split, len = split == 1 ? ELEM_TILE : ELEM_TILE / split;
        const sg::Seg seg = sg::find_seg(sg::as_const(pl.elem_tile_prefix), pl.P, tile);
        const int ti = seg.i;
        const TensorDev& T = pl.tensors[ti];
        const int start = (tile - seg.first) * ELEM_TILE + (part - tile * split) * len;
        const int cnt = min(len, T.numel - start);
        const int dtype = T.dtype;
        const float gs = grad_scale(pl, ti);
        const bool has_s = pl.sharp_nonzero[ti] != 0;       // set by the sort's key kernel: some sharpness entry of the tensor is not 0
        const float alpha = T.alpha, lamb = T.lamb, beta1 = T.beta1, bc2 = T.bc2, step_size = T.step_size;
        const float beta2 = pl.beta2, eps = pl.eps, rescale = pl.rescale, decay = pl.decay;

        // every lane runs every iteration (the matrix instructions ignore the execution mask); lanes past the end
        // of the tile recompute its last element and store nothing
        for (int k0 = 0; k0 < cnt; k0 += STEP) {
            const bool live = k0 + member < cnt;
            const int i = start + min(k0 + member, cnt - 1);
            const float g_raw = sg::load_elem(T.grad, dtype, i);        // clipped below, when the loads behind it are on their way
            float s = has_s ? sharp_raw(T, i) : 0.0f;
            float cf[DM], cb[DM], hold[GH];
            {
                const SG_GLOBAL vf4* pf = (const SG_GLOBAL vf4*)(pl.ctx + ((size_t)T.off + i) * DM);
                const SG_GLOBAL vf4* pb = (const SG_GLOBAL vf4*)(pl.ctx + ((size_t)pl.total + T.off + i) * DM);
#pragma unroll
                for (int q = 0; q < DM / 4; q++) {
                    const vf4 a = pf[q], b = pb[q];
                    cf[4 * q] = a[0]; cf[4 * q + 1] = a[1]; cf[4 * q + 2] = a[2]; cf[4 * q + 3] = a[3];
                    cb[4 * q] = b[0]; cb[4 * q + 1] = b[1]; cb[4 * q + 2] = b[2]; cb[4 * q + 3] = b[3];
                }
                const vf4 h4 = ((const SG_GLOBAL vf4*)T.gru)[i];
                hold[0] = h4[0]; hold[1] = h4[1]; hold[2] = h4[2]; hold[3] = h4[3];
            }
            // the optimizer state is requested now, so that its latency passes under the meta-net's arithmetic
            float mu = 0.0f, ea = 0.0f, easq = 0.0f, pv = 0.0f;
            if (!FWD && own == 0) {
                mu = sg::gptr(T.mu)[i]; ea = sg::gptr(T.ea)[i]; easq = sg::gptr(T.easq)[i];
                pv = sg::load_elem(T.param, dtype, i);
            }
            const float g = clipped(g_raw, gs, dtype);
            s = sharp_value(T, s);

            // ---- GRU: chain order = bias, g, s, fwd ctx, bwd ctx, h
            float zg[GH], rg[GH], hnew[GH];
            float pre_g[2 * GH], gate[2 * GH], pre_c[GH], cand[GH];      // gates and candidates share one reciprocal each
            float x[GRL];
            x[0] = g; x[1] = s;
#pragma unroll
            for (int q = 0; q < DM; q++) { x[2 + q] = cf[q]; x[2 + DM + q] = cb[q]; }
#pragma unroll
            for (int q = 0; q < GH; q++) x[2 + 2 * DM + q] = hold[q];
            // (re-read for every element, cache hits: hoisted they would take twelve registers)
            const int zo = sg::opaque_zero();
            const sg::cfloat_p bz = bz0 + zo, br = br0 + zo, bh = bh0 + zo;
            float w_gru[R_GRU], w_query[R_QUERY];
            weights(zo, w_gru);
            vf4 az = {bz[0], bz[1], bz[2], bz[3]}, ar = {br[0], br[1], br[2], br[3]}, ah = {bh[0], bh[1], bh[2], bh[3]};
            each<GRL>([&](auto c) {
                az = step4<c>(w_gru, x[c], az);
                ar = step4<GRL + c>(w_gru, x[c], ar);
                if (c < GRL - GH) ah = step4<2 * GRL + c>(w_gru, x[c], ah);
            });
#pragma unroll
            for (int j = 0; j < GH; j++) { pre_g[j] = az[j]; pre_g[GH + j] = ar[j]; }
            sg_sigmoid_block(2 * GH, pre_g, gate);
#pragma unroll
            for (int j = 0; j < GH; j++) { zg[j] = gate[j]; rg[j] = gate[GH + j]; }
            each<GH>([&](auto q) { ah = step4<2 * GRL + GRL - GH + q>(w_gru, rg[q] * hold[q], ah); });
#pragma unroll
            for (int j = 0; j < GH; j++) pre_c[j] = ah[j];
            sg_tanh_block(GH, pre_c, cand);
#pragma unroll
            for (int j = 0; j < GH; j++) hnew[j] = sg_fma(zg[j], cand[j], (1.0f - zg[j]) * hold[j]);
            if (!HEADS && live) {
                if (FWD) ((SG_GLOBAL vf4*)fwd_gru)[(size_t)T.off + i] = vf4{hnew[0], hnew[1], hnew[2], hnew[3]};
                else ((SG_GLOBAL vf4*)T.gru)[i] = vf4{hnew[0], hnew[1], hnew[2], hnew[3]};
            }

            // ---- PEER queries: chain order = h, fwd ctx, bwd ctx, g, s
            float xq[PIN];
#pragma unroll
            for (int q = 0; q < GH; q++) xq[q] = hnew[q];
#pragma unroll
            for (int q = 0; q < DM; q++) { xq[GH + q] = cf[q]; xq[GH + DM + q] = cb[q]; }
            xq[GH + 2 * DM] = g; xq[GH + 2 * DM + 1] = s;
            weights(R_GRU + own * R_QUERY + zo, w_query);
            vf4 query[Q_GROUPS];
            each<Q_GROUPS>([&](auto m) { query[m] = vf4{0.0f, 0.0f, 0.0f, 0.0f}; });
            each<PIN>([&](auto c) { each<Q_GROUPS>([&](auto m) { query[m] = step4<m * PIN + c>(w_query, xq[c], query[m]); }); });

            // ---- PEER routing + expert MLP
            // (an expert's record is requested before the next head's scores and evaluated after them)
            // Waves that route go before waves in the products above: those are long runs of matrix instructions that need no
            // other wave's time to hide anything, these wait for LDS.  (25 M elements 1.23 -> 1.20 ms; the other way round 1.22,
            // both parts ahead of the update below 1.24.)
            __builtin_amdgcn_s_setprio(1);
            float total = 0.0f, ho = 0.0f;
            float4 rec[3 * (EH / 4)];
            auto evaluate = [&]() {
#pragma unroll
                for (int q4 = 0; q4 < EH / 4; q4++) {
                    const float4 w1 = rec[q4], b1 = rec[EH / 4 + q4], w2 = rec[2 * (EH / 4) + q4];
                    float z;
                    z = sg_max(sg_fma(w1.x, g, b1.x), 0.0f); ho = sg_fma(w2.x, z, ho);
                    z = sg_max(sg_fma(w1.y, g, b1.y), 0.0f); ho = sg_fma(w2.y, z, ho);
                    z = sg_max(sg_fma(w1.z, g, b1.z), 0.0f); ho = sg_fma(w2.z, z, ho);
                    z = sg_max(sg_fma(w1.w, g, b1.w), 0.0f); ho = sg_fma(w2.w, z, ho);
                }
                total = total + ho;
                asm volatile("" : "+v"(total));       // before the next record is requested, or registers spill
            };
            each<HEADS_HERE>([&](auto head) {
                vf4 score[2][KEY_GROUPS];
                each<2>([&](auto hf) { each<KEY_GROUPS>([&](auto t) { score[hf][t] = vf4{0.0f, 0.0f, 0.0f, 0.0f}; }); });
                each<HALF>([&](auto dd) {
                    each<2>([&](auto hf) {
                        constexpr int row = head * DM + hf * HALF + dd;
                        each<KEY_GROUPS>([&](auto t) { score[hf][t] = step4<((head * 2 + hf) * KEY_GROUPS + t) * HALF + dd>(w_keys, query[row / 4][row % 4], score[hf][t]); });
                    });
                });
                int best[2];
#pragma unroll
                for (int hf = 0; hf < 2; hf++) {
                    // the first of the largest scores: the maximum, then the lowest index that has it.  (A running comparison
                    // takes two selects per key, each waiting two clocks for the comparison before it.)
                    float bs = -1e30f;
#pragma unroll
                    for (int q = 0; q < PK; q++) bs = __builtin_fmaxf(bs, score[hf][q / 4][q % 4]);
                    int bi = 0;
#pragma unroll
                    for (int q = PK - 1; q > 0; q--) bi = score[hf][q / 4][q % 4] == bs ? q : bi;
                    best[hf] = score[hf][0][0] == bs ? 0 : bi;
                }
                int e = best[0] * PK + best[1];
                if (e >= NE) e = NE - 1;
                if (live) atomicAdd(&s_cnt[e], 1);
                if (DBG && live) dbg_eidx[((size_t)T.off + i) * NH + own + head] = e;
                if (head > 0) evaluate();
                ho = s_b2[e];
#pragma unroll
                for (int q = 0; q < 3 * (EH / 4); q++) rec[q] = reinterpret_cast<const float4*>(s_exp + e * EXP_STRIDE)[q];
            });
            evaluate();
            if (HEADS) {
                s_head[turn][own][member] = total;       // 0 + the head
                __syncthreads();                         // (every wave has read the GRU state)
                if (own != 0) { turn ^= 1; continue; }
                total = 0.0f;
#pragma unroll
                for (int hh = 0; hh < NH; hh++) total = total + s_head[turn][hh][member];
                turn ^= 1;
                if (live) ((SG_GLOBAL vf4*)T.gru)[i] = vf4{hnew[0], hnew[1], hnew[2], hnew[3]};
            }
            __builtin_amdgcn_s_setprio(0);
            const float smart = g + (rescale * total) / (float)NH;
            if (FWD) {
                if (live) sg::gptr(fwd_smart)[(size_t)T.off + i] = smart;
                continue;
            }

            // ---- mu EMA, Adam moments, decoupled weight decay
            mu = sg_fma(alpha, mu, (1.0f - alpha) * g);
            if (live) sg::gptr(T.mu)[i] = mu;
            const float fg = sg_fma(lamb, mu, smart);
            ea = sg_fma(beta1, ea, (1.0f - beta1) * fg);
            easq = sg_fma(beta2, easq, ((1.0f - beta2) * fg) * fg);
            if (live) {
                sg::gptr(T.ea)[i] = ea;
                sg::gptr(T.easq)[i] = easq;
            }
            const float denom = __builtin_sqrtf(easq / bc2) + eps;
            pv = sg_fma(pv, decay, -((step_size * ea) / denom));
            if (live) sg::store_elem(T.param, dtype, i, pv);
        }
    }
    __syncthreads();
    if (expert_counts != nullptr)
        for (int i = threadIdx.x; i < NE; i += ELEM_THREADS)
            if (s_cnt[i] != 0) atomicAdd(&expert_counts[i], s_cnt[i]);
}


// The same per-element step for any dimensions the reference admits (gru_hidden <= 8, d_model <= 16, any number of
// heads, sub-keys, experts and expert width): every size is a run-time value, the loops over the bounded ones are
// unrolled to their bounds and guarded so that the small arrays stay in registers, the expert tables are read from
// global memory (per-lane gathers through the caches: 3 x E x expert_hidden floats need not fit the LDS), and the
// counts go through an LDS histogram when it fits and global atomics otherwise.  The arithmetic is the specialised
// kernel's, chain for chain (the query projection as plain fma chains: the fp32 matrix instructions compute the same
// chains); the shared reciprocals of the gates apply when gru_hidden is 4, as in the checker.  ctx rows are
// ctx_stride floats apart (d_model of the scan geometry the block was embedded in).
constexpr int MAX_DM = 16, MAX_GH = 8, MAX_HD = 8, CNT_LDS = 4096;
// fwd_smart / fwd_gru (both or neither): the net's forward alone -- smart gradient and new GRU state of every element go
// to these packed arrays, nothing of the optimizer state is read or written (sg2_meta_forward).
template <bool DBG>
__global__ __launch_bounds__(ELEM_THREADS) void k_elem_any(Plan pl, int ctx_stride, int32_t* __restrict__ expert_counts,
                                                           int32_t* __restrict__ dbg_eidx, float* __restrict__ fwd_smart,
                                                           float* __restrict__ fwd_gru) {
    __shared__ int s_cnt[CNT_LDS];
    const int dm = pl.dims.d_model, gh = pl.dims.gru_hidden, H = pl.dims.num_heads, pk = pl.dims.pk_dim;
    const int eh = pl.dims.expert_hidden, E = pl.dims.num_experts, hd = dm / 2;
    const int grl = 2 + 2 * dm + gh, pin = gh + 2 * dm + 2;
    const bool lds_counts = E <= CNT_LDS;
    if (lds_counts)
        for (int i = threadIdx.x; i < E; i += ELEM_THREADS) s_cnt[i] = 0;
    __syncthreads();
    const sg::cfloat_p Wz = sg::as_const(pl.W.w[W_GRU_WZ]), bz = sg::as_const(pl.W.w[W_GRU_BZ]);
    const sg::cfloat_p Wr = sg::as_const(pl.W.w[W_GRU_WR]), br = sg::as_const(pl.W.w[W_GRU_BR]);
    const sg::cfloat_p Wh = sg::as_const(pl.W.w[W_GRU_WH]), bh = sg::as_const(pl.W.w[W_GRU_BH]);
    const sg::cfloat_p Wq = sg::as_const(pl.W.w[W_PEER_Q]);
    const sg::cfloat_p KA = sg::as_const(pl.W.w[W_KEYS_A]), KB = sg::as_const(pl.W.w[W_KEYS_B]);
    const SG_GLOBAL float* W1 = sg::gptr(pl.W.w[W_EXP_W1]);
    const SG_GLOBAL float* B1 = sg::gptr(pl.W.w[W_EXP_B1]);
    const SG_GLOBAL float* W2 = sg::gptr(pl.W.w[W_EXP_W2]);
    const SG_GLOBAL float* B2 = sg::gptr(pl.W.w[W_EXP_B2]);

    for (int tile = blockIdx.x; tile < pl.elem_tiles; tile += gridDim.x) {
        const int ti = sg::upper_seg(sg::as_const(pl.elem_tile_prefix), pl.P, tile);
        const TensorDev& T = pl.tensors[ti];
        const int start = (tile - pl.elem_tile_prefix[ti]) * ELEM_TILE;
        const int cnt = min(ELEM_TILE, T.numel - start);
        const int dtype = T.dtype;
        const float gs = grad_scale(pl, ti);
        const bool has_s = pl.sharp_nonzero[ti] != 0;
        const float alpha = T.alpha, lamb = T.lamb, beta1 = T.beta1, bc2 = T.bc2, step_size = T.step_size;
        const float beta2 = pl.beta2, eps = pl.eps, rescale = pl.rescale, decay = pl.decay;
        for (int k0 = (int)threadIdx.x; k0 < cnt; k0 += ELEM_THREADS) {
            const int i = start + k0;
            const float g = grad_of(T, gs, i);
            const float s = has_s ? sharp_of(T, i) : 0.0f;
            float cf[MAX_DM], cb[MAX_DM], hold[MAX_GH];
            {
                const SG_GLOBAL float* pf = sg::gptr(pl.ctx) + ((size_t)T.off + i) * ctx_stride;
                const SG_GLOBAL float* pb = sg::gptr(pl.ctx) + ((size_t)pl.total + T.off + i) * ctx_stride;
#pragma unroll
                for (int q = 0; q < MAX_DM; q++) { cf[q] = q < dm ? pf[q] : 0.0f; cb[q] = q < dm ? pb[q] : 0.0f; }
#pragma unroll
                for (int q = 0; q < MAX_GH; q++) hold[q] = q < gh ? sg::gptr(T.gru)[(size_t)i * gh + q] : 0.0f;
            }
            // ---- GRU: chain order = bias, g, s, fwd ctx, bwd ctx, h
            float pre_g[2 * MAX_GH], gate[2 * MAX_GH], pre_c[MAX_GH], cand[MAX_GH], hnew[MAX_GH];
#pragma unroll
            for (int j = 0; j < MAX_GH; j++) {
                pre_g[j] = pre_g[MAX_GH + j] = 0.0f;
                if (j < gh) {
                    const sg::cfloat_p wz = Wz + j * grl, wr = Wr + j * grl;
                    float vz = bz[j], vr = br[j];
                    vz = sg_fma(wz[0], g, vz); vz = sg_fma(wz[1], s, vz);
                    vr = sg_fma(wr[0], g, vr); vr = sg_fma(wr[1], s, vr);
#pragma unroll
                    for (int q = 0; q < MAX_DM; q++) if (q < dm) { vz = sg_fma(wz[2 + q], cf[q], vz); vr = sg_fma(wr[2 + q], cf[q], vr); }
#pragma unroll
                    for (int q = 0; q < MAX_DM; q++) if (q < dm) { vz = sg_fma(wz[2 + dm + q], cb[q], vz); vr = sg_fma(wr[2 + dm + q], cb[q], vr); }
#pragma unroll
                    for (int q = 0; q < MAX_GH; q++) if (q < gh) { vz = sg_fma(wz[2 + 2 * dm + q], hold[q], vz); vr = sg_fma(wr[2 + 2 * dm + q], hold[q], vr); }
                    pre_g[j] = vz;
                    pre_g[MAX_GH + j] = vr;
                }
            }
            if (gh == GH) {       // update and reset gates of the four units share one reciprocal
                float in8[2 * GH], out8[2 * GH];
#pragma unroll
                for (int j = 0; j < GH; j++) { in8[j] = pre_g[j]; in8[GH + j] = pre_g[MAX_GH + j]; }
                sg_sigmoid_block(2 * GH, in8, out8);
#pragma unroll
                for (int j = 0; j < MAX_GH; j++) { gate[j] = j < GH ? out8[j] : 0.0f; gate[MAX_GH + j] = j < GH ? out8[GH + j] : 0.0f; }
            } else {
#pragma unroll
                for (int j = 0; j < 2 * MAX_GH; j++) gate[j] = sg_sigmoid(pre_g[j]);
            }
#pragma unroll
            for (int j = 0; j < MAX_GH; j++) {
                pre_c[j] = 0.0f;
                if (j < gh) {
                    const sg::cfloat_p wh = Wh + j * grl;
                    float v = bh[j];
                    v = sg_fma(wh[0], g, v); v = sg_fma(wh[1], s, v);
#pragma unroll
                    for (int q = 0; q < MAX_DM; q++) if (q < dm) v = sg_fma(wh[2 + q], cf[q], v);
#pragma unroll
                    for (int q = 0; q < MAX_DM; q++) if (q < dm) v = sg_fma(wh[2 + dm + q], cb[q], v);
#pragma unroll
                    for (int q = 0; q < MAX_GH; q++) if (q < gh) v = sg_fma(wh[2 + 2 * dm + q], gate[MAX_GH + q] * hold[q], v);
                    pre_c[j] = v;
                }
            }
            if (gh == GH) {
                float in4[GH], out4[GH];
#pragma unroll
                for (int j = 0; j < GH; j++) in4[j] = pre_c[j];
                sg_tanh_block(GH, in4, out4);
#pragma unroll
                for (int j = 0; j < MAX_GH; j++) cand[j] = j < GH ? out4[j] : 0.0f;
            } else {
#pragma unroll
                for (int j = 0; j < MAX_GH; j++) cand[j] = sg_tanh(pre_c[j]);
            }
#pragma unroll
            for (int j = 0; j < MAX_GH; j++) {
                hnew[j] = sg_fma(gate[j], cand[j], (1.0f - gate[j]) * hold[j]);
                if (j < gh) {
                    if (fwd_gru != nullptr) sg::gptr(fwd_gru)[((size_t)T.off + i) * gh + j] = hnew[j];
                    else sg::gptr(T.gru)[(size_t)i * gh + j] = hnew[j];
                }
            }

            // ---- PEER: per head the query (chain order = h, fwd ctx, bwd ctx, g, s), two sub-key arg-maxes, the expert
            float total = 0.0f;
            for (int hh = 0; hh < H; hh++) {
                auto query_row = [&](int row) {
                    const sg::cfloat_p qr = Wq + ((size_t)hh * dm + row) * pin;
                    float v = 0.0f;
#pragma unroll
                    for (int q = 0; q < MAX_GH; q++) if (q < gh) v = sg_fma(qr[q], hnew[q], v);
#pragma unroll
                    for (int q = 0; q < MAX_DM; q++) if (q < dm) v = sg_fma(qr[gh + q], cf[q], v);
#pragma unroll
                    for (int q = 0; q < MAX_DM; q++) if (q < dm) v = sg_fma(qr[gh + dm + q], cb[q], v);
                    v = sg_fma(qr[gh + 2 * dm], g, v);
                    v = sg_fma(qr[gh + 2 * dm + 1], s, v);
                    return v;
                };
                float qa[MAX_HD], qb[MAX_HD];
#pragma unroll
                for (int dd = 0; dd < MAX_HD; dd++) {
                    qa[dd] = qb[dd] = 0.0f;
                    if (dd < hd) { qa[dd] = query_row(dd); qb[dd] = query_row(hd + dd); }
                }
                int best[2];
#pragma unroll
                for (int hf = 0; hf < 2; hf++) {
                    const sg::cfloat_p keys = (hf ? KB : KA) + (size_t)hh * pk * hd;
                    int bi = 0;
                    float bs = -1e30f;
                    for (int q = 0; q < pk; q++) {
                        float dot = 0.0f;
#pragma unroll
                        for (int dd = 0; dd < MAX_HD; dd++) if (dd < hd) dot = sg_fma(hf ? qb[dd] : qa[dd], keys[q * hd + dd], dot);
                        if (dot > bs) { bs = dot; bi = q; }
                    }
                    best[hf] = bi;
                }
                int e = best[0] * pk + best[1];
                if (e >= E) e = E - 1;
                if (lds_counts) atomicAdd(&s_cnt[e], 1);
                else if (expert_counts != nullptr) atomicAdd(&expert_counts[e], 1);
                if (DBG) dbg_eidx[((size_t)T.off + i) * H + hh] = e;
                float ho = B2[e];
                for (int q = 0; q < eh; q++) {
                    const float z = sg_max(sg_fma(W1[(size_t)e * eh + q], g, B1[(size_t)e * eh + q]), 0.0f);
                    ho = sg_fma(W2[(size_t)e * eh + q], z, ho);
                }
                total = total + ho;
            }
            const float smart = g + (rescale * total) / (float)H;
            if (fwd_smart != nullptr) {
                sg::gptr(fwd_smart)[(size_t)T.off + i] = smart;
                continue;
            }

            // ---- mu EMA, Adam moments, decoupled weight decay
            float mu = sg::gptr(T.mu)[i], ea = sg::gptr(T.ea)[i], easq = sg::gptr(T.easq)[i];
            float pv = sg::load_elem(T.param, dtype, i);
            mu = sg_fma(alpha, mu, (1.0f - alpha) * g);
            sg::gptr(T.mu)[i] = mu;
            const float fg = sg_fma(lamb, mu, smart);
            ea = sg_fma(beta1, ea, (1.0f - beta1) * fg);
            easq = sg_fma(beta2, easq, ((1.0f - beta2) * fg) * fg);
            sg::gptr(T.ea)[i] = ea;
            sg::gptr(T.easq)[i] = easq;
            const float denom = __builtin_sqrtf(easq / bc2) + eps;
            pv = sg_fma(pv, decay, -((step_size * ea) / denom));
            sg::store_elem(T.param, dtype, i, pv);
        }
    }
    __syncthreads();
    if (lds_counts && expert_counts != nullptr)
        for (int i = threadIdx.x; i < E; i += ELEM_THREADS)
            if (s_cnt[i] != 0) atomicAdd(&expert_counts[i], s_cnt[i]);
}

}  // namespace

// A wave per head while that takes at most one workgroup per compute unit.  Beyond, the element's chain is shorter still, but
// every 64 elements pay for an LDS fill of 36 KB that otherwise serves 256: 8 small tensors -2.1 us a step, 1000 elements in 3
// tensors -2, 5000 in 4 -2; taken up to twice as many parts, 15 000 in 6 (about 300) no difference, 28 000 in 5 +1.6.  (0.42 M: +62
// with the scalar form.)
constexpr int HEADS_PARTS = 256;
inline bool by_heads(const Plan& pl) { return pl.elem_kind != ELEM_ANY && pl.elem_tiles * (ELEM_TILE / 64) <= HEADS_PARTS; }

// Workgroups of the per-element kernel, and the parts its tiles are cut into.  Large calls: about five workgroups per
// resident slot (768 at three per CU): measured 1.38 / 1.35 / 1.33 / 1.33 / 1.37 ms with 768 / 2048 / 4096 / 8192 / 16384
// workgroups on 24 424 tiles (fewer leave the chip unevenly loaded at the end, more pay the LDS fill too often).  Calls of
// at most 1024 tiles would leave most of the chip idle while some workgroups run four rounds of 256 elements: they take
// rounds as units, spread evenly over at most 1024 resident workgroups.
int elem_grid(const Plan& pl, bool heads, int* split) {
    *split = 1;
    if (heads && by_heads(pl)) {
        *split = ELEM_TILE / 64;
        return pl.elem_tiles * *split;
    }
    if (pl.elem_tiles > 1024 || pl.elem_kind == ELEM_ANY) return pl.elem_tiles < 4096 ? pl.elem_tiles : 4096;
    *split = ELEM_TILE / ELEM_THREADS;
    const int parts = pl.elem_tiles * *split, rounds = (parts + 1023) / 1024;
    return (parts + rounds - 1) / rounds;
}

int launch_elem_forward(const Plan& pl, int32_t* expert_counts, float* smart_out, float* gru_out, hipStream_t st) {
    if (pl.total == 0) return 0;
    int split;
    const int grid = elem_grid(pl, false, &split);
    int32_t* const no_dbg = nullptr;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(ELEM_THREADS), 0, st, pl, expert_counts, no_dbg, smart_out, gru_out, split); };
    if (pl.elem_kind == ELEM_ANY)
        hipLaunchKernelGGL(k_elem_any<false>, dim3(grid), dim3(ELEM_THREADS), 0, st, pl, geo_info(pl.geo).dm, expert_counts, no_dbg, smart_out, gru_out);
    else if (pl.geo == GEO_LARGE) go(k_elem<GeoLarge, 16, false, true>);
    else if (pl.elem_kind == ELEM_FAST4) go(k_elem<GeoDefault, 4, false, true>);
    else go(k_elem<GeoDefault, 16, false, true>);
    SG_LAUNCH_CHECK("k_elem<forward>");
    return 0;
}

int launch_elem(const Plan& pl, int32_t* expert_counts, int32_t* dbg_expert_idx, hipStream_t st) {
    if (pl.total == 0) return 0;
    int split;
    const int grid = elem_grid(pl, dbg_expert_idx == nullptr, &split);
    float* const none = nullptr;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(ELEM_THREADS), 0, st, pl, expert_counts, dbg_expert_idx, none, none, split); };
    if (pl.elem_kind == ELEM_ANY) {
        const int stride = geo_info(pl.geo).dm;
        if (dbg_expert_idx) hipLaunchKernelGGL(k_elem_any<true>, dim3(grid), dim3(ELEM_THREADS), 0, st, pl, stride, expert_counts, dbg_expert_idx, none, none);
        else hipLaunchKernelGGL(k_elem_any<false>, dim3(grid), dim3(ELEM_THREADS), 0, st, pl, stride, expert_counts, dbg_expert_idx, none, none);
    } else if (pl.geo == GEO_LARGE) {
        if (dbg_expert_idx) go(k_elem<GeoLarge, 16, true>);
        else if (by_heads(pl)) go(k_elem<GeoLarge, 16, false, false, true>);
        else go(k_elem<GeoLarge, 16, false>);
    } else if (pl.elem_kind == ELEM_FAST4) {
        if (dbg_expert_idx) go(k_elem<GeoDefault, 4, true>);
        else if (by_heads(pl)) go(k_elem<GeoDefault, 4, false, false, true>);
        else go(k_elem<GeoDefault, 4, false>);
    } else if (dbg_expert_idx) {
        go(k_elem<GeoDefault, 16, true>);
    } else if (by_heads(pl)) {
        go(k_elem<GeoDefault, 16, false, false, true>);
    } else {
        go(k_elem<GeoDefault, 16, false>);
    }
    SG_LAUNCH_CHECK("k_elem");
    return 0;
}

}  // namespace sg2
