// Bidirectional Mamba-3 selective scan over the magnitude-sorted sequence of
// every parameter tensor, all tensors and both directions in each launch.
//
// Replaces the reference's precompute + Blelloch scan kernels
// (csrc/supergrok2_mamba_peer_kernels.cu:289-346, 577-781), the sequential
// kernels (:138-272, :1241-1390), the x_sorted gather (:1882-1906) and the
// scan-output unsort + out_proj (:2057-2060, :917-937).
//
// The sorted sequence of a tensor is cut into chunks of chunk_len timesteps
// (scan order: t ascending for the forward direction, descending for the
// backward one).  One workgroup owns one chunk: one wave for the default geometry, four for the
// large one; a lane owns one RoPE pair p of two columns j, i.e. the states h[j][2p], h[j][2p+1] of both.  (Calls that do
// not fill the chip that way: twice the waves, one column per lane.)
//   k_summary      every chunk but the last of a tensor: 2x2 affine summary
//                  (M,b) of the chunk, accumulated from the identity.  The
//                  recurrence contracts (|A_bar| < 1), so the chunk is walked
//                  backwards in blocks of `window` steps and the walk stops as
//                  soon as every |entry| of the running M, in all lanes, is
//                  below 2^-64: the state entering that block is multiplied
//                  by less than 2^-64, and the summary is (0, b).  A first
//                  attempt covers one block sized from the weights with the
//                  state part only and a norm bound instead of M.
//   k_chunk_prefix start state of each chunk: summaries applied in order to
//                  the carried state of the tensor.
//   k_replay       every chunk replayed from its start state: y = h.C, gate,
//   (k_replay_cols D skip, out_proj, and the 8-float (16-float) context written
//   for the large  straight to the element's original position (the "unsort").
//   geometry and   The last chunk stores the new carried state.
//   small calls)
//   compose_block  (sg2_compose_block.hpp) runs beside the sort's first kernel: the input of a timestep is two numbers (g, s)
//                  and every projection of the block is linear in their 8-float
//                  input projection, so input_proj, in_proj, dt_proj, B_proj and
//                  C_proj are folded into 5 x d_inner coefficient triples per
//                  direction (include/sg2_compose.h).
// Per-timestep projections (x-branch, z, dt, B, C) are evaluated from those
// triples in both passes for tiles of 64 timesteps and staged through LDS
// instead of being materialised in HBM (the reference writes 320 B per
// element per direction).
// The inputs of a timestep come coalesced from the sort's own output: the key
// is |g|, the payload carries the sign of g and the element index, and the
// sharpness has been gathered into sorted order once.
//
// The kernels are bound by fp32 VALU issue, not by HBM: per (timestep, column,
// pair) one shared reciprocal, one sin/cos pair and the 2x2 update.  The
// recurrence loop therefore works on blocks of 8 timesteps: all LDS operands of
// the block are fetched first, the state-independent coefficients of the 8
// steps are computed as independent instruction streams, and only the short
// h-update chain is serial.  The A_bar denominators of a lane's 8 steps are
// inverted together (one division per block, sg_abar_block_*).  When every
// lane of the wave holds a small rotation angle the sin/cos range reduction is
// skipped (bit-identical results, see sg_sincos_small); when every angle of
// the block is below 0.3 a shorter polynomial pair is used (sg_sincos_tiny,
// not bit-identical to the general form: the choice depends on the angles only
// and the CPU checker makes the same one).
// Where the inputs are small (the usual case: sg2_taylor_ok, sg2_poly_ok in sg2_compose.h) the step size and the gate
// of a tile come from cubic Taylor polynomials around their zero-input arguments, and A_bar, sin and cos of a block
// from per-lane polynomials in dt - dt0; the forms above serve the remaining tiles and blocks.  The ragged tile at the end
// of a tensor takes the polynomials like any other (its missing steps are zero inputs whose effect on the state is taken
// back): single steps with their own divisions were 10 % of a step whose tensors are all below 256 elements.
// For the bilevel pass k_replay<G, true> also stores the state entering every
// HT_STEP-th step (Plan::htile), which the adjoint kernels restart from.
#include <type_traits>
#include "sg2_internal.hpp"
#include "sg2_pair_sums.hpp"
#include "../../include/sg2_compose.h"

namespace sg2 {
namespace {

constexpr int LDS_STRIDE = SCAN_TT + 4;   // [row][timestep] rows: 16-byte aligned (the recurrence fetches 4 timesteps per LDS read)
                                          // and padded so the 8 rows a wave reads start 4 banks apart
typedef float f32x4 __attribute__((ext_vector_type(4)));
#ifndef SG2_SCAN_UB
#define SG2_SCAN_UB 8
#endif
constexpr int UB = SG2_SCAN_UB;           // timesteps per unrolled block of the recurrence
static_assert(UB % 4 == 0 && SCAN_TT % UB == 0 && SCAN_TT == 64, "blocks are fetched 4 timesteps per LDS read; one ballot covers a tile");
static_assert(HT_STEP % UB == 0 && SCAN_TT % HT_STEP == 0, "kept states fall on block borders");
template <int HP>
__device__ __forceinline__ float pair_tree_max(float f) {
    f = sg_max(f, dpp_quad_swap1(f));
    f = sg_max(f, dpp_quad_swap2(f));
    f = sg_max(f, dpp_half_mirror(f));
    if (HP == 16) f = sg_max(f, dpp_row_mirror(f));
    return f;
}

// scan state of one lane: OUT -> (he,ho) only; summary -> also the two columns of M
struct LaneState {
    float he, ho, c0e, c0o, c1e, c1o;
};
// the lane's pair as polynomials in dt - dt0 (sg2_abar_poly, sg2_sincos_poly): dt0 = step size of its column for a zero input
// The summary pass keeps A_bar and sin/cos apart (its bound needs the A_bar); the output pass holds the four products.
template <bool OUT>
struct LanePoly {
    float dt0, pe[4], po[4], qs[3], qc[3];
};
template <>
struct LanePoly<true> {
    float dt0, k[12];
};

// LITE (summary pass only): the state part alone, and in c0e the running product of max(|A_bar_e|, |A_bar_o|), a bound
// on the norm of the 2x2 part that is not formed
template <bool OUT, bool LITE = false>
__device__ __forceinline__ void step_update(LaneState& S, float ae, float ao, float sn, float cs, float be, float bo) {
    if (!OUT && LITE) S.c0e = S.c0e * sg_max(sg_abs(ae), sg_abs(ao));
    if (!OUT && !LITE) {
        float re = sg_fma(S.c0e, cs, -(S.c0o * sn)), ro = sg_fma(S.c0o, cs, S.c0e * sn);
        S.c0e = ae * re;
        S.c0o = ao * ro;
        re = sg_fma(S.c1e, cs, -(S.c1o * sn));
        ro = sg_fma(S.c1o, cs, S.c1e * sn);
        S.c1e = ae * re;
        S.c1o = ao * ro;
    }
    const float re = sg_fma(S.he, cs, -(S.ho * sn));
    const float ro = sg_fma(S.ho, cs, S.he * sn);
    S.he = sg_fma(ae, re, be);
    S.ho = sg_fma(ao, ro, bo);
}

// UB consecutive timesteps (all valid): coefficients first, then the serial chain.  ux = dt * x-branch
// (formed once per timestep in phase A).  The A_bar of the block share one reciprocal per lane
// (sg_abar_block_*) unless some lane of the wave has a product of denominators too large for it.
// ANGLE: 0 full sin/cos, 1 sg_sincos_small (bit-identical to 0), 2 sg_sincos_tiny_dt (its own values, polynomials in dt),
// 3: every timestep of the block has passed sg2_poly_ok: A_bar, sin and cos from the lane's polynomials in dt - dt0.
template <int HP, bool OUT, int ANGLE, bool LITE = false>
__device__ __forceinline__ void block_steps(LaneState& S, const float (&dt)[UB], const float (&ux)[UB], const float (&Be)[UB],
                                            const float (&Bo)[UB], const float (&Ce)[UB], const float (&Co)[UB], float hAe,
                                            float hAo, float freq, const LanePoly<OUT>& LP, float (&y)[UB]) {
    float ae[UB], ao[UB], sn[UB], cs[UB], be[UB], bo[UB];
    if constexpr (ANGLE == 3 && OUT) {
        // the four products of the update as quadratics: ae = P1, sn = N2, ao = P3, cs = P4 (see the update below)
#pragma unroll
        for (int u = 0; u < UB; u++) {
            const float d = dt[u] - LP.dt0;
            ae[u] = sg2_poly2(LP.k, d);
            sn[u] = sg2_poly2(LP.k + 3, d);
            ao[u] = sg2_poly2(LP.k + 6, d);
            cs[u] = sg2_poly2(LP.k + 9, d);
        }
    } else if constexpr (ANGLE == 3) {
#pragma unroll
        for (int u = 0; u < UB; u++) {
            const float d = dt[u] - LP.dt0;
            ae[u] = sg2_poly3(LP.pe, d);
            ao[u] = sg2_poly3(LP.po, d);
            sn[u] = sg2_poly2(LP.qs, d);
            cs[u] = sg2_poly2(LP.qc, d);
        }
    } else {
        float d_e[UB], d_o[UB], P[UB];
        const float last = sg_abar_block_prefix(UB, dt, hAe, hAo, d_e, d_o, P);
        if (__builtin_amdgcn_ballot_w64(!(last < SG_ABAR_BLOCK_LIMIT)) == 0) {
            sg_abar_block_finish(UB, d_e, d_o, P, ae, ao);
        } else {
#pragma unroll
            for (int u = 0; u < UB; u++) sg_abar_pair(dt[u], hAe, hAo, &ae[u], &ao[u]);
        }
    }
    float tcoef[6];             // tiny-angle sin/cos of this lane's pair as polynomials in dt (formed here: a block that comes this way is the exception)
    if (ANGLE == 2) sg_sincos_tiny_coef(freq, tcoef);
#pragma unroll
    for (int u = 0; u < UB; u++) {
        if (ANGLE == 2) sg_sincos_tiny_dt(dt[u], tcoef, &sn[u], &cs[u]);
        else if (ANGLE == 1) sg_sincos_small(dt[u] * freq, &sn[u], &cs[u]);
        else if (ANGLE == 0) sg_sincos(dt[u] * freq, &sn[u], &cs[u]);
        be[u] = ux[u] * Be[u];
        bo[u] = ux[u] * Bo[u];
    }
#pragma unroll
    for (int u = 0; u < UB; u++) {
        if constexpr (ANGLE == 3 && OUT) {
            const float he = sg_fma(ae[u], S.he, sg_fma(sn[u], S.ho, be[u]));      // P1 he + N2 ho + b_e
            S.ho = sg_fma(ao[u], S.ho, sg_fma(cs[u], S.he, bo[u]));                // P3 ho + P4 he + b_o
            S.he = he;
        } else {
            step_update<OUT, LITE>(S, ae[u], ao[u], sn[u], cs[u], be[u], bo[u]);
        }
        if (OUT) y[u] = sg_fma(S.ho, Co[u], S.he * Ce[u]);
    }
    if (OUT) {
        static_assert(UB == 8, "block_pair_sums folds blocks of 8 steps");
        block_pair_sums<HP>(y);
    }
}

// How the waves of a chunk share its recurrences: a lane owns one RoPE pair of CL columns (two, or one where the call has
// too few chunks to fill the chip with waves of two), so a chunk takes THREADS / (64 CL) waves, wave w the columns
// CPW w .. CPW w + CPW - 1: lane (jl, p) = (lane / HP, lane % HP) pair p of columns CPW w + jl (and CPW w + CPH + jl).
template <class G, int CL>
struct Split {
    static constexpr int WAVES = G::THREADS / (64 * CL);
    static constexpr int CPW = G::DI / WAVES;       // columns (and rows of B and C) of a wave
    static constexpr int CPH = CPW / CL;            // ... of one of a lane's columns over the lanes
    static constexpr int SPL = CPW;                 // row owners: lane (row r, part q) takes SPL consecutive timesteps of row r
    static_assert(CPH * G::HP == 64 && G::DI == G::DS && SPL * (64 / CPW) == SCAN_TT && SPL % 4 == 0, "64 lanes: CPH columns x HP pairs, CPW rows x parts");
};
// Where row r of B or C lies: the even rows first.  The lanes of a wave read rows 2 p and 2 p + 1 of all pairs p; with 16 pairs
// the even rows in their own order would start 8 banks apart and meet on half of them.
template <class G>
__device__ __forceinline__ int bc_slot(int r) { return (r & 1) * G::HP + (r >> 1); }

// Projections of one timestep, for a tile that does not run on the polynomials throughout (row owners form the usual tile):
// the lane computes its wave's rows of every group for its timestep.  Step size, dt * x-branch, B and C go to LDS for
// the recurrence; the skip terms D * x-branch stay in the lane's registers, because the lane that forms them is the one
// that uses them after the recurrence, and for the same reason the gates are not formed here at all (gates_of).
// coef: [group][row] composed triple + one more float (D next to the x-branch triple); tay: [step size | gate][row][4].
// c0: first column of the wave.  angle[h]: bit 0 / 1 = every rotation angle of columns c0 + CPH h .. + CPH - 1 at this timestep is
// small enough for sg_sincos_small / sg_sincos_tiny (fmax: per column, the largest |rope frequency| of its pairs; dt >= 0
// and rounding is monotone, so dt*fmax < limit is the same statement as |dt*freq| < limit for all pairs).
// TAYLOR: every timestep of the tile has passed sg2_taylor_ok: step size and gate come from their cubic Taylor polynomials.
// HAS_S is false for a tensor whose sharpness is all zero: fma(c_s, 0, c_0) is c_0 itself, so the term is skipped.
// SLOTTED: rows of B and C at bc_slot.
template <class G, int CL, bool OUT, bool SLOTTED, bool HAS_S, bool TAYLOR>
__device__ __forceinline__ void project_steps(float g, float s, int tu, int c0, const float* s_coef, const float* s_tay, const float* s_fmax, float* s_dt,
                                              float* s_ux, float* s_B, float* s_C, float (&dxv)[Split<G, CL>::CPW], int (&angle)[CL]) {
    constexpr int DI = G::DI, CPW = Split<G, CL>::CPW, CPH = Split<G, CL>::CPH;
    auto delta = [&](const f32x4 t) { return HAS_S ? sg_fma(t[0], g, t[1] * s) : t[0] * g; };
    auto poly = [&](const f32x4 t, float d) { return sg_fma(sg_fma(sg_fma(t[3], d, t[2]), d, t[1]), d, t[0]); };
    auto eval = [&](const f32x4 t) { return sg_fma(t[0], g, HAS_S ? sg_fma(t[1], s, t[2]) : t[2]); };
    auto coef = [&](int group, int row) { return *reinterpret_cast<const f32x4*>(s_coef + (group * DI + row) * 4); };
#pragma unroll
    for (int h = 0; h < CL; h++) {
        bool small = true, tiny = true;
#pragma unroll
        for (int q = 0; q < CPH; q++) {
            const int jj = c0 + CPH * h + q;
            const f32x4 cd = coef(SG2_COMP_DT, jj);
            const float dtv = TAYLOR ? poly(*reinterpret_cast<const f32x4*>(s_tay + jj * 4), delta(cd)) : sg_softplus(eval(cd));
            const float amax = dtv * s_fmax[jj];
            small = small && (amax < SG_SINCOS_SMALL_LIMIT);
            tiny = tiny && (amax < SG_SINCOS_TINY_LIMIT);
            const f32x4 cx = coef(SG2_COMP_XB, jj);       // x-branch coefficients; [3] = D of this column
            const float xbv = eval(cx);
            s_dt[jj * LDS_STRIDE + tu] = dtv;
            s_ux[jj * LDS_STRIDE + tu] = dtv * xbv;
            if (OUT) dxv[CPH * h + q] = cx[3] * xbv;
        }
        angle[h] = (small ? 1 : 0) | (tiny ? 2 : 0);
    }
#pragma unroll
    for (int q = 0; q < CPW; q++) {
        const int ss = c0 + q, at = SLOTTED ? bc_slot<G>(ss) : ss;
        s_B[at * LDS_STRIDE + tu] = eval(coef(SG2_COMP_B, ss));
        if (OUT) s_C[at * LDS_STRIDE + tu] = eval(coef(SG2_COMP_C, ss));
    }
}
// The gates silu(z) of the wave's columns at one timestep: Taylor polynomials for a tile that qualifies, else one column of
// every lane at a time (CPH of them) on one shared reciprocal, the groups the checker forms.
template <class G, int CL, bool HAS_S, bool TAYLOR>
__device__ __forceinline__ void gates_of(float g, float s, int c0, const float* s_coef, const float* s_tay, float (&gv)[Split<G, CL>::CPW]) {
    constexpr int DI = G::DI, CPH = Split<G, CL>::CPH;
    auto delta = [&](const f32x4 t) { return HAS_S ? sg_fma(t[0], g, t[1] * s) : t[0] * g; };
    auto poly = [&](const f32x4 t, float d) { return sg_fma(sg_fma(sg_fma(t[3], d, t[2]), d, t[1]), d, t[0]); };
    auto eval = [&](const f32x4 t) { return sg_fma(t[0], g, HAS_S ? sg_fma(t[1], s, t[2]) : t[2]); };
    auto coef = [&](int row) { return *reinterpret_cast<const f32x4*>(s_coef + (SG2_COMP_Z * DI + row) * 4); };
    if (TAYLOR) {
#pragma unroll
        for (int q = 0; q < CL * CPH; q++) gv[q] = poly(*reinterpret_cast<const f32x4*>(s_tay + (DI + c0 + q) * 4), delta(coef(c0 + q)));
    } else {
        static_assert(CPH <= 8, "sg_silu_block takes at most 8 values");
#pragma unroll
        for (int h = 0; h < CL; h++) {
            float zv[CPH], out[CPH];
#pragma unroll
            for (int q = 0; q < CPH; q++) zv[q] = eval(coef(c0 + CPH * h + q));
            sg_silu_block(CPH, zv, out);
#pragma unroll
            for (int q = 0; q < CPH; q++) gv[CPH * h + q] = out[q];
        }
    }
}

// Projections of a whole tile that runs on the polynomials (every step size and gate inside its Taylor range, every
// block of the recurrence on the lane polynomials), formed by lanes that own ROWS instead of timesteps: lane (column cj,
// quarter cq) forms dt - dt0, dt * x-branch and D * x-branch of column cj for timesteps 16 cq .. 16 cq + 15, and lane
// (row br, half bh) one row of B (br < 16) or C for timesteps 32 bh .. 32 bh + 31.  A row's coefficients are then four
// 16-byte LDS reads per tile and lane instead of one per (timestep, row), the 64 (g, s) of the tile travel through the
// four padding floats of the rows of s_B / s_C, and the results leave as 16-byte LDS writes: the same arithmetic as
// the timestep-per-lane form with a fifth of its LDS instructions.  Every value is formed by the expressions of
// project_steps (Taylor form) on the same operands, so it is the same float; the step-size row receives dt - dt0, which
// is what the lane polynomials of the recurrence take.
// dxk: this lane's 16 skips D * x-branch of (column cj, timestep 16 cq + k), kept for gate_rows.
// DELTA false, for a tile whose steps are inside the Taylor range but not all on the polynomials (with timesteps per lane there, 3.1 M
// bf16 elements took 1020 us a step for 991, 0.42 M 248 for 243, 25 M the same): the step-size row receives dt itself,
// and angle the lane's verdict on the two blocks of its timesteps (bits 0 / 1: every angle of its column small enough for
// sg_sincos_small / sg_sincos_tiny in the first, bits 2 / 3 in the second; see project_steps).
template <class G, bool HAS_S, bool DELTA>
__device__ __forceinline__ void project_rows(float g, float s, int tid, const float* s_coef, const float* s_tay, const float* s_fmax, float* s_dt,
                                             float* s_ux, float* s_B, float* s_C, float (&dxk)[G::DI], int& angle) {
    constexpr int DI = G::DI, DS = G::DS;
    static_assert(DI == 16 && DS == 16 && SCAN_TT == 64 && LDS_STRIDE == SCAN_TT + 4, "64 lanes: 16 columns x 4 quarters, 32 rows x 2 halves");
    auto delta = [&](const f32x4 t, float gg, float ss) { return HAS_S ? sg_fma(t[0], gg, t[1] * ss) : t[0] * gg; };
    auto poly = [&](const f32x4 t, float d) { return sg_fma(sg_fma(sg_fma(t[3], d, t[2]), d, t[1]), d, t[0]); };
    auto eval = [&](const f32x4 t, float gg, float ss) { return sg_fma(t[0], gg, HAS_S ? sg_fma(t[1], ss, t[2]) : t[2]); };
    auto coef = [&](int group, int row) { return *reinterpret_cast<const f32x4*>(s_coef + (group * DI + row) * 4); };
    s_B[(tid >> 2) * LDS_STRIDE + SCAN_TT + (tid & 3)] = g;      // timestep t: padding float t % 4 of row t / 4
    if (HAS_S) s_C[(tid >> 2) * LDS_STRIDE + SCAN_TT + (tid & 3)] = s;
    __syncthreads();
    auto inputs = [&](int t4, f32x4& g4, f32x4& s4) {            // (g, s) of timesteps 4 t4 .. 4 t4 + 3
        g4 = *reinterpret_cast<const f32x4*>(s_B + t4 * LDS_STRIDE + SCAN_TT);
        s4 = HAS_S ? *reinterpret_cast<const f32x4*>(s_C + t4 * LDS_STRIDE + SCAN_TT) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    {
        const int cj = tid & 15, cq = tid >> 4;
        const f32x4 cd = coef(SG2_COMP_DT, cj), cx = coef(SG2_COMP_XB, cj);
        const f32x4 tp = *reinterpret_cast<const f32x4*>(s_tay + cj * 4);
        float* const r_dt = s_dt + cj * LDS_STRIDE + 16 * cq;
        float* const r_ux = s_ux + cj * LDS_STRIDE + 16 * cq;
        const float fmax = DELTA ? 0.0f : s_fmax[cj];
        bool small[2] = {true, true}, tiny[2] = {true, true};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            f32x4 g4, s4, d4, u4;
            inputs(4 * cq + i, g4, s4);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float dtv = poly(tp, delta(cd, g4[e], s4[e]));
                const float xbv = eval(cx, g4[e], s4[e]);
                d4[e] = DELTA ? dtv - tp[0] : dtv;
                u4[e] = dtv * xbv;
                dxk[4 * i + e] = cx[3] * xbv;
                if (!DELTA) {
                    small[i / 2] = small[i / 2] && (dtv * fmax < SG_SINCOS_SMALL_LIMIT);
                    tiny[i / 2] = tiny[i / 2] && (dtv * fmax < SG_SINCOS_TINY_LIMIT);
                }
            }
            *reinterpret_cast<f32x4*>(r_dt + 4 * i) = d4;
            *reinterpret_cast<f32x4*>(r_ux + 4 * i) = u4;
        }
        if (!DELTA) angle = (small[0] ? 1 : 0) | (tiny[0] ? 2 : 0) | (small[1] ? 4 : 0) | (tiny[1] ? 8 : 0);
    }
    {
        const int br = tid & 31, bh = tid >> 5;
        const f32x4 cb = coef(br < DS ? SG2_COMP_B : SG2_COMP_C, br & (DS - 1));
        float* const r_bc = (br < DS ? s_B : s_C) + (br & (DS - 1)) * LDS_STRIDE + 32 * bh;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            f32x4 g4, s4, v4;
            inputs(8 * bh + i, g4, s4);
#pragma unroll
            for (int e = 0; e < 4; e++) v4[e] = eval(cb, g4[e], s4[e]);
            *reinterpret_cast<f32x4*>(r_bc + 4 * i) = v4;
        }
    }
}

// The row owners' part after the recurrence: y of (column cj, timesteps 16 cq .. 16 cq + 15) becomes
// y * gate + D * x-branch in place.  The gates are formed here, from the (g, s) that project_rows left in the padding floats, so that they do
// not occupy 16 registers during the recurrence.
template <class G, bool HAS_S>
__device__ __forceinline__ void gate_rows(int tid, const float* s_coef, const float* s_tay, const float* s_B, const float* s_C, float* s_y,
                                          const float (&dxk)[G::DI]) {
    constexpr int DI = G::DI;
    auto delta = [&](const f32x4 t, float gg, float ss) { return HAS_S ? sg_fma(t[0], gg, t[1] * ss) : t[0] * gg; };
    auto poly = [&](const f32x4 t, float d) { return sg_fma(sg_fma(sg_fma(t[3], d, t[2]), d, t[1]), d, t[0]); };
    const int cj = tid & 15, cq = tid >> 4;
    const f32x4 cz = *reinterpret_cast<const f32x4*>(s_coef + (SG2_COMP_Z * DI + cj) * 4);
    const f32x4 tz = *reinterpret_cast<const f32x4*>(s_tay + (DI + cj) * 4);
    float* const r_y = s_y + cj * LDS_STRIDE + 16 * cq;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const f32x4 g4 = *reinterpret_cast<const f32x4*>(s_B + (4 * cq + i) * LDS_STRIDE + SCAN_TT);
        const f32x4 s4 = HAS_S ? *reinterpret_cast<const f32x4*>(s_C + (4 * cq + i) * LDS_STRIDE + SCAN_TT) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        f32x4 y4 = *reinterpret_cast<const f32x4*>(r_y + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; e++) y4[e] = sg_fma(y4[e], poly(tz, delta(cz, g4[e], s4[e])), dxk[4 * i + e]);
        *reinterpret_cast<f32x4*>(r_y + 4 * i) = y4;
    }
}

// UB steps of all columns of a lane on the products, dt - dt0 given (what block_steps<HP, true, 3> does for one column
// with dt), written as one straight-line block so that two independent recurrences interleave.
// OUT false (summary): the states alone.  PARTIAL: the steps from `rem` on lie beyond the end of the tensor; they are
// computed (on projections of zero inputs) and their effect on the state is taken back.
template <int HP, bool LINEAR, bool OUT, bool PARTIAL, int CL>
__device__ __forceinline__ void block_steps_cols(LaneState (&S)[CL], const float (&dt)[CL][UB], const float (&ux)[CL][UB], const float (&Be)[UB],
                                                 const float (&Bo)[UB], const float (&Ce)[UB], const float (&Co)[UB], const LanePoly<true> (&LP)[CL],
                                                 int rem, float (&y)[CL][UB]) {
    float keep[2 * CL];
#pragma unroll
    for (int u = 0; u < UB; u++) {
#pragma unroll
        for (int h = 0; h < CL; h++) {
            const float d = dt[h][u];
            const float p1 = LINEAR ? sg2_poly1(LP[h].k, d) : sg2_poly2(LP[h].k, d);
            const float n2 = LINEAR ? sg2_poly1(LP[h].k + 3, d) : sg2_poly2(LP[h].k + 3, d);
            const float p3 = LINEAR ? sg2_poly1(LP[h].k + 6, d) : sg2_poly2(LP[h].k + 6, d);
            const float p4 = LINEAR ? sg2_poly1(LP[h].k + 9, d) : sg2_poly2(LP[h].k + 9, d);
            const float be = ux[h][u] * Be[u], bo = ux[h][u] * Bo[u];
            const float he = sg_fma(p1, S[h].he, sg_fma(n2, S[h].ho, be));      // P1 he + N2 ho + b_e
            S[h].ho = sg_fma(p3, S[h].ho, sg_fma(p4, S[h].he, bo));            // P3 ho + P4 he + b_o
            S[h].he = he;
            if (OUT) y[h][u] = sg_fma(S[h].ho, Co[u], S[h].he * Ce[u]);
        }
        if (PARTIAL && u == rem - 1) {
#pragma unroll
            for (int h = 0; h < CL; h++) { keep[2 * h] = S[h].he; keep[2 * h + 1] = S[h].ho; }
        }
    }
    if (PARTIAL) {
#pragma unroll
        for (int h = 0; h < CL; h++) { S[h].he = keep[2 * h]; S[h].ho = keep[2 * h + 1]; }
    }
    if (OUT) {
#pragma unroll
        for (int h = 0; h < CL; h++) block_pair_sums<HP>(y[h]);
    }
}

// The replay of the default geometry as ONE wave per chunk: lane (jl, p) owns RoPE pair p of the two columns jl and
// jl + 8.  The lanes that need the same B / C entries of a timestep are then 8, and each entry a lane fetches from LDS
// feeds two recurrences: a third less LDS traffic per step than with a column per lane of two waves -- the pass was bound
// by the LDS queue and the vector ALU together, and the B / C fetches alone were a fifth of
// its time.  A single wave also needs no workgroup barrier between the phases of a tile (its LDS accesses execute in
// program order), forms the 16 gated outputs of a timestep once, and holds all eight context
// entries of its timestep: the two 16-byte stores of an element are adjacent in one lane and leave as one 32-byte
// write.  Columns jl + 8 h of all lanes form a group that decides together (angle masks, the shared reciprocals, gates eight
// at a time), as in the checker.
// A tile has three lane roles.  Recurrence (phase B): lane (jl, p) as above.  Timestep: lane t loads the inputs of
// timestep t, votes on the form the tile takes, and at the end multiplies its 16 gated outputs by out_proj and stores
// its element's row.  Row owner (the usual tile, on the polynomials throughout): lane (column, quarter of the tile)
// forms that column's projections before the recurrence and gates its outputs after it (project_rows, gate_rows);
// other tiles keep the timestep-per-lane projections (project_steps, gates_of).
// KEEP (bilevel pass): also store the state entering every HT_STEP-th step for the adjoint kernels, and the gated outputs
// where they are asked for.  (5.9 ms for 25 M elements; 7.1 as a variant of the two-wave kernel.)
template <class G, bool KEEP>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_replay(Plan pl) {
    constexpr int DM = G::DM, DS = G::DS, DI = G::DI, HP = G::HP, LANES = G::THREADS;
    static_assert(G::PARTS == 2 && LANES == 128 && HP == 8, "two columns per lane of one wave");
    constexpr bool OUT = true;
    __shared__ __attribute__((aligned(16))) float s_dt[DI * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) float s_ux[DI * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) float s_B[DS * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) float s_C[DS * LDS_STRIDE];
    float* const s_y = s_dt;      // y of column j goes where dt of column j was: both are touched by the same lanes, in program order
    __shared__ float s_fmax[DI];
    __shared__ __attribute__((aligned(16))) float s_coef[SG2_COMP_GROUPS * DI * 4];   // [group][row]: composed triple, D beside the x-branch's
    __shared__ __attribute__((aligned(16))) float s_tay[2 * DI * 4];                  // [step size | gate][row]: cubic Taylor polynomials
    __shared__ __attribute__((aligned(16))) float s_wout[DM * DI];
    // four arrays of 16 x 68 floats and 2.4 KB of tables: 19.8 KB, eight workgroups (two waves per SIMD) share a compute unit

    const int per_dir = pl.chunks;
    const int dir = (int)blockIdx.x >= per_dir ? 1 : 0;
    const int cidx = (int)blockIdx.x - dir * per_dir;
    const sg::cint_p prefix = sg::as_const(pl.chunk_prefix);
    const sg::Seg seg = sg::find_seg(prefix, pl.P, cidx);
    const int ti = seg.i;
    const int c = cidx - seg.first;
    const TensorDev& T = pl.tensors[ti];
    const int N = T.numel, off = T.off;
    const int u0 = c * pl.chunk_len;
    const int u1 = min(u0 + pl.chunk_len, N);
    const uint32_t* __restrict__ skey = pl.keys[0] + off;
    const int32_t* __restrict__ sval = pl.vals[0] + off;
    const float* __restrict__ ssrt = pl.ssorted + off;
    const bool has_s = __builtin_amdgcn_readfirstlane(pl.sharp_nonzero[ti]) != 0;

    const int tid = threadIdx.x;
    const int tu = tid;                      // projection role: timestep of the tile
    const int jl = tid >> 3, p = tid & 7;    // scan role: pair p of columns jl and jl + 8
    const float* alog = pl.W.w[dir ? W_B_ALOG : W_F_ALOG];
    const float* rope = pl.W.w[dir ? W_B_ROPE : W_F_ROPE];
    // -A/2 with A = -exp(A_log) of the two poles of a pair, and its frequency, in registers (256 now): with module-made poles about half
    // of the blocks of ordinary gradients take a form that needs them, and forming them again in each, two loads and two
    // exponentials, cost 6 to 10 % of a step (3.1 M bf16 1112 -> 1020 us, 0.42 M 263 -> 248, wide geometry 628 -> 566; 25 M the same).
    float poles[2][3];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        poles[h][0] = -0.5f * -sg_exp(alog[(jl + 8 * h) * DS + 2 * p]);
        poles[h][1] = -0.5f * -sg_exp(alog[(jl + 8 * h) * DS + 2 * p + 1]);
        poles[h][2] = rope[(jl + 8 * h) * HP + p];
        asm("" : "+v"(poles[h][0]), "+v"(poles[h][1]), "+v"(poles[h][2]));       // (keeps the compiler from forming them where they are used)
    }
    auto pole_e = [&](int h) { return poles[h][0]; };
    auto pole_o = [&](int h) { return poles[h][1]; };
    auto rope_f = [&](int h) { return poles[h][2]; };
    LanePoly<true> LP[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        LP[h].dt0 = pl.comp[2 * SG2_COMP_GROUPS * G::ROWS * 3 + dir * 2 * G::ROWS * 4 + (jl + 8 * h) * 4];
        sg2_pair_products(LP[h].dt0, pole_e(h), pole_o(h), rope_f(h), LP[h].k);
    }
    {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float f = pair_tree_max<HP>(sg_abs(rope_f(h)));
            if (p == 0) s_fmax[jl + 8 * h] = f;
        }
        const float* comp = pl.comp + dir * (SG2_COMP_GROUPS * G::ROWS * 3);
        const float* tay = pl.comp + 2 * SG2_COMP_GROUPS * G::ROWS * 3 + dir * 2 * G::ROWS * 4;
        const float* Dw = pl.W.w[dir ? W_B_D : W_F_D];
        for (int i = tid; i < SG2_COMP_GROUPS * DI; i += 64) {
            const float* t = comp + i * 3;
            *reinterpret_cast<f32x4*>(s_coef + i * 4) = f32x4{t[0], t[1], t[2], i / DI == SG2_COMP_XB ? Dw[i % DI] : 0.0f};
        }
        for (int i = tid; i < 2 * DI * 4; i += 64) s_tay[i] = tay[i];
        s_wout[tid] = pl.W.w[dir ? W_B_OUT : W_F_OUT][tid];
        s_wout[tid + 64] = pl.W.w[dir ? W_B_OUT : W_F_OUT][tid + 64];
        __syncthreads();
    }
    const sg::cfloat_p lim = sg::as_const(pl.comp) + 2 * SG2_COMP_GROUPS * G::ROWS * 3 + 2 * 2 * G::ROWS * 4;
    const float cmax_g = lim[2 * dir], cmax_s = lim[2 * dir + 1];
    const float kpoly_g = lim[8 + 2 * dir], kpoly_s = lim[8 + 2 * dir + 1];

    LaneState S[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        S[h] = {0.0f, 0.0f, 1.0f, 0.0f, 0.0f, 1.0f};
        const int lane = tid + 64 * h;       // (column jl + 8 h, pair p) in the order of the summaries and start states
        if (c > 0 && __builtin_amdgcn_readfirstlane(*pl.contracted) != 0) {
            const float* sm = pl.summaries + (size_t)(dir * pl.wchunks + pl.wchunk_prefix[ti] + c - 1) * 6 * LANES;
            S[h].he = sm[4 * LANES + lane];
            S[h].ho = sm[5 * LANES + lane];
        } else if (T.nchunks == 1) {       // nothing before it: the carried state itself (no other workgroup writes it)
            const float* st = dir ? T.mbwd : T.mfwd;
            const int j = jl + 8 * h;
            if (j < pl.st_di && 2 * p < pl.st_ds) {
                S[h].he = st[j * pl.st_ds + 2 * p];
                S[h].ho = st[j * pl.st_ds + 2 * p + 1];
            }
        } else {
            const float* hs = pl.hstart + ((size_t)(dir * pl.chunks + cidx) * 2) * LANES;
            S[h].he = hs[lane];
            S[h].ho = hs[LANES + lane];
        }
    }

    const bool in_order = KEEP && sorted_rows(pl);
    uint32_t nx_key = 0;
    int32_t nx_val = 0;
    float nx_sh = 0.0f;
    auto load_inputs = [&](int tile0) {
        const int u = tile0 + tu;
        if (u < u1) {
            const int t = dir ? (N - 1 - u) : u;
            nx_key = skey[t];
            nx_val = sval[t];
            nx_sh = has_s ? ssrt[t] : 0.0f;
        }
    };
    load_inputs(u0);
    // The context row of a timestep leaves one tile late, after the next tile's inputs have arrived: the counter that
    // tells a wave that its loads have landed also counts its stores, in order, so a store issued just before that
    // wait would make every tile wait for a scattered write to be acknowledged.
    static_assert(DM == 8, "two 16-byte stores per lane");
    float4 held[2];
    float4* held_dst = nullptr;
    auto flush = [&]() {
        if (held_dst != nullptr) {
            held_dst[0] = held[0];
            held_dst[1] = held[1];
        }
    };
    for (int tile0 = u0; tile0 < u1; tile0 += SCAN_TT) {
        const int cnt = min(SCAN_TT, u1 - tile0);
        // ---------------- phase A: projections of SCAN_TT timesteps -> LDS (both halves of every output group)
        const uint32_t kbits = nx_key;
        const int32_t v = nx_val;
        const float shv = nx_sh;
        const bool valid = tile0 + tu < u1;
        asm volatile("" : : "v"(kbits), "v"(v), "v"(shv) : "memory");      // the wait for this tile's inputs goes here, before the stores
        flush();
        if (tile0 + SCAN_TT < u1) load_inputs(tile0 + SCAN_TT);
        int orig = v & 0x7fffffff;
        orig = ((unsigned)orig < (unsigned)N) ? orig : 0;   // never index outside the tensor
        const float g = valid ? sg_i2f((int32_t)kbits | (v & (int32_t)0x80000000)) : 0.0f;
        const float sh = valid ? shv : 0.0f;
        const unsigned long long notpoly = __builtin_amdgcn_ballot_w64(!sg2_poly_ok(kpoly_g, kpoly_s, g, sh));
        const unsigned long long notlin =
            __builtin_amdgcn_ballot_w64(!sg2_poly_ok(SG2_PROD_LINEAR_FACTOR * kpoly_g, SG2_PROD_LINEAR_FACTOR * kpoly_s, g, sh));
        const bool tay = __builtin_amdgcn_ballot_w64(!sg2_taylor_ok(cmax_g, cmax_s, g, sh)) == 0;
        const bool dgiven = tay && notpoly == 0 && (!KEEP || cnt == SCAN_TT);       // (steps beyond the end of the tensor carry zero inputs and qualify)
        unsigned long long large[2] = {0, 0}, nottiny[2] = {0, 0};
        float dxv[DI];           // D * x-branch, kept for phase C: of this lane's timestep, or (dgiven) of its column's 16 timesteps
        if (dgiven) {
            int none;
            if (has_s) project_rows<G, true, true>(g, sh, tid, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, s_C, dxv, none);
            else project_rows<G, false, true>(g, sh, tid, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, s_C, dxv, none);
        } else if (tay) {
            int angle;
            if (has_s) project_rows<G, true, false>(g, sh, tid, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, s_C, dxv, angle);
            else project_rows<G, false, false>(g, sh, tid, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, s_C, dxv, angle);
            // blocks 2 q and 2 q + 1 are in the hands of lanes 16 q .. 16 q + 15, a column each
#pragma unroll
            for (int odd = 0; odd < 2; odd++) {
                const unsigned long long l = __builtin_amdgcn_ballot_w64(!(angle & (odd ? 4 : 1))), n = __builtin_amdgcn_ballot_w64(!(angle & (odd ? 8 : 2)));
#pragma unroll
                for (int q = 0; q < 4; q++)
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const unsigned long long blk = 255ull << (16 * q + 8 * odd);
                        if ((l >> (16 * q + 8 * h)) & 255u) large[h] |= blk;
                        if ((n >> (16 * q + 8 * h)) & 255u) nottiny[h] |= blk;
                    }
            }
        } else {
            int angle[2];
            if (has_s) project_steps<G, 2, true, false, true, false>(g, sh, tu, 0, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, s_C, dxv, angle);
            else project_steps<G, 2, true, false, false, false>(g, sh, tu, 0, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, s_C, dxv, angle);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                large[h] = __builtin_amdgcn_ballot_w64(!(angle[h] & 1));
                nottiny[h] = __builtin_amdgcn_ballot_w64(!(angle[h] & 2));
            }
        }
        __syncthreads();      // one wave: no s_barrier is issued, the LDS writes above are ordered before the reads below

        auto keep_state = [&](int u) {
            float* ht = pl.htile + ((size_t)dir * htile_count(pl.total, pl.P) + htile_index(off, ti, u)) * 2 * LANES;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                ht[tid + 64 * h] = S[h].he;
                ht[LANES + tid + 64 * h] = S[h].ho;
            }
        };

        // ---------------- phase B: the recurrences of this lane's two columns over the tile
        const float* __restrict__ r_Be = s_B + (2 * p) * LDS_STRIDE;
        const float* __restrict__ r_Bo = s_B + (2 * p + 1) * LDS_STRIDE;
        const float* __restrict__ r_Ce = s_C + (2 * p) * LDS_STRIDE;
        const float* __restrict__ r_Co = s_C + (2 * p + 1) * LDS_STRIDE;
        int k0 = 0;
        if (dgiven) {
            // a tile on the products throughout (the usual case): both columns in one instruction stream
            float Be[UB], Bo[UB], Ce[UB], Co[UB], dt[2][UB], xv[2][UB];
            auto fetch = [&](int kb, float (&tBe)[UB], float (&tBo)[UB], float (&tCe)[UB], float (&tCo)[UB], float (&tdt)[2][UB], float (&tux)[2][UB]) {
#pragma unroll
                for (int q = 0; q < UB; q += 4) {
                    const f32x4 c4 = *reinterpret_cast<const f32x4*>(r_Be + kb + q), d4 = *reinterpret_cast<const f32x4*>(r_Bo + kb + q);
                    const f32x4 f4 = *reinterpret_cast<const f32x4*>(r_Ce + kb + q), g4 = *reinterpret_cast<const f32x4*>(r_Co + kb + q);
#pragma unroll
                    for (int e = 0; e < 4; e++) { tBe[q + e] = c4[e]; tBo[q + e] = d4[e]; tCe[q + e] = f4[e]; tCo[q + e] = g4[e]; }
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const f32x4 a4 = *reinterpret_cast<const f32x4*>(s_dt + (jl + 8 * h) * LDS_STRIDE + kb + q);
                        const f32x4 b4 = *reinterpret_cast<const f32x4*>(s_ux + (jl + 8 * h) * LDS_STRIDE + kb + q);
#pragma unroll
                        for (int e = 0; e < 4; e++) { tdt[h][q + e] = a4[e]; tux[h][q + e] = b4[e]; }
                    }
                }
            };
            auto compute = [&](int kb, const float (&tBe)[UB], const float (&tBo)[UB], const float (&tCe)[UB], const float (&tCo)[UB],
                               const float (&tdt)[2][UB], const float (&tux)[2][UB]) {
                float y[2][UB];
                const unsigned long long blk = ((1ull << UB) - 1) << kb;
                if (kb + UB > cnt) block_steps_cols<HP, false, true, true>(S, tdt, tux, tBe, tBo, tCe, tCo, LP, cnt - kb, y);      // the tensor's last block
                else if ((notlin & blk) == 0) block_steps_cols<HP, true, true, false>(S, tdt, tux, tBe, tBo, tCe, tCo, LP, UB, y);
                else block_steps_cols<HP, false, true, false>(S, tdt, tux, tBe, tBo, tCe, tCo, LP, UB, y);
                if ((p & 3) == 0) {      // the first lane of every bank holds the totals of its bank's steps (block_pair_sums)
                    *reinterpret_cast<f32x4*>(&s_y[jl * LDS_STRIDE + kb + 4 * (p >> 2)]) = f32x4{y[0][0], y[0][1], y[0][2], y[0][3]};
                    *reinterpret_cast<f32x4*>(&s_y[(jl + 8) * LDS_STRIDE + kb + 4 * (p >> 2)]) = f32x4{y[1][0], y[1][1], y[1][2], y[1][3]};
                }
            };
#pragma unroll 1
            for (; k0 < cnt; k0 += UB) {
                if (KEEP && k0 % HT_STEP == 0) keep_state(tile0 + k0);
                fetch(k0, Be, Bo, Ce, Co, dt, xv);
                compute(k0, Be, Bo, Ce, Co, dt, xv);
            }
        }
        for (; k0 + UB <= cnt; k0 += UB) {
            if (KEEP && k0 % HT_STEP == 0) keep_state(tile0 + k0);
            float Be[UB], Bo[UB], Ce[UB], Co[UB];
#pragma unroll
            for (int q = 0; q < UB; q += 4) {
                const f32x4 c4 = *reinterpret_cast<const f32x4*>(r_Be + k0 + q), d4 = *reinterpret_cast<const f32x4*>(r_Bo + k0 + q);
                const f32x4 f4 = *reinterpret_cast<const f32x4*>(r_Ce + k0 + q), g4 = *reinterpret_cast<const f32x4*>(r_Co + k0 + q);
#pragma unroll
                for (int e = 0; e < 4; e++) { Be[q + e] = c4[e]; Bo[q + e] = d4[e]; Ce[q + e] = f4[e]; Co[q + e] = g4[e]; }
            }
            const unsigned long long blk = ((1ull << UB) - 1) << k0;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int j = jl + 8 * h;
                float dt[UB], xv[UB], y[UB];
#pragma unroll
                for (int q = 0; q < UB; q += 4) {
                    const f32x4 a4 = *reinterpret_cast<const f32x4*>(s_dt + j * LDS_STRIDE + k0 + q), b4 = *reinterpret_cast<const f32x4*>(s_ux + j * LDS_STRIDE + k0 + q);
#pragma unroll
                    for (int e = 0; e < 4; e++) { dt[q + e] = a4[e]; xv[q + e] = b4[e]; }
                }
                if ((notpoly & blk) == 0)
                    block_steps<HP, OUT, 3, false>(S[h], dt, xv, Be, Bo, Ce, Co, 0.0f, 0.0f, 0.0f, LP[h], y);
                else if ((nottiny[h] & blk) == 0)
                    block_steps<HP, OUT, 2, false>(S[h], dt, xv, Be, Bo, Ce, Co, pole_e(h), pole_o(h), rope_f(h), LP[h], y);
                else if ((large[h] & blk) == 0)
                    block_steps<HP, OUT, 1, false>(S[h], dt, xv, Be, Bo, Ce, Co, pole_e(h), pole_o(h), rope_f(h), LP[h], y);
                else
                    block_steps<HP, OUT, 0, false>(S[h], dt, xv, Be, Bo, Ce, Co, pole_e(h), pole_o(h), rope_f(h), LP[h], y);
                if ((p & 3) == 0)        // the first lane of every bank holds the totals of its bank's steps (block_pair_sums)
                    *reinterpret_cast<f32x4*>(&s_y[j * LDS_STRIDE + k0 + 4 * (p >> 2)]) = f32x4{y[0], y[1], y[2], y[3]};
            }
        }
        if (KEEP && k0 % HT_STEP == 0 && k0 < cnt) keep_state(tile0 + k0);      // the ragged end starts right there
        for (; k0 < cnt; k0++) {       // ragged end of the last tile of a tensor
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int j = jl + 8 * h;
                const float dt = s_dt[j * LDS_STRIDE + k0], ux = s_ux[j * LDS_STRIDE + k0];
                float ae, ao, sn, cs;
                sg_abar_pair(dt, pole_e(h), pole_o(h), &ae, &ao);
                sg_sincos(dt * rope_f(h), &sn, &cs);
                step_update<OUT>(S[h], ae, ao, sn, cs, ux * r_Be[k0], ux * r_Bo[k0]);
                const float y = pair_tree_sum<HP>(sg_fma(S[h].ho, r_Co[k0], S[h].he * r_Ce[k0]));
                if (p == 0) s_y[j * LDS_STRIDE + k0] = y;
            }
        }
        __syncthreads();

        // ---------------- phase C: gate, D skip, out_proj, scatter to element order (one 32-byte row per lane)
        {
            float o[DI];
            if (tay) {           // the row owners gate their 16 outputs in place, then every timestep collects its 16 columns
                if (has_s) gate_rows<G, true>(tid, s_coef, s_tay, s_B, s_C, s_y, dxv);
                else gate_rows<G, false>(tid, s_coef, s_tay, s_B, s_C, s_y, dxv);
                __syncthreads();
#pragma unroll
                for (int jj = 0; jj < DI; jj++) o[jj] = s_y[jj * LDS_STRIDE + tu];
            } else {
                if (has_s) gates_of<G, 2, true, false>(g, sh, 0, s_coef, s_tay, o);
                else gates_of<G, 2, false, false>(g, sh, 0, s_coef, s_tay, o);
#pragma unroll
                for (int jj = 0; jj < DI; jj++) o[jj] = sg_fma(s_y[jj * LDS_STRIDE + tu], o[jj], dxv[jj]);
            }
            // out_proj on the matrix pipe: v_mfma_f32_4x4x1_16b is one fused multiply-add per output and step, so 16 of them
            // in the order of the columns are the fmaf chain of the scalar form, bit for bit.  Block b of the instruction
            // is timesteps 4 b .. 4 b + 3: the lane of a timestep supplies its gated output as the B operand and receives
            // its own four outputs; the A operand of lane l is row l % 4 of out_proj (rows 4 .. 7 for the second chain).
            static_assert(DM == 8 && DI % 4 == 0, "two chains of four output rows");
            f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = {0.0f, 0.0f, 0.0f, 0.0f};
            const float* wlo = s_wout + (tid & 3) * DI;
            const float* whi = s_wout + (4 + (tid & 3)) * DI;
#pragma unroll
            for (int m = 0; m < DI; m += 4) {
                const f32x4 wa = *reinterpret_cast<const f32x4*>(wlo + m), wb = *reinterpret_cast<const f32x4*>(whi + m);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    lo = __builtin_amdgcn_mfma_f32_4x4x1f32(wa[e], o[m + e], lo, 0, 0, 0);
                    hi = __builtin_amdgcn_mfma_f32_4x4x1f32(wb[e], o[m + e], hi, 0, 0, 0);
                }
            }
            const float cx[DM] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            const int at = KEEP && in_order ? (dir ? N - 1 - (tile0 + tu) : tile0 + tu) : orig;
            held_dst = valid ? reinterpret_cast<float4*>(pl.ctx + ((size_t)dir * pl.total + off + at) * DM) : nullptr;
            held[0] = make_float4(cx[0], cx[1], cx[2], cx[3]);
            held[1] = make_float4(cx[4], cx[5], cx[6], cx[7]);
            if constexpr (KEEP) {
                if (pl.scan_out[dir] != nullptr && valid) {        // the gated scan output itself (before out_proj), in scan order
                    float4* so = reinterpret_cast<float4*>(pl.scan_out[dir] + ((size_t)off + tile0 + tu) * DI);
#pragma unroll
                    for (int m = 0; m < DI; m += 4) so[m / 4] = make_float4(o[m], o[m + 1], o[m + 2], o[m + 3]);
                }
            }
        }
        __syncthreads();
    }
    flush();
    if (u1 == N && !(KEEP && pl.whole_pass)) {   // last chunk in scan order: new carried state of the tensor
        float* st = dir ? T.mbwd : T.mfwd;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int j = jl + 8 * h;
            if (j < pl.st_di && 2 * p < pl.st_ds) {
                st[j * pl.st_ds + 2 * p] = S[h].he;
                st[j * pl.st_ds + 2 * p + 1] = S[h].ho;
            }
        }
    }
}

// Which chunk a workgroup of a scan launch owns (per_dir chunks of each direction, found through `prefix`).
struct ChunkOf {
    int dir, cidx, ti, c, N, off, u0, u1;
    bool has_s;
};
__device__ __forceinline__ ChunkOf chunk_of(const Plan& pl, const int* chunk_prefix, int per_dir) {
    ChunkOf k;
    k.dir = (int)blockIdx.x >= per_dir ? 1 : 0;
    k.cidx = (int)blockIdx.x - k.dir * per_dir;
    const sg::cint_p prefix = sg::as_const(chunk_prefix);
    const sg::Seg seg = sg::find_seg(prefix, pl.P, k.cidx);
    k.ti = seg.i;
    k.c = k.cidx - seg.first;
    k.N = pl.tensors[k.ti].numel;
    k.off = pl.tensors[k.ti].off;
    k.u0 = k.c * pl.chunk_len;
    k.u1 = min(k.u0 + pl.chunk_len, k.N);
    k.has_s = __builtin_amdgcn_readfirstlane(pl.sharp_nonzero[k.ti]) != 0;
    return k;
}

// The projections of a tile that runs on the products throughout, formed by lanes that own rows: lane (row r, part q) of
// wave w forms column CPW w + r (dt - dt0, dt * x-branch, D * x-branch) and row CPW w + r of B (and C) for timesteps SPL q ..
// SPL q + SPL - 1.  s_in: the tile's 64 g and 64 s, the wave's own copy.  Values and reasons as in project_rows.
// DELTA false: as there (0.42 M elements 247.5 -> 242 us a step, 3.1 M bf16 932 -> 919, 30 000 102 -> 100); large / nottiny[h] receive the blocks of 8 timesteps in which an angle of columns c0 + CPH h ..
// c0 + CPH h + CPH - 1 is too large for sg_sincos_small / sg_sincos_tiny.
template <class G, int CL, bool OUT, bool HAS_S, bool DELTA>
__device__ __forceinline__ void project_own_rows(const float* s_in, int lane, int c0, const float* s_coef, const float* s_tay, const float* s_fmax,
                                                 float* s_dt, float* s_ux, float* s_B, float* s_C, float (&dxk)[Split<G, CL>::SPL],
                                                 unsigned long long (&large)[CL], unsigned long long (&nottiny)[CL]) {
    constexpr int DI = G::DI, CPW = Split<G, CL>::CPW, SPL = Split<G, CL>::SPL;
    auto delta = [&](const f32x4 t, float gg, float ss) { return HAS_S ? sg_fma(t[0], gg, t[1] * ss) : t[0] * gg; };
    auto poly = [&](const f32x4 t, float d) { return sg_fma(sg_fma(sg_fma(t[3], d, t[2]), d, t[1]), d, t[0]); };
    auto eval = [&](const f32x4 t, float gg, float ss) { return sg_fma(t[0], gg, HAS_S ? sg_fma(t[1], ss, t[2]) : t[2]); };
    const int row = c0 + lane % CPW, t0 = SPL * (lane / CPW);
    auto coef = [&](int group) { return *reinterpret_cast<const f32x4*>(s_coef + (group * DI + row) * 4); };
    const f32x4 cd = coef(SG2_COMP_DT), cx = coef(SG2_COMP_XB), cb = coef(SG2_COMP_B), cc = OUT ? coef(SG2_COMP_C) : cb;
    const f32x4 tp = *reinterpret_cast<const f32x4*>(s_tay + row * 4);
    float* const r_dt = s_dt + row * LDS_STRIDE + t0;
    float* const r_ux = s_ux + row * LDS_STRIDE + t0;
    float* const r_B = s_B + bc_slot<G>(row) * LDS_STRIDE + t0;
    float* const r_C = OUT ? s_C + bc_slot<G>(row) * LDS_STRIDE + t0 : nullptr;
    constexpr int NB = SPL > UB ? SPL / UB : 1;              // blocks that a lane has timesteps of
    static_assert(UB == 8 && (SPL == 4 || SPL % 8 == 0), "a lane has half a block or whole ones");
    const float fmax = DELTA ? 0.0f : s_fmax[row];
    bool is_large[NB] = {}, not_tiny[NB] = {};
#pragma unroll
    for (int i = 0; i < SPL / 4; i++) {
        const f32x4 g4 = *reinterpret_cast<const f32x4*>(s_in + t0 + 4 * i);
        const f32x4 s4 = HAS_S ? *reinterpret_cast<const f32x4*>(s_in + SCAN_TT + t0 + 4 * i) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        f32x4 d4, u4, b4, k4;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float dtv = poly(tp, delta(cd, g4[e], s4[e]));
            const float xbv = eval(cx, g4[e], s4[e]);
            d4[e] = DELTA ? dtv - tp[0] : dtv;
            if (!DELTA) {
                is_large[i * 4 / UB] = is_large[i * 4 / UB] || !(dtv * fmax < SG_SINCOS_SMALL_LIMIT);
                not_tiny[i * 4 / UB] = not_tiny[i * 4 / UB] || !(dtv * fmax < SG_SINCOS_TINY_LIMIT);
            }
            u4[e] = dtv * xbv;
            if (OUT) dxk[4 * i + e] = cx[3] * xbv;
            b4[e] = eval(cb, g4[e], s4[e]);
            if (OUT) k4[e] = eval(cc, g4[e], s4[e]);
        }
        *reinterpret_cast<f32x4*>(r_dt + 4 * i) = d4;
        *reinterpret_cast<f32x4*>(r_ux + 4 * i) = u4;
        *reinterpret_cast<f32x4*>(r_B + 4 * i) = b4;
        if (OUT) *reinterpret_cast<f32x4*>(r_C + 4 * i) = k4;
    }
    if (!DELTA) {
        constexpr int CPH = Split<G, CL>::CPH;
#pragma unroll
        for (int k = 0; k < NB; k++) {
            const unsigned long long l = __builtin_amdgcn_ballot_w64(is_large[k]), n = __builtin_amdgcn_ballot_w64(not_tiny[k]);
#pragma unroll
            for (int q = 0; q < 64 / CPW; q++)
#pragma unroll
                for (int h = 0; h < CL; h++) {
                    const int at = CPW * q + CPH * h;
                    const unsigned long long blk = 255ull << (SPL * q / UB * UB + UB * k);
                    if ((l >> at) & ((1u << CPH) - 1)) large[h] |= blk;
                    if ((n >> at) & ((1u << CPH) - 1)) nottiny[h] |= blk;
                }
        }
    }
}

// The tables a workgroup of the scan reads from LDS: composed triples (D beside the x-branch's), Taylor polynomials, the
// largest |rope frequency| of each column.
template <class G>
__device__ __forceinline__ void stage_tables(const Plan& pl, int dir, int tid, int threads, float* s_coef, float* s_tay, float* s_fmax) {
    constexpr int DI = G::DI, HP = G::HP;
    const float* comp = pl.comp + dir * (SG2_COMP_GROUPS * G::ROWS * 3);
    const float* tay = pl.comp + 2 * SG2_COMP_GROUPS * G::ROWS * 3 + dir * 2 * G::ROWS * 4;
    const float* Dw = pl.W.w[dir ? W_B_D : W_F_D];
    const float* rope = pl.W.w[dir ? W_B_ROPE : W_F_ROPE];
    for (int i = tid; i < SG2_COMP_GROUPS * DI; i += threads) {
        const float* t = comp + i * 3;
        *reinterpret_cast<f32x4*>(s_coef + i * 4) = f32x4{t[0], t[1], t[2], i / DI == SG2_COMP_XB ? Dw[i % DI] : 0.0f};
    }
    for (int i = tid; i < 2 * DI * 4; i += threads) s_tay[i] = tay[i];
    if (tid < DI) {
        float m = 0.0f;
#pragma unroll
        for (int p = 0; p < HP; p++) m = sg_max(m, sg_abs(rope[tid * HP + p]));
        s_fmax[tid] = m;
    }
}

// What block_pair_sums leaves in the first lane of every bank: the totals of its bank's steps.
template <int HP>
__device__ __forceinline__ void store_sums(float* row, int p, const float (&y)[UB]) {
    if constexpr (HP == 8) *reinterpret_cast<f32x4*>(row + 4 * (p >> 2)) = f32x4{y[0], y[1], y[2], y[3]};
    else *reinterpret_cast<float2*>(row + 2 * (p >> 2)) = make_float2(y[0], y[1]);
}

// ---- chunk summaries
// Bound by the vector ALU like the replay, and laid out like it: a lane owns one pair of two columns, a wave CPW columns and
// as many rows of B, which feed both columns of a lane.  The first attempt walks the states alone on the products of
// the output pass: ten instructions per step, column and pair on their linear parts, 14 on the quadratics, where the separate
// A_bar, sin, cos and the bound on the 2x2 part took 22.  The bound needs nothing per step there: while a tile
// qualifies, |dt - dt0| is below pl.comp's limit, so a pair's part shrinks at least by sg2_abar_bound in every step.
// (The bilevel pass keeps the separate factors: a fresh net's sums nearly cancel, and an optimizer that divides by their size
// turns other last bits of its contexts into other thresholds of the next pass.)
// 39 us on 0.42 M elements, 100 us on 3.1 M, 89 us on 25 M whose tiles qualify, 79 us on 0.42 M with the large geometry; with one
// column per lane of 128 or 512 and the separate factors throughout 46, 113, 141 and 255 us.
template <class G, int CL>
__global__ __launch_bounds__((64 * Split<G, CL>::WAVES)) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_summary(Plan pl) {
    constexpr int DS = G::DS, DI = G::DI, HP = G::HP, LANES = G::THREADS, WAVES = Split<G, CL>::WAVES, CPW = Split<G, CL>::CPW, CPH = Split<G, CL>::CPH;
    __shared__ __attribute__((aligned(16))) float s_dt[DI * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) float s_ux[DI * LDS_STRIDE];       // dt * x-branch
    __shared__ __attribute__((aligned(16))) float s_B[DS * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) float s_in_all[WAVES * 2 * SCAN_TT];
    __shared__ __attribute__((aligned(16))) float s_coef[SG2_COMP_GROUPS * DI * 4];
    __shared__ __attribute__((aligned(16))) float s_tay[2 * DI * 4];
    __shared__ float s_fmax[DI];

    const ChunkOf K = chunk_of(pl, pl.wchunk_prefix, pl.wchunks);
    const int dir = K.dir, N = K.N, u0 = K.u0, u1 = K.u1;
    const bool has_s = K.has_s;
    const uint32_t* __restrict__ skey = pl.keys[0] + K.off;      // sorted |g| bits
    const int32_t* __restrict__ sval = pl.vals[0] + K.off;       // element index | sign of g
    const float* __restrict__ ssrt = pl.ssorted + K.off;          // sharpness in sorted order

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = CPW * wave, jl = lane / HP, p = lane % HP;       // scan role: pair p of columns c0 + jl and c0 + CPH + jl
    const int tu = lane;                                            // projection role: timestep of the tile
    float* const s_in = s_in_all + wave * 2 * SCAN_TT;
    const float* alog = pl.W.w[dir ? W_B_ALOG : W_F_ALOG];
    const float* rope = pl.W.w[dir ? W_B_ROPE : W_F_ROPE];
    const float* tay = pl.comp + 2 * SG2_COMP_GROUPS * G::ROWS * 3 + dir * 2 * G::ROWS * 4;
    auto col = [&](int h) { return c0 + jl + CPH * h; };
    // -A/2 with A = -exp(A_log): the two poles of a pair, and its frequency (see k_replay)
    float poles[CL][3];
#pragma unroll
    for (int h = 0; h < CL; h++) {
        poles[h][0] = -0.5f * -sg_exp(alog[col(h) * DS + 2 * p]);
        poles[h][1] = -0.5f * -sg_exp(alog[col(h) * DS + 2 * p + 1]);
        poles[h][2] = rope[col(h) * HP + p];
        asm("" : "+v"(poles[h][0]), "+v"(poles[h][1]), "+v"(poles[h][2]));       // (keeps the compiler from forming them where they are used)
    }
    auto pole_e = [&](int h) { return poles[h][0]; };
    auto pole_o = [&](int h) { return poles[h][1]; };
    auto rope_f = [&](int h) { return poles[h][2]; };
    const sg::cfloat_p lim = sg::as_const(pl.comp) + 2 * SG2_COMP_GROUPS * G::ROWS * 3 + 2 * 2 * G::ROWS * 4;
    const float cmax_g = lim[2 * dir], cmax_s = lim[2 * dir + 1];              // what decides whether a tile may use the Taylor polynomials
    const float kpoly_g = lim[4 + 2 * dir], kpoly_s = lim[5 + 2 * dir];        // ... a block the lane polynomials (sg2_poly_ok)
    const float kprod_g = lim[8 + 2 * dir], kprod_s = lim[9 + 2 * dir];        // ... a tile of the first attempt the products
    LanePoly<true> LP[CL];
    float shrink[CL];            // what eight steps on the products multiply a pair's 2x2 part by at most
#pragma unroll
    for (int h = 0; h < CL; h++) {
        LP[h].dt0 = tay[col(h) * 4];
        const float ae = pole_e(h), ao = pole_o(h);
        sg2_pair_products(LP[h].dt0, ae, ao, rope_f(h), LP[h].k);
        shrink[h] = sg2_shrink8(LP[h].dt0, ae, ao, lim[16 + dir]);
    }
    stage_tables<G>(pl, dir, tid, 64 * WAVES, s_coef, s_tay, s_fmax);
    __syncthreads();

    const LaneState identity = {0.0f, 0.0f, 1.0f, 0.0f, 0.0f, 1.0f};
    LaneState S[CL], late[CL];
#pragma unroll
    for (int h = 0; h < CL; h++) S[h] = late[h] = identity;
    bool fully_contracted = false;      // the walk stopped because the 2x2 part had contracted
    bool have_late = false;
    // The chunk is walked backwards in blocks of `window` steps.  Each block is summarised from the identity and the
    // summary of everything after it (`late`) is applied on top; as soon as the 2x2 part of the running summary has
    // contracted below 2^-64 the steps before the block cannot matter and the walk stops.
    int blk_end = u1;
    int blk_first = u0;
    if (pl.window > 0 && pl.window < pl.chunk_len) blk_first = max(u0, u1 - pl.window);
    // First attempt: ONE block of as many steps as compose_block expects the slowest pair to need, walked with the state
    // part only (LITE) and a bound on the 2x2 part in its place.  If the bound is below 2^-64 in every lane the summary
    // is (0, b) as below; if not, the walk starts over in its general form.
    bool lite = false;
    if (blk_first > u0) {
        const int first_block = __builtin_amdgcn_readfirstlane(pl.contracted[1]);
        if (first_block > 0 && u1 - first_block > u0) {
            lite = true;
            blk_first = u1 - first_block;
        }
    }
    // inputs of one tile (sorted |g| bits, payload, sorted sharpness) for this lane's timestep; zero beyond the block
    uint32_t nx_key = 0;
    int32_t nx_val = 0;
    float nx_sh = 0.0f;
    auto load_inputs = [&](int tile0) {
        const int u = tile0 + tu;
        if (u < blk_end) {
            const int t = dir ? (N - 1 - u) : u;
            nx_key = skey[t];
            nx_val = sval[t];
            nx_sh = has_s ? ssrt[t] : 0.0f;      // an all-zero tensor has no sorted copy of its sharpness (uniform branch)
        }
    };
    const float* const r_Be = s_B + p * LDS_STRIDE;
    const float* const r_Bo = s_B + (HP + p) * LDS_STRIDE;
    auto fetch4 = [&](const float* r, float (&out)[UB], int k0) {
#pragma unroll
        for (int q = 0; q < UB; q += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(r + k0 + q);
#pragma unroll
            for (int e = 0; e < 4; e++) out[q + e] = v[e];
        }
    };
    // the steps from blk_first to blk_end
    auto walk = [&](auto lite_c) {
        constexpr bool LITE = decltype(lite_c)::value;
        load_inputs(blk_first);
        for (int tile0 = blk_first; tile0 < blk_end; tile0 += SCAN_TT) {
            const int cnt = min(SCAN_TT, blk_end - tile0);
            const bool valid = tile0 + tu < blk_end;
            // this tile's inputs were requested one tile ago (or just before the loop); request the next tile's now
            const float g = valid ? sg_i2f((int32_t)nx_key | (nx_val & (int32_t)0x80000000)) : 0.0f;
            const float sh = valid ? nx_sh : 0.0f;
            if (tile0 + SCAN_TT < blk_end) load_inputs(tile0 + SCAN_TT);
            // the same 64 timesteps in every wave of the workgroup: the same decisions without talking to one another
            const bool ty = __builtin_amdgcn_ballot_w64(!sg2_taylor_ok(cmax_g, cmax_s, g, sh)) == 0;
            const bool fast = LITE && pl.htile == nullptr && ty && cnt % UB == 0 && __builtin_amdgcn_ballot_w64(!sg2_poly_ok(kprod_g, kprod_s, g, sh)) == 0;
            unsigned long long notpoly = 0, large[CL] = {}, nottiny[CL] = {};
            float unused[CPW];
            if (!fast) notpoly = __builtin_amdgcn_ballot_w64(!sg2_poly_ok(kpoly_g, kpoly_s, g, sh));
            if (ty) {
                s_in[tu] = g;
                if (has_s) s_in[SCAN_TT + tu] = sh;
                __builtin_amdgcn_wave_barrier();      // one wave's LDS accesses execute in program order
                auto run = [&](auto has_s_c, auto delta_c) {
                    project_own_rows<G, CL, false, decltype(has_s_c)::value, decltype(delta_c)::value>(s_in, lane, c0, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B,
                                                                                                       nullptr, unused, large, nottiny);
                };
                if (fast) { if (has_s) run(std::true_type{}, std::true_type{}); else run(std::false_type{}, std::true_type{}); }
                else { if (has_s) run(std::true_type{}, std::false_type{}); else run(std::false_type{}, std::false_type{}); }
            } else {
                int angle[CL];
                if (has_s) project_steps<G, CL, false, true, true, false>(g, sh, tu, c0, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, nullptr, unused, angle);
                else project_steps<G, CL, false, true, false, false>(g, sh, tu, c0, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, nullptr, unused, angle);
#pragma unroll
                for (int h = 0; h < CL; h++) {
                    large[h] = __builtin_amdgcn_ballot_w64(!(angle[h] & 1));
                    nottiny[h] = __builtin_amdgcn_ballot_w64(!(angle[h] & 2));
                }
            }
            __syncthreads();
            if (fast) {
                const unsigned long long notlin =
                    __builtin_amdgcn_ballot_w64(!sg2_poly_ok(SG2_PROD_LINEAR_FACTOR * kprod_g, SG2_PROD_LINEAR_FACTOR * kprod_s, g, sh));
#pragma unroll 1
                for (int k0 = 0; k0 < cnt; k0 += UB) {
                    float dt[CL][UB], ux[CL][UB], Be[UB], Bo[UB], y[CL][UB];
                    fetch4(r_Be, Be, k0);
                    fetch4(r_Bo, Bo, k0);
#pragma unroll
                    for (int h = 0; h < CL; h++) {
                        fetch4(s_dt + col(h) * LDS_STRIDE, dt[h], k0);
                        fetch4(s_ux + col(h) * LDS_STRIDE, ux[h], k0);
                    }
                    const unsigned long long blk = ((1ull << UB) - 1) << k0;
                    if ((notlin & blk) == 0) block_steps_cols<HP, true, false, false>(S, dt, ux, Be, Bo, Be, Bo, LP, UB, y);
                    else block_steps_cols<HP, false, false, false>(S, dt, ux, Be, Bo, Be, Bo, LP, UB, y);
#pragma unroll
                    for (int h = 0; h < CL; h++) S[h].c0e = S[h].c0e * shrink[h];
                }
            } else {
                // exceptional: one column after the other, the forms of its blocks chosen one by one
#pragma unroll
                for (int h = 0; h < CL; h++) {
                    LanePoly<false> GP;
                    const float ae0 = pole_e(h), ao0 = pole_o(h), f0 = rope_f(h);
                    GP.dt0 = tay[col(h) * 4];
                    sg2_abar_poly(GP.dt0, ae0, GP.pe);
                    sg2_abar_poly(GP.dt0, ao0, GP.po);
                    sg2_sincos_poly(GP.dt0, f0, GP.qs, GP.qc);
                    LaneState T = S[h];
                    const unsigned long long lg = large[h], nt = nottiny[h];
                    const float* r_dt = s_dt + col(h) * LDS_STRIDE;
                    const float* r_ux = s_ux + col(h) * LDS_STRIDE;
                    int k0 = 0;
                    for (; k0 + UB <= cnt; k0 += UB) {
                        float dt[UB], ux[UB], Be[UB], Bo[UB], y[UB];
                        fetch4(r_Be, Be, k0);
                        fetch4(r_Bo, Bo, k0);
                        fetch4(r_dt, dt, k0);
                        fetch4(r_ux, ux, k0);
                        const unsigned long long blk = ((1ull << UB) - 1) << k0;
                        if ((notpoly & blk) == 0) block_steps<HP, false, 3, LITE>(T, dt, ux, Be, Bo, Be, Bo, 0.0f, 0.0f, 0.0f, GP, y);
                        else if ((nt & blk) == 0) block_steps<HP, false, 2, LITE>(T, dt, ux, Be, Bo, Be, Bo, ae0, ao0, f0, GP, y);
                        else if ((lg & blk) == 0) block_steps<HP, false, 1, LITE>(T, dt, ux, Be, Bo, Be, Bo, ae0, ao0, f0, GP, y);
                        else block_steps<HP, false, 0, LITE>(T, dt, ux, Be, Bo, Be, Bo, ae0, ao0, f0, GP, y);
                    }
                    for (; k0 < cnt; k0++) {
                        float ae, ao, sn, cs;
                        sg_abar_pair(r_dt[k0], ae0, ao0, &ae, &ao);
                        sg_sincos(r_dt[k0] * f0, &sn, &cs);
                        step_update<false, LITE>(T, ae, ao, sn, cs, r_ux[k0] * r_Be[k0], r_ux[k0] * r_Bo[k0]);
                    }
                    S[h] = T;
                }
            }
            __syncthreads();
        }
    };
    if (lite) {
        walk(std::true_type{});      // c0e holds the bound (a NaN counts as "not contracted")
        bool open = false;
#pragma unroll
        for (int h = 0; h < CL; h++) open = open || !(S[h].c0e < SG2_FORGOTTEN);
        fully_contracted = !__syncthreads_or(open);
        if (!fully_contracted) {     // the general walk, from the end of the chunk
            blk_first = max(u0, u1 - pl.window);
#pragma unroll
            for (int h = 0; h < CL; h++) S[h] = identity;
        }
    }
    while (!fully_contracted) {
        walk(std::false_type{});
        bool open = false;
#pragma unroll
        for (int h = 0; h < CL; h++) {
            if (have_late) {     // S covers [blk_first, blk_end), late covers [blk_end, u1): the summary of both is late o S
                const LaneState E = S[h], &L = late[h];
                S[h].c0e = sg_fma(L.c0e, E.c0e, L.c1e * E.c0o);
                S[h].c0o = sg_fma(L.c0o, E.c0e, L.c1o * E.c0o);
                S[h].c1e = sg_fma(L.c0e, E.c1e, L.c1e * E.c1o);
                S[h].c1o = sg_fma(L.c0o, E.c1e, L.c1o * E.c1o);
                S[h].he = sg_fma(L.c0e, E.he, sg_fma(L.c1e, E.ho, L.he));
                S[h].ho = sg_fma(L.c0o, E.he, sg_fma(L.c1o, E.ho, L.ho));
            }
            // has the running summary contracted?  (a NaN counts as "no")
            const float mx = sg_max(sg_max(sg_abs(S[h].c0e), sg_abs(S[h].c0o)), sg_max(sg_abs(S[h].c1e), sg_abs(S[h].c1o)));
            open = open || !(mx < SG2_FORGOTTEN);
        }
        if (blk_first == u0) break;       // the whole chunk is covered
        fully_contracted = !__syncthreads_or(open);
        if (fully_contracted) break;
#pragma unroll
        for (int h = 0; h < CL; h++) {
            late[h] = S[h];
            S[h] = identity;
        }
        have_late = true;
        blk_end = blk_first;
        blk_first = max(u0, blk_first - pl.window);
    }
    if (fully_contracted) {
#pragma unroll
        for (int h = 0; h < CL; h++) S[h].c0e = S[h].c0o = S[h].c1e = S[h].c1o = 0.0f;
    }
    float* sm = pl.summaries + (size_t)(dir * pl.wchunks + K.cidx) * 6 * LANES;
#pragma unroll
    for (int h = 0; h < CL; h++) {
        const int at = 64 * (CL * wave + h) + lane;       // (column, pair) in the order of the columns
        sm[0 * LANES + at] = S[h].c0e;   // M = [c0e c1e; c0o c1o]
        sm[1 * LANES + at] = S[h].c0o;
        sm[2 * LANES + at] = S[h].c1e;
        sm[3 * LANES + at] = S[h].c1o;
        sm[4 * LANES + at] = S[h].he;
        sm[5 * LANES + at] = S[h].ho;
    }
    if (!fully_contracted && tid == 0) *pl.contracted = 0;      // plain store: every writer stores the same value
}

// ---- the replay with several waves per chunk: the large geometry (four, two columns per lane) and small calls (one column
// per lane: two for the default geometry, eight for the large one)
// A wave forms its own columns and as many rows of B and C, walks its columns and gates them; what the waves share is
// B and C, and the outputs that out_proj sums over all columns.  So a tile has two barriers (B and C stand; the gated
// outputs stand), the rows s_dt / s_y alternate between two buffers, and two workgroups of the large geometry (103 KB of LDS,
// 246 registers a lane) share a compute unit to work across them.  Each B / C entry a lane fetches feeds CL recurrences, and
// a context leaves as contiguous bytes: a wave multiplies 64 / WAVES timesteps by all of out_proj (4x4x1
// matrix instructions, block (timestep quad, four rows): the fmaf chain over the columns, bit for bit).
// Large geometry, 0.42 M elements: 300 us; as one 512-lane workgroup per compute unit with a column per lane, a barrier
// after every phase and 8-byte pieces of the contexts 409 us.
template <class G, int CL>
__global__ __launch_bounds__((64 * Split<G, CL>::WAVES)) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_replay_cols(Plan pl) {
    constexpr int DM = G::DM, DS = G::DS, DI = G::DI, HP = G::HP, LANES = G::THREADS, WAVES = Split<G, CL>::WAVES, CPW = Split<G, CL>::CPW, CPH = Split<G, CL>::CPH;
    constexpr int SPL = Split<G, CL>::SPL, WSTRIDE = DI + 4;        // out_proj rows: 16 lanes read 16 rows at once
    static_assert((SCAN_TT / WAVES) % 4 == 0 && 4 * (SCAN_TT / WAVES) * (DM / 4) <= 4 * 64, "out_proj roles");
    __shared__ __attribute__((aligned(16))) float s_dty[2][DI * LDS_STRIDE];    // dt (dt - dt0) of a column, then its y, then its gated output
    __shared__ __attribute__((aligned(16))) float s_ux[DI * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) float s_B[DS * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) float s_C[DS * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) float s_in_all[WAVES * 2 * SCAN_TT];
    __shared__ __attribute__((aligned(16))) float s_coef[SG2_COMP_GROUPS * DI * 4];
    __shared__ __attribute__((aligned(16))) float s_tay[2 * DI * 4];
    __shared__ __attribute__((aligned(16))) float s_wout[DM * WSTRIDE];
    __shared__ float s_fmax[DI];

    const ChunkOf K = chunk_of(pl, pl.chunk_prefix, pl.chunks);
    const int dir = K.dir, N = K.N, off = K.off, u0 = K.u0, u1 = K.u1, c = K.c;
    const bool has_s = K.has_s;
    const TensorDev& T = pl.tensors[K.ti];
    const uint32_t* __restrict__ skey = pl.keys[0] + off;
    const int32_t* __restrict__ sval = pl.vals[0] + off;
    const float* __restrict__ ssrt = pl.ssorted + off;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = CPW * wave, jl = lane / HP, p = lane % HP;
    const int tu = lane;
    float* const s_in = s_in_all + wave * 2 * SCAN_TT;
    const float* alog = pl.W.w[dir ? W_B_ALOG : W_F_ALOG];
    const float* rope = pl.W.w[dir ? W_B_ROPE : W_F_ROPE];
    auto col = [&](int h) { return c0 + jl + CPH * h; };
    float poles[CL][3];
#pragma unroll
    for (int h = 0; h < CL; h++) {
        poles[h][0] = -0.5f * -sg_exp(alog[col(h) * DS + 2 * p]);
        poles[h][1] = -0.5f * -sg_exp(alog[col(h) * DS + 2 * p + 1]);
        poles[h][2] = rope[col(h) * HP + p];
        asm("" : "+v"(poles[h][0]), "+v"(poles[h][1]), "+v"(poles[h][2]));       // (keeps the compiler from forming them where they are used)
    }
    auto pole_e = [&](int h) { return poles[h][0]; };
    auto pole_o = [&](int h) { return poles[h][1]; };
    auto rope_f = [&](int h) { return poles[h][2]; };
    LanePoly<true> LP[CL];
#pragma unroll
    for (int h = 0; h < CL; h++) {
        LP[h].dt0 = pl.comp[2 * SG2_COMP_GROUPS * G::ROWS * 3 + dir * 2 * G::ROWS * 4 + col(h) * 4];
        sg2_pair_products(LP[h].dt0, pole_e(h), pole_o(h), rope_f(h), LP[h].k);
    }
    stage_tables<G>(pl, dir, tid, 64 * WAVES, s_coef, s_tay, s_fmax);
    for (int i = tid; i < DM * DI; i += 64 * WAVES) s_wout[i / DI * WSTRIDE + i % DI] = pl.W.w[dir ? W_B_OUT : W_F_OUT][i];
    __syncthreads();
    const sg::cfloat_p lim = sg::as_const(pl.comp) + 2 * SG2_COMP_GROUPS * G::ROWS * 3 + 2 * 2 * G::ROWS * 4;
    const float cmax_g = lim[2 * dir], cmax_s = lim[2 * dir + 1];
    const float kpoly_g = lim[8 + 2 * dir], kpoly_s = lim[8 + 2 * dir + 1];

    LaneState S[CL];
#pragma unroll
    for (int h = 0; h < CL; h++) {
        S[h] = {0.0f, 0.0f, 1.0f, 0.0f, 0.0f, 1.0f};
        const int at = 64 * (CL * wave + h) + lane;
        if (c > 0 && __builtin_amdgcn_readfirstlane(*pl.contracted) != 0) {
            const float* sm = pl.summaries + (size_t)(dir * pl.wchunks + pl.wchunk_prefix[K.ti] + c - 1) * 6 * LANES;
            S[h].he = sm[4 * LANES + at];
            S[h].ho = sm[5 * LANES + at];
        } else if (T.nchunks == 1) {       // nothing before it: the carried state itself (no other workgroup writes it)
            const float* st = dir ? T.mbwd : T.mfwd;
            if (col(h) < pl.st_di && 2 * p < pl.st_ds) {
                S[h].he = st[col(h) * pl.st_ds + 2 * p];
                S[h].ho = st[col(h) * pl.st_ds + 2 * p + 1];
            }
        } else {
            const float* hs = pl.hstart + ((size_t)(dir * pl.chunks + K.cidx) * 2) * LANES;
            S[h].he = hs[at];
            S[h].ho = hs[LANES + at];
        }
    }
    uint32_t nx_key = 0;
    int32_t nx_val = 0;
    float nx_sh = 0.0f;
    auto load_inputs = [&](int tile0) {
        const int u = tile0 + tu;
        if (u < u1) {
            const int t = dir ? (N - 1 - u) : u;
            nx_key = skey[t];
            nx_val = sval[t];
            nx_sh = has_s ? ssrt[t] : 0.0f;
        }
    };
    load_inputs(u0);
    // a context leaves one tile late, after the next tile's inputs have arrived (see k_replay)
    f32x4 held = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4* held_dst = nullptr;
    const float* const r_Be = s_B + p * LDS_STRIDE;
    const float* const r_Bo = s_B + (HP + p) * LDS_STRIDE;
    const float* const r_Ce = s_C + p * LDS_STRIDE;
    const float* const r_Co = s_C + (HP + p) * LDS_STRIDE;
    auto fetch4 = [&](const float* r, float (&out)[UB], int k0) {
#pragma unroll
        for (int q = 0; q < UB; q += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(r + k0 + q);
#pragma unroll
            for (int e = 0; e < 4; e++) out[q + e] = v[e];
        }
    };
    int buffer = 0;
    for (int tile0 = u0; tile0 < u1; tile0 += SCAN_TT, buffer ^= 1) {
        float* const s_dt = s_dty[buffer];      // read by other waves until the tile after the next begins: two barriers lie between
        const int cnt = min(SCAN_TT, u1 - tile0);
        const uint32_t kbits = nx_key;
        const int32_t v = nx_val;
        const float shv = nx_sh;
        const bool valid = tile0 + tu < u1;
        asm volatile("" : : "v"(kbits), "v"(v), "v"(shv) : "memory");      // the wait for this tile's inputs goes here, before the store
        if (held_dst != nullptr) *held_dst = held;
        if (tile0 + SCAN_TT < u1) load_inputs(tile0 + SCAN_TT);
        int orig = v & 0x7fffffff;
        orig = valid && (unsigned)orig < (unsigned)N ? orig : 0;   // never index outside the tensor
        const float g = valid ? sg_i2f((int32_t)kbits | (v & (int32_t)0x80000000)) : 0.0f;
        const float sh = valid ? shv : 0.0f;
        const unsigned long long notpoly = __builtin_amdgcn_ballot_w64(!sg2_poly_ok(kpoly_g, kpoly_s, g, sh));
        const bool ty = __builtin_amdgcn_ballot_w64(!sg2_taylor_ok(cmax_g, cmax_s, g, sh)) == 0;
        const bool fast = ty && notpoly == 0;
        unsigned long long large[CL] = {}, nottiny[CL] = {};
        float dx[CPW];           // D * x-branch: of this lane's column for its SPL timesteps (ty), or of its timestep for the wave's columns
        if (ty) {
            s_in[tu] = g;
            if (has_s) s_in[SCAN_TT + tu] = sh;
            __builtin_amdgcn_wave_barrier();
            auto run = [&](auto has_s_c, auto delta_c) {
                project_own_rows<G, CL, true, decltype(has_s_c)::value, decltype(delta_c)::value>(s_in, lane, c0, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, s_C, dx, large, nottiny);
            };
            if (fast) { if (has_s) run(std::true_type{}, std::true_type{}); else run(std::false_type{}, std::true_type{}); }
            else { if (has_s) run(std::true_type{}, std::false_type{}); else run(std::false_type{}, std::false_type{}); }
        } else {
            int angle[CL];
            if (has_s) project_steps<G, CL, true, true, true, false>(g, sh, tu, c0, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, s_C, dx, angle);
            else project_steps<G, CL, true, true, false, false>(g, sh, tu, c0, s_coef, s_tay, s_fmax, s_dt, s_ux, s_B, s_C, dx, angle);
#pragma unroll
            for (int h = 0; h < CL; h++) {
                large[h] = __builtin_amdgcn_ballot_w64(!(angle[h] & 1));
                nottiny[h] = __builtin_amdgcn_ballot_w64(!(angle[h] & 2));
            }
        }
        __syncthreads();

        // the recurrences of this lane's two columns; lanes whose p is a multiple of four hold two steps' totals each
        if (fast) {
            const unsigned long long notlin =
                __builtin_amdgcn_ballot_w64(!sg2_poly_ok(SG2_PROD_LINEAR_FACTOR * kpoly_g, SG2_PROD_LINEAR_FACTOR * kpoly_s, g, sh));
#pragma unroll 1
            for (int k0 = 0; k0 < cnt; k0 += UB) {
                float dt[CL][UB], ux[CL][UB], Be[UB], Bo[UB], Ce[UB], Co[UB], y[CL][UB];
                fetch4(r_Be, Be, k0);
                fetch4(r_Bo, Bo, k0);
                fetch4(r_Ce, Ce, k0);
                fetch4(r_Co, Co, k0);
#pragma unroll
                for (int h = 0; h < CL; h++) {
                    fetch4(s_dt + col(h) * LDS_STRIDE, dt[h], k0);
                    fetch4(s_ux + col(h) * LDS_STRIDE, ux[h], k0);
                }
                const unsigned long long blk = ((1ull << UB) - 1) << k0;
                if (k0 + UB > cnt) block_steps_cols<HP, false, true, true>(S, dt, ux, Be, Bo, Ce, Co, LP, cnt - k0, y);
                else if ((notlin & blk) == 0) block_steps_cols<HP, true, true, false>(S, dt, ux, Be, Bo, Ce, Co, LP, UB, y);
                else block_steps_cols<HP, false, true, false>(S, dt, ux, Be, Bo, Ce, Co, LP, UB, y);
                if ((p & 3) == 0) {
#pragma unroll
                    for (int h = 0; h < CL; h++) store_sums<HP>(s_dt + col(h) * LDS_STRIDE + k0, p, y[h]);
                }
            }
        } else {
            int k0 = 0;
            for (; k0 + UB <= cnt; k0 += UB) {
                float Be[UB], Bo[UB], Ce[UB], Co[UB];
                fetch4(r_Be, Be, k0);
                fetch4(r_Bo, Bo, k0);
                fetch4(r_Ce, Ce, k0);
                fetch4(r_Co, Co, k0);
                const unsigned long long blk = ((1ull << UB) - 1) << k0;
#pragma unroll
                for (int h = 0; h < CL; h++) {
                    float dt[UB], ux[UB], y[UB];
                    fetch4(s_dt + col(h) * LDS_STRIDE, dt, k0);
                    fetch4(s_ux + col(h) * LDS_STRIDE, ux, k0);
                    if ((notpoly & blk) == 0)
                        block_steps<HP, true, 3>(S[h], dt, ux, Be, Bo, Ce, Co, 0.0f, 0.0f, 0.0f, LP[h], y);
                    else if ((nottiny[h] & blk) == 0)
                        block_steps<HP, true, 2>(S[h], dt, ux, Be, Bo, Ce, Co, pole_e(h), pole_o(h), rope_f(h), LP[h], y);
                    else if ((large[h] & blk) == 0)
                        block_steps<HP, true, 1>(S[h], dt, ux, Be, Bo, Ce, Co, pole_e(h), pole_o(h), rope_f(h), LP[h], y);
                    else
                        block_steps<HP, true, 0>(S[h], dt, ux, Be, Bo, Ce, Co, pole_e(h), pole_o(h), rope_f(h), LP[h], y);
                    if ((p & 3) == 0) store_sums<HP>(s_dt + col(h) * LDS_STRIDE + k0, p, y);
                }
            }
            for (; k0 < cnt; k0++) {       // ragged end of the last tile of a tensor
#pragma unroll
                for (int h = 0; h < CL; h++) {
                    const float dt = s_dt[col(h) * LDS_STRIDE + k0], ux = s_ux[col(h) * LDS_STRIDE + k0];
                    float ae, ao, sn, cs;
                    sg_abar_pair(dt, pole_e(h), pole_o(h), &ae, &ao);
                    sg_sincos(dt * rope_f(h), &sn, &cs);
                    step_update<true>(S[h], ae, ao, sn, cs, ux * r_Be[k0], ux * r_Bo[k0]);
                    const float y = pair_tree_sum<HP>(sg_fma(S[h].ho, r_Co[k0], S[h].he * r_Ce[k0]));
                    if (p == 0) s_dt[col(h) * LDS_STRIDE + k0] = y;
                }
            }
        }
        __builtin_amdgcn_wave_barrier();        // a wave gates its own columns: its LDS accesses execute in program order

        // gate and D skip, in place
        if (ty) {
            const int row = c0 + lane % CPW, t0 = SPL * (lane / CPW);
            const f32x4 cz = *reinterpret_cast<const f32x4*>(s_coef + (SG2_COMP_Z * DI + row) * 4);
            const f32x4 tz = *reinterpret_cast<const f32x4*>(s_tay + (DI + row) * 4);
            auto gate = [&](auto has_s_c) {
                constexpr bool HS = decltype(has_s_c)::value;
#pragma unroll
                for (int i = 0; i < SPL / 4; i++) {
                    const f32x4 g4 = *reinterpret_cast<const f32x4*>(s_in + t0 + 4 * i);
                    const f32x4 s4 = HS ? *reinterpret_cast<const f32x4*>(s_in + SCAN_TT + t0 + 4 * i) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    f32x4 y4 = *reinterpret_cast<const f32x4*>(s_dt + row * LDS_STRIDE + t0 + 4 * i);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float d = HS ? sg_fma(cz[0], g4[e], cz[1] * s4[e]) : cz[0] * g4[e];
                        y4[e] = sg_fma(y4[e], sg_fma(sg_fma(sg_fma(tz[3], d, tz[2]), d, tz[1]), d, tz[0]), dx[4 * i + e]);
                    }
                    *reinterpret_cast<f32x4*>(s_dt + row * LDS_STRIDE + t0 + 4 * i) = y4;
                }
            };
            if (has_s) gate(std::true_type{});
            else gate(std::false_type{});
        } else {
            float gv[CPW];
            if (has_s) gates_of<G, CL, true, false>(g, sh, c0, s_coef, s_tay, gv);
            else gates_of<G, CL, false, false>(g, sh, c0, s_coef, s_tay, gv);
#pragma unroll
            for (int q = 0; q < CPW; q++) s_dt[(c0 + q) * LDS_STRIDE + tu] = sg_fma(s_dt[(c0 + q) * LDS_STRIDE + tu], gv[q], dx[q]);
        }
        __syncthreads();

        // out_proj of the wave's SCAN_TT / WAVES timesteps: a block of the matrix instruction is four timesteps by four rows
        {
            constexpr int GROUPS = DM / 4, TW = SCAN_TT / WAVES;
            const int n = lane & 3, rows4 = (lane >> 2) % GROUPS, quad = (lane >> 2) / GROUPS, t = (TW * wave + 4 * quad + n) & (SCAN_TT - 1);
            const float* w = s_wout + (4 * rows4 + n) * WSTRIDE;      // A operand: row lane % 4 of the block's four
            const float* o = s_dt + t;                                // B operand: the lane's timestep
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int m = 0; m < DI; m += 4) {
                const f32x4 w4 = *reinterpret_cast<const f32x4*>(w + m);
#pragma unroll
                for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_4x4x1f32(w4[e], o[(m + e) * LDS_STRIDE], acc, 0, 0, 0);
            }
            const int at = __shfl(orig, t, 64);
            const bool mine = 4 * quad < TW && tile0 + t < u1;       // (eight waves have twice the lanes that the timesteps need)
            held_dst = mine ? reinterpret_cast<f32x4*>(pl.ctx + ((size_t)dir * pl.total + off + at) * DM + 4 * rows4) : nullptr;
            held = acc;
        }
    }
    if (held_dst != nullptr) *held_dst = held;
    if (u1 == N) {   // last chunk in scan order: new carried state of the tensor
        float* st = dir ? T.mbwd : T.mfwd;
#pragma unroll
        for (int h = 0; h < CL; h++)
            if (col(h) < pl.st_di && 2 * p < pl.st_ds) {
                st[col(h) * pl.st_ds + 2 * p] = S[h].he;
                st[col(h) * pl.st_ds + 2 * p + 1] = S[h].ho;
            }
    }
}

// Start state of every chunk: h_{c+1} = M_c h_c + b_c, applied in order from
// the carried state of the tensor.  One workgroup per (tensor, direction).
// The recurrence itself is a handful of fmas per chunk; what matters is the
// latency of fetching 3 KB (12 KB for the large geometry) of summaries per chunk,
// so the 1024 lanes of the workgroup, as groups of one chunk's lanes each, stream
// batches of chunks into LDS (next batch prefetched into registers) and group 0
// applies them.
constexpr int PREFIX_PER_GROUP = 4;

template <class G>
__global__ __launch_bounds__(1024) void k_chunk_prefix(Plan pl) {
    constexpr int HP = G::HP, SCAN_THREADS = G::THREADS;
    constexpr int PREFIX_GROUPS = 1024 / SCAN_THREADS;             // 8 groups of 128 lanes, or 2 of 512
    constexpr int PREFIX_BATCH = PREFIX_PER_GROUP * PREFIX_GROUPS;
    __shared__ float lds[PREFIX_BATCH * 6 * SCAN_THREADS];     // 96 KB
    const int ti = blockIdx.x % pl.P, dir = blockIdx.x / pl.P;
    const TensorDev& T = pl.tensors[ti];
    if (T.numel == 0) return;
    const int lane = threadIdx.x % SCAN_THREADS, grp = threadIdx.x / SCAN_THREADS;
    const int j = lane / HP, p = lane % HP;
    float* __restrict__ hs = pl.hstart + ((size_t)(dir * pl.chunks + pl.chunk_prefix[ti]) * 2) * SCAN_THREADS;
    const float* __restrict__ sm = pl.summaries + (size_t)(dir * pl.wchunks + pl.wchunk_prefix[ti]) * 6 * SCAN_THREADS;
    const int ns = T.nchunks - 1;                               // summaries to apply
    float he = 0.0f, ho = 0.0f;
    if (grp == 0) {
        // the caller's state is [st_di][st_ds] (its own d_inner, d_state); the rest of the kernel geometry starts at 0
        const float* st = dir ? T.mbwd : T.mfwd;
        if (j < pl.st_di && 2 * p < pl.st_ds) {
            he = st[j * pl.st_ds + 2 * p];
            ho = st[j * pl.st_ds + 2 * p + 1];
        }
        hs[lane] = he;
        hs[SCAN_THREADS + lane] = ho;
    }
    // every summary has an exactly zero 2x2 part: the replay takes its start states from the summaries themselves
    if (__builtin_amdgcn_readfirstlane(*pl.contracted) != 0) return;
    float r[PREFIX_PER_GROUP][6];
    auto prefetch = [&](int b) {
#pragma unroll
        for (int q = 0; q < PREFIX_PER_GROUP; q++) {
            const int c = b * PREFIX_BATCH + grp + PREFIX_GROUPS * q;
#pragma unroll
            for (int k = 0; k < 6; k++) r[q][k] = (c < ns) ? sm[((size_t)c * 6 + k) * SCAN_THREADS + lane] : 0.0f;
        }
    };
    prefetch(0);
    for (int b = 0; b * PREFIX_BATCH < ns; b++) {
#pragma unroll
        for (int q = 0; q < PREFIX_PER_GROUP; q++)
#pragma unroll
            for (int k = 0; k < 6; k++) lds[((grp + PREFIX_GROUPS * q) * 6 + k) * SCAN_THREADS + lane] = r[q][k];
        __syncthreads();
        prefetch(b + 1);
        if (grp == 0) {
            const int lim = min(PREFIX_BATCH, ns - b * PREFIX_BATCH);
            for (int cc = 0; cc < lim; cc++) {
                const float* m = lds + cc * 6 * SCAN_THREADS + lane;
                // a lane whose 2x2 part is exactly zero takes the offset itself, which is what 0 * h + b is for every finite h;
                // a state that is not finite goes through the product and stays non-finite to the end of the tensor
                const bool zero = m[0] == 0.0f && m[SCAN_THREADS] == 0.0f && m[2 * SCAN_THREADS] == 0.0f && m[3 * SCAN_THREADS] == 0.0f &&
                                  sg_isfinite(he) && sg_isfinite(ho);
                const float ne = sg_fma(m[0], he, sg_fma(m[2 * SCAN_THREADS], ho, m[4 * SCAN_THREADS]));
                const float no = sg_fma(m[SCAN_THREADS], he, sg_fma(m[3 * SCAN_THREADS], ho, m[5 * SCAN_THREADS]));
                he = zero ? m[4 * SCAN_THREADS] : ne;
                ho = zero ? m[5 * SCAN_THREADS] : no;
                float* h1 = hs + (size_t)(b * PREFIX_BATCH + cc + 1) * 2 * SCAN_THREADS;
                h1[lane] = he;
                h1[SCAN_THREADS + lane] = ho;
            }
        }
        __syncthreads();
    }
}

template <class G, int CL>
void launch_summary(const Plan& pl, hipStream_t st) {
    hipLaunchKernelGGL((k_summary<G, CL>), dim3(2 * pl.wchunks), dim3(64 * Split<G, CL>::WAVES), 0, st, pl);
}
template <class G, int CL>
void launch_replay_cols(const Plan& pl, hipStream_t st) {
    hipLaunchKernelGGL((k_replay_cols<G, CL>), dim3(2 * pl.chunks), dim3(64 * Split<G, CL>::WAVES), 0, st, pl);
}

template <class G>
int launch_scan_geo(const Plan& pl, hipStream_t st) {
    // One column per lane while all waves of the call are then resident at once (two per SIMD): a chunk's steps are a serial
    // chain, and a wave alone on its SIMD takes as long for one column's instructions as two waves for theirs.  Replay and
    // summaries of 30 000 elements 137 -> 102 us a step (large geometry 222 -> 160), of 200 000 229 -> 183; past the line
    // two columns are ahead, by 3 % at 300 000 elements, by 7 % at 120 000 of the large geometry.
    constexpr int RESIDENT = 2 * 4 * 256;
    const auto single = [](int chunks) { return 2 * chunks * Split<G, 1>::WAVES <= RESIDENT; };
    if (pl.wchunks > 0) {
        if (single(pl.wchunks)) launch_summary<G, 1>(pl, st);
        else launch_summary<G, 2>(pl, st);
        SG_LAUNCH_CHECK("k_summary");
    }
    prof_mark(2, st);
    if (pl.wchunks > 0) {      // (tensors of one chunk start from their carried state without it)
        hipLaunchKernelGGL(k_chunk_prefix<G>, dim3(2 * pl.P), dim3(1024), 0, st, pl);
        SG_LAUNCH_CHECK("k_chunk_prefix");
    }
    prof_mark(3, st);
    constexpr bool DEFAULT = G::THREADS == 128;
    if (pl.htile != nullptr && !DEFAULT) return sg::fail("the bilevel pass is built for the default meta-net dimensions only");
    if (pl.htile == nullptr && single(pl.chunks)) {
        launch_replay_cols<G, 1>(pl, st);
    } else if constexpr (DEFAULT) {          // one wave per chunk, two columns per lane
        if (pl.htile != nullptr) hipLaunchKernelGGL((k_replay<G, true>), dim3(2 * pl.chunks), dim3(64), 0, st, pl);
        else hipLaunchKernelGGL((k_replay<G, false>), dim3(2 * pl.chunks), dim3(64), 0, st, pl);
    } else {
        launch_replay_cols<G, 2>(pl, st);
    }
    SG_LAUNCH_CHECK("k_replay");
    prof_mark(4, st);
    return 0;
}

}  // namespace

int launch_scan(const Plan& pl, hipStream_t st) {
    if (pl.total == 0) return 0;
    return pl.geo == GEO_LARGE ? launch_scan_geo<GeoLarge>(pl, st) : launch_scan_geo<GeoDefault>(pl, st);
}

}  // namespace sg2
