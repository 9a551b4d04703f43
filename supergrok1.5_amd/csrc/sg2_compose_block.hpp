// What the scan derives from the meta-net's weights once per call: composed
// coefficient triples, Taylor polynomials, polynomial limits and the length of
// a summary's first block (include/sg2_compose.h).  One workgroup's work, and
// nothing of it depends on the gradients: it runs as an extra workgroup of the
// sort's first launch, so its latency (a launch of its own took 15 us, 51 us for
// the large geometry, on the critical path of every step) passes under the sort.
// The composition is carried by d_inner x 3 x 2 lanes into LDS first instead of
// by every row's lane for itself; the order of the products is
// sg2_compose_one's, so the bits are too.
#pragma once

#include "sg2_internal.hpp"
#include "../../include/sg2_compose.h"

namespace sg2 {
namespace {

// threads: block size, at least 2 * SG2_COMP_GROUPS * G::ROWS
template <class G>
__device__ __forceinline__ void compose_block(const Plan& pl, int threads) {
    constexpr int ROWS = G::ROWS, DM = G::DM, DI = G::DI, LANES = 2 * SG2_COMP_GROUPS * ROWS;
    static_assert(ROWS == DI, "one row of dt, B, C and z per column");
    __shared__ double s_xb[2][DI][3];
    __shared__ float s_dt0[2][ROWS];
    __shared__ int s_largest, s_zero, s_bad, s_cmax[2][2], s_cdt[2][2], s_amax[2], s_fmax[2], s_slope[2];
    const int tid = threadIdx.x;
    if (tid == 0) {
        s_largest = 0; s_zero = 0; s_bad = 0;
        for (int k = 0; k < 2; k++) { s_cmax[k][0] = s_cmax[k][1] = s_cdt[k][0] = s_cdt[k][1] = s_amax[k] = s_fmax[k] = s_slope[k] = 0; }
    }
    const float* const Win = pl.W.w[W_IN_W];
    const float* const bin = pl.W.w[W_IN_B];
    // one linear form of the 8 (16) input-projection entries: w . (W_in[:, c] | b_in)
    auto through_input = [&](const float* w, int c) {
        double acc = 0.0;
#pragma unroll
        for (int k = 0; k < DM; k++) acc = acc + (double)w[k] * (double)(c == 2 ? bin[k] : Win[2 * k + c]);
        return acc;
    };
    for (int t = tid; t < 2 * DI * 3; t += threads) {
        const int dir = t / (DI * 3), j = t / 3 % DI, c = t % 3;
        s_xb[dir][j][c] = through_input(pl.W.w[dir ? W_B_INPROJ : W_F_INPROJ] + j * DM, c);
    }
    __syncthreads();
    const bool active = tid < LANES;
    const int dir = active ? tid / (SG2_COMP_GROUPS * ROWS) : 0, r = tid % (SG2_COMP_GROUPS * ROWS);
    const int group = r / ROWS, row = r % ROWS;
    const int b = dir ? W_B_INPROJ : W_F_INPROJ;
    float out[3] = {0.0f, 0.0f, 0.0f};
    if (active) {
        if (group == SG2_COMP_XB) {
            for (int c = 0; c < 3; c++) out[c] = (float)s_xb[dir][row][c];
        } else if (group == SG2_COMP_Z) {
            for (int c = 0; c < 3; c++) out[c] = (float)through_input(pl.W.w[b] + (DI + row) * DM, c);
        } else {
            const float* w = pl.W.w[b + (group == SG2_COMP_DT ? 1 : group == SG2_COMP_B ? 3 : 4)] + row * DI;
            double acc[3] = {0.0, 0.0, group == SG2_COMP_DT ? (double)pl.W.w[b + 2][row] : 0.0};
            for (int j = 0; j < DI; j++)
                for (int c = 0; c < 3; c++) acc[c] = acc[c] + (double)w[j] * s_xb[dir][j][c];
            for (int c = 0; c < 3; c++) out[c] = (float)acc[c];
        }
        float* dst = pl.comp + (size_t)tid * 3;
        dst[0] = out[0];
        dst[1] = out[1];
        dst[2] = out[2];
    }
    // Taylor polynomials of the step size and of the gate around their zero-input arguments (sg2_compose.h), and the
    // largest |c_g|, |c_s| of those rows (bit patterns of non-negative floats order like integers)
    if (active && (group == SG2_COMP_DT || group == SG2_COMP_Z)) {
        float t[4];
        if (group == SG2_COMP_DT) sg2_softplus_taylor(out[2], t);
        else sg2_silu_taylor(out[2], t);
        float* tay = pl.comp + 2 * SG2_COMP_GROUPS * ROWS * 3 + ((dir * 2 + (group == SG2_COMP_Z ? 1 : 0)) * ROWS + row) * 4;
        tay[0] = t[0]; tay[1] = t[1]; tay[2] = t[2]; tay[3] = t[3];
        atomicMax(&s_cmax[dir][0], sg_f2i(sg_abs(out[0])));
        atomicMax(&s_cmax[dir][1], sg_f2i(sg_abs(out[1])));
        if (group == SG2_COMP_DT) {
            atomicMax(&s_cdt[dir][0], sg_f2i(sg_abs(out[0])));
            atomicMax(&s_cdt[dir][1], sg_f2i(sg_abs(out[1])));
            atomicMax(&s_slope[dir], sg_f2i(sg2_dt_slope(out[2])));       // positive: its bit pattern orders like the value
            s_dt0[dir][row] = sg_softplus(out[2]);
        }
    }
    for (int i = tid; i < pl.P; i += threads)
        if (pl.state_bad[i] != 0) s_bad = 1;       // plain store: every writer stores the same value
    __syncthreads();
    // How many steps the first block of a chunk summary should cover: what the slowest pair of either direction needs
    // to contract at the step size a zero input gives (sg2_contraction_steps, sg2_first_block_steps).
    // For sg2_poly_ok: the largest -A/2 and the largest |rotation frequency| of each direction.
    for (int t = tid; t < 2 * ROWS * G::HP; t += threads) {
        const int d = t / (ROWS * G::HP), j = t / G::HP % ROWS, p = t % G::HP;
        const float* alog = pl.W.w[d ? W_B_ALOG : W_F_ALOG] + j * G::DS;
        const float a_e = -0.5f * -sg_exp(alog[2 * p]), a_o = -0.5f * -sg_exp(alog[2 * p + 1]);
        const int n = sg2_contraction_steps(s_dt0[d][j], a_e, a_o);
        if (n == 0) atomicOr(&s_zero, 1);
        atomicMax(&s_largest, n);
        atomicMax(&s_amax[d], sg_f2i(sg_max(a_e, a_o)));
        atomicMax(&s_fmax[d], sg_f2i(sg_abs(pl.W.w[d ? W_B_ROPE : W_F_ROPE][j * G::HP + p])));
    }
    __syncthreads();
    if (tid == 0) {
        pl.contracted[0] = s_bad == 0 ? 1 : 0;      // until a summary kernel finds a chunk that has not contracted; never while a carried state is not finite
        pl.contracted[2] = s_bad;
        pl.contracted[1] = sg2_first_block_steps(s_largest, s_zero);
        float* cmax = pl.comp + 2 * SG2_COMP_GROUPS * ROWS * 3 + 2 * 2 * ROWS * 4;
        cmax[0] = sg_i2f(s_cmax[0][0]); cmax[1] = sg_i2f(s_cmax[0][1]);
        cmax[2] = sg_i2f(s_cmax[1][0]); cmax[3] = sg_i2f(s_cmax[1][1]);
        for (int k = 0; k < 2; k++) {
            const float slope = sg_i2f(s_slope[k]);      // how much of a change of its argument the step size follows at most
            const float kp = sg2_limit_factor(sg_max(128.0f * sg_i2f(s_amax[k]), 256.0f * sg_i2f(s_fmax[k])), slope);
            cmax[4 + 2 * k] = kp * sg_i2f(s_cdt[k][0]);
            cmax[5 + 2 * k] = kp * sg_i2f(s_cdt[k][1]);
            // ... and for the products of the output pass (sg2_pair_products)
            const float kprod = sg_fma(416.0f, sg_i2f(s_amax[k]), 184.0f * sg_i2f(s_fmax[k]));
            const float kq = sg2_limit_factor(kprod, slope);
            cmax[16 + k] = 1.0f / kprod;                // how far dt can be from dt0 there (sg2_shrink8)
            cmax[8 + 2 * k] = kq * sg_i2f(s_cdt[k][0]);
            cmax[9 + 2 * k] = kq * sg_i2f(s_cdt[k][1]);
            // ... and for the polynomials of the adjoint (sg2_bilevel.hip)
            const float kc = sg2_limit_factor(sg_max(80.0f * sg_i2f(s_amax[k]), 256.0f * sg_i2f(s_fmax[k])), slope);
            cmax[12 + 2 * k] = kc * sg_i2f(s_cdt[k][0]);
            cmax[13 + 2 * k] = kc * sg_i2f(s_cdt[k][1]);
        }
    }
}

}  // namespace
}  // namespace sg2
