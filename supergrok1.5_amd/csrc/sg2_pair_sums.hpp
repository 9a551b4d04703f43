// Sums over the lanes that hold the RoPE pairs of one column, for the scan and its adjoint.
#pragma once

#include "sg_common.hpp"

namespace sg2 {
namespace {

__device__ __forceinline__ float dpp_quad_swap1(float v) {   // lane ^ 1
    return sg_i2f(__builtin_amdgcn_update_dpp(0, sg_f2i(v), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_quad_swap2(float v) {   // lane ^ 2
    return sg_i2f(__builtin_amdgcn_update_dpp(0, sg_f2i(v), 0x4E, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_half_mirror(float v) {  // lane -> 7 - lane within each group of 8
    return sg_i2f(__builtin_amdgcn_update_dpp(0, sg_f2i(v), 0x141, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_row_mirror(float v) {   // lane -> 15 - lane within each group of 16
    return sg_i2f(__builtin_amdgcn_update_dpp(0, sg_f2i(v), 0x140, 0xF, 0xF, true));
}
// sum over the HP lanes of a (column) group.  The tree folds the group in halves, mirrored, until four sums are left:
// HP = 8: s_i = y_i + y_(7-i), total = (s_0 + s_1) + (s_2 + s_3); HP = 16: r_i = y_i + y_(15-i) first, then the same on r.
// (Mirrored folds first, because a fold across DPP banks can be written to some banks only: see block_pair_sums.)
template <int HP>
__device__ __forceinline__ float pair_tree_sum(float y) {
    if (HP == 16) y = y + dpp_row_mirror(y);
    y = y + dpp_half_mirror(y);
    y = y + dpp_quad_swap1(y);
    y = y + dpp_quad_swap2(y);
    return y;
}
// The same sums for the 8 steps of a block in 16 instructions instead of 24 (32 for HP = 16).  A DPP instruction can
// be restricted to some banks (groups of four lanes) of every row of 16, leaving the destination's other lanes as
// they were.  After a mirrored fold both halves of the folded group hold the same sums, so two steps' folds are
// written into ONE register - step u into the first half's lanes, step u + 4 into the second half's - and the rest
// of the tree runs on half as many registers.  Additions commute bit for bit, so every lane that ends up holding a
// step's total holds pair_tree_sum's value.  On return, for HP = 8, y[k] (k < 4) is the total of step k + 4 (p >> 2)
// in lane (j, p); for HP = 16, y[m] (m < 2) that of step m + 2 (p >> 2).
// (Inline assembly: the compiler has no form for a bank-masked DPP addition that keeps the other lanes, and it does
// not see a hazard between instructions inside the block - a DPP operand must not be read within two instructions of the
// vector instruction that wrote it, hence the order of the instructions and the s_nop.)
template <int HP>
__device__ __forceinline__ void block_pair_sums(float (&y)[8]) {
    float z0, z1, z2, z3;
    if (HP == 8) {
        asm volatile(
            "s_nop 1\n\t"
            "v_add_f32_dpp %0, %4, %4 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
            "v_add_f32_dpp %0, %8, %8 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
            "v_add_f32_dpp %1, %5, %5 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
            "v_add_f32_dpp %1, %9, %9 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
            "v_add_f32_dpp %2, %6, %6 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
            "v_add_f32_dpp %2, %10, %10 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
            "v_add_f32_dpp %3, %7, %7 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
            "v_add_f32_dpp %3, %11, %11 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
            "v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_add_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_add_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_add_f32_dpp %3, %3, %3 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_add_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_add_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_add_f32_dpp %3, %3, %3 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "s_nop 1"
            : "=&v"(z0), "=&v"(z1), "=&v"(z2), "=&v"(z3)
            : "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "v"(y[4]), "v"(y[5]), "v"(y[6]), "v"(y[7]));
        y[0] = z0; y[1] = z1; y[2] = z2; y[3] = z3;
    } else {
        asm volatile(
            "s_nop 1\n\t"
            "v_add_f32_dpp %0, %4, %4 row_mirror row_mask:0xf bank_mask:0x3\n\t"
            "v_add_f32_dpp %0, %8, %8 row_mirror row_mask:0xf bank_mask:0xc\n\t"
            "v_add_f32_dpp %1, %5, %5 row_mirror row_mask:0xf bank_mask:0x3\n\t"
            "v_add_f32_dpp %1, %9, %9 row_mirror row_mask:0xf bank_mask:0xc\n\t"
            "v_add_f32_dpp %2, %6, %6 row_mirror row_mask:0xf bank_mask:0x3\n\t"
            "v_add_f32_dpp %2, %10, %10 row_mirror row_mask:0xf bank_mask:0xc\n\t"
            "v_add_f32_dpp %3, %7, %7 row_mirror row_mask:0xf bank_mask:0x3\n\t"
            "v_add_f32_dpp %3, %11, %11 row_mirror row_mask:0xf bank_mask:0xc\n\t"
            "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
            "v_add_f32_dpp %1, %1, %1 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
            "s_nop 0\n\t"
            "v_add_f32_dpp %0, %2, %2 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
            "v_add_f32_dpp %1, %3, %3 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
            "s_nop 1\n\t"
            "v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_add_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "s_nop 1\n\t"
            "v_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_add_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "s_nop 1"
            : "=&v"(z0), "=&v"(z1), "=&v"(z2), "=&v"(z3)
            : "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "v"(y[4]), "v"(y[5]), "v"(y[6]), "v"(y[7]));
        y[0] = z0; y[1] = z1;
    }
}

}  // namespace
}  // namespace sg2
