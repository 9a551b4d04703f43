// Muon step: momentum (which also leaves the bf16 work copy), Frobenius norm (folded into the first iteration), quintic Newton-Schulz
// orthogonalisation as 16-bit MFMA GEMMs with fp32 accumulation, parameter
// update.  Replaces the body of muon_fused_step (csrc/ops.cpp:663-746 of the
// reference: ATen norm + one host sync, three torch::mm per iteration,
// muon_ns_combine_kernel / muon_update_kernel of csrc/muon_kernels.cu:37-72).
//
// Every matrix is worked on in its "wide" orientation Y [m x n] (m = min dim)
// so the Gram matrix is always the small m x m one:
//     G = Y Y^T            H = a I + b G + c G G            Y <- H Y
// (the a Y term rides on H's diagonal, so the apply step is one product with no third operand; the diagonal entry
// is rounded to bf16 like every other entry of H: against the fp32 iteration this is no less accurate than adding
// a Y in the epilogue, the error of either form is set by the rounding of G)
// (for a tall parameter X this is X^T X and X (bG + cG^2): the reference's
// X X^T form re-associated, 6 m^2 n instead of 6 n^2 m flops per iteration).
// Forming G from Y costs as much as n / m small products, the apply step as much as 2 n / m.  The polynomials of one iterate
// commute, so several iterations share both (a stage): with G tracked instead of formed again,
//     P = a I + b G + c G G        Q <- P Q        G <- P G P, as S = P G and S P
// and Y <- Q Y at the stage's end.  Five iterations are two stages, of two and three: 2 (n/m + 2 n/m) + 14 small products where
// one stage an iteration takes 5 (n/m + 2 n/m) + 5.  A tracked G drifts from Y Y^T by its roundings, which small singular
// values feel (they grow by a = 3.4 an iteration, those of G by its square): not more than three iterations a stage, and
// everything but the momentum itself and what multiplies it in half precision, eight times finer than bf16 (numbers stay
// below 1.3 resp. 41, scales in F16_SCALE).  Distance from float64 over Gaussian, low-rank, power-law, sparse and row-scaled
// matrices: 0.24-0.98 of that of five stages in bf16 (1024 x 4096 Gaussian 3.0e-3 against 6.9e-3).  Columns (of the wide
// orientation) spread over six decades and more are the exception: there the drift of the second stage is 0.011 to 0.018
// where bf16 is at 0.0095 (three iterations before two would be 0.006, but 6.4e-3 on a Gaussian).  All five in one stage
// would be 0.107 against 0.017 on a power law.  24 bf16 matrices of 1024 x 4096: 2178 -> 1622 us a step.
// The Gram and polynomial products are "NT" GEMMs (both operands K-contiguous).
// The apply step is (on 256x256 tiles) an "NN" one: its B operand is Y itself, whose K axis is
// the slow one.  Its tiles are staged in LDS as they lie in memory
// ([k][n], n contiguous) and the MFMA operand (8 consecutive k per lane) is
// fetched with gfx950's transposing LDS read (ds_read_b64_tr_b16), so no
// transposed copy of Y is kept: an iteration reads Y as an operand of two products and writes it once,
// into the other of two buffers (the current one is still being read as the B
// operand by other workgroups).  A tall parameter enters and leaves the wide
// orientation in the momentum and update kernels, which transpose 64x64 tiles
// through LDS.
// Work buffers are padded with zeros to multiples of 256 (64 where no product takes 256x256 tiles), written by the momentum
// kernel, so the products need no edge handling (zero rows/columns stay zero through the iteration).
// A call whose matrices all fit the LDS of a CU (k_newton_schulz) takes one launch for the whole iteration instead of
// three products a step; products that would leave most of the chip idle go to 64x64 tiles (k_gemm_64, choose_tiles).
//
// GEMM: 256x256 output tile per 512-thread workgroup, 8 waves as 2x4, each
// wave 128x64 = 4x2 MFMA 32x32x16 bf16 tiles (128 fp32 accumulators per
// lane, two waves per SIMD), K tiles of 32 in four LDS stages, filled by loads that go from global
// memory straight into LDS (global_load_lds_dwordx4) three tiles ahead of their
// use; no padding is possible in such a copy, so the tiles are swizzled by the
// choice of the chunk each lane fetches (conflict-free operand fetches); memory
// instructions are dealt between the MFMAs.  A 256x256 tile takes 128 flop per
// byte fetched, which keeps the MFMA pipe ahead of the ~64 B/clk a CU can pull
// from L2; the symmetric products (G and G*G) compute only the tiles on or above
// the diagonal.  Tile index -> XCD-contiguous order so that the workgroups
// sharing operand panels share an L2.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "sg_common.hpp"
#include <type_traits>

namespace sgmu {
namespace {

typedef uint16_t bf16_t;           // sixteen bits of either type: what a buffer holds is known where it is used
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
enum { T_BF16 = 0, T_F16 = 1 };
// Half-precision iterates and Gram matrices (and S) are held times 2^14: the largest singular value stays below 1.3 throughout,
// so no entry can overflow, and full precision reaches down to 4e-9.  Polynomials and their products, below 41, are held times
// 2^10: a row far below the others meets them only in entries as small as it is, and at a scale of one rows 1e-5 and 1e-6 times
// as large as the others of 700 x 2800 came out 4 and 40 % off after five iterations (now 0.4 %; 0.6 % at 1e-7).  (Powers of two:
// the factors round nothing.)
constexpr float F16_SCALE = 16384.0f, F16_UNSCALE = 1.0f / 16384.0f, POLY_SCALE = 1024.0f, POLY_UNSCALE = 1.0f / 1024.0f;

constexpr int BT = 256;            // GEMM tile (M and N)
// Waves of a workgroup along N (2 along M).  Eight waves of 128 x 64 (two per SIMD, 128 accumulators each) measured
// 3.5 % faster per step than four waves of 128 x 128: they fetch 1.5 x the operand bytes from LDS, but a second wave per
// SIMD covers the fetch latencies that one wave cannot.
constexpr int GWN = 4;
constexpr int GWAVES = 2 * GWN, GTHREADS = 64 * GWAVES;
constexpr int WCOLS = BT / GWN;      // columns of a wave's block
constexpr int GEMM_LDS_BYTES = 4 * 2 * BT * 32 * 2;          // four stages of {A tile, B tile} of 32 k: 131,072 bytes of the CU's 160 KB
constexpr float NS_A = 3.4445f, NS_B = -4.7750f, NS_C = 2.0315f;

struct Mat {
    void* param;
    const void* grad;
    float* buf;
    bf16_t *Y, *Y2;                // [mp x np] twice (an apply step reads one and writes the other)
    bf16_t* W[5];                  // [mp x mp]: Gram matrices, polynomials and their products (the last three only where iterations can share them)
    bf16_t *T, *T2;                // the transposes of Y and Y2 [np x mp], or NULL (kept for k_gemm_64's apply step)
    int rows, cols, dtype;
    int m, n, mp, np;              // min / max dim and their padded sizes
    int wide;                      // rows <= cols
    int vec8;                      // cols % 8 == 0 and param/grad/buf 16-byte aligned: elementwise kernels move 8 elements per lane
};

struct Batch {
    const Mat* mats;
    const int* gtile_prefix[3];    // [P+1] GEMM output tiles for the three products
    const int* ttile_prefix;       // [P+1] 64x64 tiles of Y (the elementwise kernels work on these)
    int P, gtiles[3], ttiles;
    double* partials;              // [ttiles] sums of squares of the 64x64 tiles
    float* inv_norm;               // [P]
};

// ---- momentum + sum of squares ------------------------------------------------
__device__ __forceinline__ double block_sum(double v, double* sm) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_down(v, d, 64);
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = v;
    __syncthreads();
    const double r = (sm[0] + sm[1]) + (sm[2] + sm[3]);
    __syncthreads();
    return r;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// eight consecutive elements in the tensor's storage type; i a multiple of 8, base 16-byte aligned
__device__ __forceinline__ void load8(const void* p, int dtype, size_t i, float v[8]) {
    if (dtype == SG_F32) {
        const SG_GLOBAL f32x4* q = (const SG_GLOBAL f32x4*)(static_cast<const float*>(p) + i);
        const f32x4 a = q[0], b = q[1];
#pragma unroll
        for (int k = 0; k < 4; k++) { v[k] = a[k]; v[4 + k] = b[k]; }
    } else {
        const u32x4 w = *(const SG_GLOBAL u32x4*)(static_cast<const uint16_t*>(p) + i);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint16_t h = (uint16_t)((k & 1) ? (w[k >> 1] >> 16) : (w[k >> 1] & 0xffffu));
            v[k] = (dtype == SG_F16) ? __half2float(__ushort_as_half(h)) : sg::bf16_bits_to_f(h);
        }
    }
}
__device__ __forceinline__ void store8(void* p, int dtype, size_t i, const float v[8]) {
    if (dtype == SG_F32) {
        SG_GLOBAL f32x4* q = (SG_GLOBAL f32x4*)(static_cast<float*>(p) + i);
        q[0] = f32x4{v[0], v[1], v[2], v[3]};
        q[1] = f32x4{v[4], v[5], v[6], v[7]};
    } else {
        u32x4 w;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t lo = (dtype == SG_F16) ? __half_as_ushort(__float2half_rn(v[2 * k])) : sg::f_to_bf16_bits(v[2 * k]);
            const uint32_t hi = (dtype == SG_F16) ? __half_as_ushort(__float2half_rn(v[2 * k + 1])) : sg::f_to_bf16_bits(v[2 * k + 1]);
            w[k] = lo | (hi << 16);
        }
        *(SG_GLOBAL u32x4*)(static_cast<uint16_t*>(p) + i) = w;
    }
}

// buf = momentum * buf + grad, the sum of squares of the new buf, and the new buf as bf16 into Y ([mp x np], the wide
// orientation) - NOT yet divided by its norm, which is only known once every tile of the matrix has been summed: the
// first iteration's Gram and apply epilogues carry the factors 1/norm^2 and 1/norm instead (bf16 rounding is relative,
// so rounding before or after the scaling costs the same), and no separate normalisation pass reads buf again.
// One 64x64 tile of the parameter's own orientation per workgroup: rows are read and written along the fast axis, a
// tall parameter's tile is transposed through LDS.
__global__ __launch_bounds__(256) void k_momentum(Batch B, float momentum) {
    __shared__ bf16_t t[64][66];
    __shared__ double sm[4];
    const int mi = sg::upper_seg(B.ttile_prefix, B.P, blockIdx.x);
    const Mat& M = B.mats[mi];
    bf16_t* own = M.wide ? M.Y : M.T;             // [R x C] in the parameter's orientation, padded
    bf16_t* other = M.wide ? M.T : M.Y;           // [C x R]
    const int R = M.wide ? M.mp : M.np, C = M.wide ? M.np : M.mp;
    const int tile = (int)blockIdx.x - B.ttile_prefix[mi];
    const int tc = C / 64, tr0 = (tile / tc) * 64, tc0 = (tile % tc) * 64;
    const bool w_own = own != nullptr, w_other = other != nullptr;               // uniform over the workgroup
    const bool full = tr0 + 64 <= M.rows && tc0 + 64 <= M.cols && M.vec8;
    double acc = 0.0;
    if (full) {
        // interior tile: a lane moves 16 consecutive elements of a row
        const int lr = threadIdx.x >> 2, c0 = (threadIdx.x & 3) * 16;
        const size_t at = (size_t)(tr0 + lr) * M.cols + tc0 + c0;
        float g[16], b[16], part = 0.0f;
        load8(M.grad, M.dtype, at, g);
        load8(M.grad, M.dtype, at + 8, g + 8);
        load8(M.buf, SG_F32, at, b);
        load8(M.buf, SG_F32, at + 8, b + 8);
#pragma unroll
        for (int e = 0; e < 16; e++) { b[e] = sg_fma(momentum, b[e], g[e]); part = sg_fma(b[e], b[e], part); }
        store8(M.buf, SG_F32, at, b);
        store8(M.buf, SG_F32, at + 8, b + 8);
        acc = (double)part;
        uint32_t pk[8];
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const uint32_t b0 = sg::f_to_bf16_bits(b[2 * q]), b1 = sg::f_to_bf16_bits(b[2 * q + 1]);
            pk[q] = b0 | (b1 << 16);
            t[lr][c0 + 2 * q] = (bf16_t)b0;
            t[lr][c0 + 2 * q + 1] = (bf16_t)b1;
        }
        if (w_own) {
            SG_GLOBAL u32x4* dst = (SG_GLOBAL u32x4*)(own + (size_t)(tr0 + lr) * C + tc0 + c0);
            dst[0] = u32x4{pk[0], pk[1], pk[2], pk[3]};
            dst[1] = u32x4{pk[4], pk[5], pk[6], pk[7]};
        }
        if (w_other) {
            __syncthreads();
            // transposed copy: output row lr (= own column), 16 consecutive output columns (= own rows)
#pragma unroll
            for (int q = 0; q < 8; q++) pk[q] = (uint32_t)t[c0 + 2 * q][lr] | ((uint32_t)t[c0 + 2 * q + 1][lr] << 16);
            SG_GLOBAL u32x4* dt = (SG_GLOBAL u32x4*)(other + (size_t)(tc0 + lr) * R + tr0 + c0);
            dt[0] = u32x4{pk[0], pk[1], pk[2], pk[3]};
            dt[1] = u32x4{pk[4], pk[5], pk[6], pk[7]};
        }
    } else {
        float part = 0.0f;
        for (int k = threadIdx.x; k < 64 * 64; k += 256) {
            const int r = tr0 + (k >> 6), c = tc0 + (k & 63);
            bf16_t v = 0;
            if (r < M.rows && c < M.cols) {
                const size_t i = (size_t)r * M.cols + c;
                const float bv = sg_fma(momentum, M.buf[i], sg::load_elem(M.grad, M.dtype, (int64_t)i));
                M.buf[i] = bv;
                part = sg_fma(bv, bv, part);
                v = sg::f_to_bf16_bits(bv);
            }
            if (w_own) own[(size_t)r * C + c] = v;
            t[k >> 6][k & 63] = v;
        }
        acc = (double)part;
        if (w_other) {
            __syncthreads();
            for (int k = threadIdx.x; k < 64 * 64; k += 256) {
                const int r = k >> 6, c = k & 63;     // output row r (= own column), column c (= own row)
                other[(size_t)(tc0 + r) * R + tr0 + c] = t[c][r];
            }
        }
    }
    const double tot = block_sum(acc, sm);
    if (threadIdx.x == 0) B.partials[blockIdx.x] = tot;
}

__global__ __launch_bounds__(256) void k_norm(Batch B) {
    __shared__ double sm[4];
    const int mi = blockIdx.x;
    double acc = 0.0;
    for (int k = B.ttile_prefix[mi] + (int)threadIdx.x; k < B.ttile_prefix[mi + 1]; k += 256) acc += B.partials[k];
    const double tot = block_sum(acc, sm);
    if (threadIdx.x == 0) B.inv_norm[mi] = 1.0f / ((float)sqrt(tot) + 1e-7f);
}

// ---- GEMM  C[M x N] = A[M x K] * B  with fused epilogues; B given as [N x K] (Gram, polynomial) or as [K x N] (apply)
// 256x256 output tile per workgroup of 2 x GWN waves, each wave 128 x (256/GWN) as MFMA 32x32x16 tiles.
// Per 16-wide k step a wave fetches 4+4 16-byte operands from LDS for 16 MFMAs.
// The Gram and polynomial products are symmetric: only tiles on or above the diagonal are
// computed, each off-diagonal tile is also stored transposed.
// EPI_MUL is a plain product of two commuting symmetric matrices, as symmetric as they are.
enum { EPI_GRAM = 0, EPI_POLY = 1, EPI_APPLY = 2, EPI_MUL = 3 };
constexpr int shape_of(int epi) { return epi == EPI_MUL ? EPI_POLY : epi; }      // whose tiles and tables it takes
// Which of Mat::W a launch reads and writes: W[c] = A(a) B(b); c2 >= 0: the second half of the grid forms W[c2] = W[a2] W[b2]
struct Ops {
    int a, b, c, a2, b2, c2;
};
// explicit global address space: a generic (flat) load would count against the LDS wait counter as well
typedef const __attribute__((address_space(1))) u32x4* gvec_p;
typedef __attribute__((address_space(1))) u32x4* gvec_w;

// two floats rounded to bf16 (nearest even, NaN stays NaN), packed lo | hi << 16: one v_cvt_pk_bf16_f32 on gfx950
__device__ __forceinline__ uint32_t bf16r2(float lo, float hi) {
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
}

template <int T>
__device__ __forceinline__ uint32_t round2(float lo, float hi) {
    if (T == T_BF16) return bf16r2(lo, hi);
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){lo, hi}, f16x2));
}
// entry k of two packed ones
template <int T>
__device__ __forceinline__ float widen(uint32_t w, int k) {
    if (T == T_BF16) return sg_i2f((int32_t)((k & 1) ? (w & 0xffff0000u) : (w << 16)));
    return __half2float(__ushort_as_half((uint16_t)((k & 1) ? (w >> 16) : (w & 0xffffu))));
}
template <int T>
__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
    if (T == T_BF16) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
// what a product is multiplied by besides the norm: the scales of half-precision operands and results (above)
template <int EPI, int IN, int OUT>
constexpr float epi_factor() {
    if (EPI == EPI_GRAM) return (IN == T_F16 ? F16_UNSCALE * F16_UNSCALE : 1.0f) * (OUT == T_F16 ? F16_SCALE : 1.0f);
    if (EPI == EPI_APPLY) return IN == T_F16 ? POLY_UNSCALE : OUT == T_F16 ? F16_SCALE : 1.0f;
    if (EPI == EPI_MUL) return OUT == T_F16 ? POLY_UNSCALE : POLY_UNSCALE * POLY_UNSCALE;       // one factor is a polynomial, both are where the result is one in bf16
    return 1.0f;
}
// b G + c G G from a product of G and an entry of it, and the a of the diagonal, as the operands and the result are held
template <int T>
__device__ __forceinline__ float polynomial(float gg, float g) {
    if (T == T_BF16) return sg_fma(NS_C, gg, NS_B * g);
    return sg_fma(NS_C * F16_UNSCALE * F16_UNSCALE * POLY_SCALE, gg, NS_B * F16_UNSCALE * POLY_SCALE * g);
}
template <int T>
constexpr float diagonal() { return T == T_BF16 ? NS_A : NS_A * POLY_SCALE; }

// The R operand reads of the next k step are dealt over the first eight of a phase's M MFMAs (R/8 after each, one more
// after the first R%8), the other MFMAs follow on their own
#define SG_MUON_SCHED_READS(R, M)                                                       \
    do {                                                                               \
        _Pragma("unroll") for (int g_ = 0; g_ < 8; g_++) {                              \
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                          \
            if ((R) / 8 + (g_ < (R) % 8 ? 1 : 0) == 2) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0); \
            else if ((R) / 8 + (g_ < (R) % 8 ? 1 : 0) == 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); \
        }                                                                              \
        if ((M) > 8) __builtin_amdgcn_sched_group_barrier(0x008, (M) - 8, 0);           \
    } while (0)

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4* lds_i16x4_p;

// y_sel: which of the two Y buffers holds the current iterate
// iter_flags: bit 1 = first iteration (Y still carries the factor norm: see k_momentum)
// IN, OUT: what the operands and the result are held in
template <int EPI, int IN, int OUT>
__global__ __launch_bounds__(GTHREADS) void k_gemm_nt(Batch Bt, Ops ops, int y_sel, int iter_flags) {
    constexpr bool BKN = EPI == EPI_APPLY;             // B operand stored [K x N]
    constexpr int TM = BT / 64, TN = WCOLS / 32;       // MFMA tiles per wave in each direction (4 x 4 or 4 x 2)
    constexpr int LPT = 16 / GWAVES;                  // loads per wave, tile and operand (a tile is 16 blocks of 1 KB)
    extern __shared__ __attribute__((aligned(16))) bf16_t smem[];

    // XCD-contiguous tile order: hardware deals consecutive workgroups round-robin over the 8 XCDs,
    // so that tiles that run together on an XCD share operand panels in its L2
    const int nblk = gridDim.x;
    int lb = blockIdx.x;
    if (nblk % 8 == 0) lb = (blockIdx.x % 8) * (nblk / 8) + blockIdx.x / 8;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / GWN, wn = wave % GWN;
    const sg::cint_p prefix = sg::as_const(Bt.gtile_prefix[shape_of(EPI)]);
    if (EPI == EPI_MUL && ops.c2 >= 0 && lb >= nblk / 2) { lb -= nblk / 2; ops.a = ops.a2; ops.b = ops.b2; ops.c = ops.c2; }
    const int mi = sg::upper_seg(prefix, Bt.P, lb);
    const Mat& Mt = Bt.mats[mi];
    int tile = lb - prefix[mi];

    const bf16_t *A, *B;
    bf16_t *C, *CT;         // CT: where the transposed tile goes (the symmetric products mirror into C itself)
    int K, lda, ldb, ldc, ldct, tm, tn;
    if (EPI == EPI_APPLY) {
        A = Mt.W[ops.a]; B = y_sel ? Mt.Y2 : Mt.Y; C = y_sel ? Mt.Y : Mt.Y2; K = Mt.mp; lda = Mt.mp; ldb = ldc = Mt.np;
        CT = C; ldct = ldc;      // unused: the apply step never mirrors
        // bands of 8 tile columns: 32 tiles that run together span 4 x 8 tiles instead of 2 x 16,
        // which halves the panel bytes they pull into L2
        const int ntm = Mt.mp / BT, ntn = Mt.np / BT;
        if (ntn % 8 == 0) {
            const int band = tile / (ntm * 8), w = tile % (ntm * 8);
            tm = w / 8;
            tn = band * 8 + w % 8;
        } else {
            tm = tile / ntn;
            tn = tile % ntn;
        }
    } else {
        C = Mt.W[ops.c];
        if (EPI == EPI_GRAM) { A = y_sel ? Mt.Y2 : Mt.Y; B = A; K = Mt.np; lda = ldb = Mt.np; ldc = Mt.mp; }
        else { A = Mt.W[ops.a]; B = Mt.W[ops.b]; K = Mt.mp; lda = ldb = ldc = Mt.mp; }
        CT = C; ldct = ldc;
        const int nt = Mt.mp / BT;      // upper-triangular enumeration: row tm holds nt - tm tiles
        tm = 0;
        while (tile >= nt - tm) { tile -= nt - tm; tm++; }
        tn = tm + tile;
    }
    A += (size_t)tm * BT * lda;
    B += BKN ? (size_t)tn * BT : (size_t)tn * BT * ldb;

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    // Global memory -> LDS without passing through registers (global_load_lds_dwordx4: the 64 lanes' 16-byte chunks land
    // contiguously, 1 KB per instruction, at the wave-uniform LDS address in M0).  K tiles of 32, four stages of
    // {A tile, B tile} (16 KB each): the loads of a tile are issued three tiles ahead of its use and nothing of the
    // copy occupies the wave's registers or its LDS-write slots.  A 1 KB block cannot carry padding, so the tiles are
    // swizzled instead, by the choice of the chunk each lane fetches:
    //   [256 rows x 32 k] tile (K-contiguous operand): block = 16 rows x 4 chunks, chunk c of row r at position
    //                          c ^ ((r >> 2) & 3) of its row: 16 consecutive rows read one k chunk without a bank conflict
    //   [32 k x 256 n] tile (the apply step's B): block = 2 k rows x 32 chunks, the 64-byte group g of row k at
    //                          g ^ sw(k), sw(k) = (k & 3) | ((k >> 1) & 4): the 8 rows one transposing read touches
    //                          (k0..k0+3 and k0+8..k0+11) fall on 8 different groups
    constexpr int BKD = 32, STAGES = 4;
    constexpr int OP_BYTES = BT * BKD * 2, STAGE_BYTES = 2 * OP_BYTES;
    static_assert(STAGES * STAGE_BYTES <= GEMM_LDS_BYTES, "four stages fit the GEMM's LDS");
    const unsigned char* const lds = reinterpret_cast<const unsigned char*>(smem);
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)smem;     // LDS byte address of smem
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    // address = wave-uniform 64-bit base (scalar registers, advanced by scalar adds) + this lane's constant 32-bit offset
    auto dma16 = [](uint32_t lane_off, const void* base, uint32_t lds_addr) {
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n" : : "v"(lane_off), "s"(base), "s"(lds_addr) : "memory");
    };
    // this lane's share of a block: row lane/4 of the block's 16 (block 4i + w of the tile), chunk (lane%4) ^ ((lane/16)%4)
    // (block GWAVES*i + w of the tile for this wave's i-th load)
    const uint32_t lo_a = (uint32_t)((((lane >> 2) + 16 * wv) * lda + (((lane & 3) ^ ((lane >> 4) & 3)) * 8)) * 2);
    const uint32_t lo_b = (uint32_t)((((lane >> 2) + 16 * wv) * ldb + (((lane & 3) ^ ((lane >> 4) & 3)) * 8)) * 2);
    // [k][n] tile: wave w's i-th load fetches k rows 2(GWAVES*i + w) + lane/32; sw of a row k is (k & 3) | ((k >> 1) & 4)
    const int kn_row = 2 * wv + (lane >> 5);
    const int kn_c0 = (lane & 31) ^ ((((kn_row & 3) | ((kn_row >> 1) & 4)) & 7) << 2);
    const uint32_t lo_kn0 = (uint32_t)((kn_row * ldb + kn_c0 * 8) * 2);            // rows whose bit 3 is that of 2w + lane/32
    const uint32_t lo_kn1 = (uint32_t)((kn_row * ldb + (kn_c0 ^ 16) * 8) * 2);     // ... the other value (four waves: odd i)
    // the q-th of a tile's 2*LPT loads (first the A tile's, then the B tile's)
    auto dma_one = [&](int kt, int q) {
        const uint32_t st = lds0 + (uint32_t)(kt & (STAGES - 1)) * STAGE_BYTES;
        const int i = q % LPT, blk = GWAVES * i + wv;
        if (q < LPT) dma16(lo_a, reinterpret_cast<const char*>(A) + ((size_t)i * 16 * GWAVES * lda + (size_t)kt * BKD) * 2, st + blk * 1024);
        else if (BKN) dma16(((2 * GWAVES * i) & 8) ? lo_kn1 : lo_kn0, reinterpret_cast<const char*>(B) + (size_t)(kt * BKD + 2 * GWAVES * i) * ldb * 2, st + OP_BYTES + blk * 1024);
        else dma16(lo_b, reinterpret_cast<const char*>(B) + ((size_t)i * 16 * GWAVES * ldb + (size_t)kt * BKD) * 2, st + OP_BYTES + blk * 1024);
    };
    auto dma_tile = [&](int kt) {
#pragma unroll
        for (int q = 0; q < 2 * LPT; q++) dma_one(kt, q);
    };
    // operand fetches.  K-contiguous tile: lane = row lane%32 of a 32-row MFMA block, k chunk 2kk + lane/32
    const int ra0 = wm * (BT / 2) + (lane & 31), rb0 = wn * WCOLS + (lane & 31);
    const int a_rd0 = (ra0 >> 4) * 1024 + (ra0 & 15) * 64 + (((lane >> 5) ^ ((ra0 >> 2) & 3)) * 16);                 // kk = 0; kk = 1 is this ^ 32
    const int b_rd0 = OP_BYTES + (rb0 >> 4) * 1024 + (rb0 & 15) * 64 + (((lane >> 5) ^ ((rb0 >> 2) & 3)) * 16);
    // [k][n] tile, transposing read (ds_read_b64_tr_b16: within a 16-lane group, lane i receives as element e element i%4 of
    // the 8 bytes that lane 4e + i/4 addressed; groups 0/1 cover columns 0-15 / 16-31 of a 32-column MFMA block, groups 2/3
    // the same columns of the next 8 k): lane -> k row 8(lane/32) + (lane%16)/4,
    // columns 16((lane/16)%2) + 4(lane%4) of the 32-column MFMA block j of this wave; the block's 64-byte group is wn*4 + j
    const int kn_q2 = (lane & 15) >> 2, kn_h = lane >> 5;
    const int kn_rd0 = OP_BYTES + (8 * kn_h + kn_q2) * 512 + 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
    const int kn_sw = kn_q2 | (kn_h << 2);
    constexpr int NREADS = TM + TN * (BKN ? 2 : 1);     // LDS reads of a k step's operands
    bf16x8 av[2][TM], bv[2][TN];
    auto lds_load = [&](int stage, int kk, int s) {
        const unsigned char* base = lds + stage * STAGE_BYTES;
#pragma unroll
        for (int i = 0; i < TM; i++) av[s][i] = *reinterpret_cast<const bf16x8*>(base + ((a_rd0 ^ (kk * 32)) + i * 2048));
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if (BKN) {
                const unsigned char* q = base + kn_rd0 + (((wn * TN + j) ^ kn_sw) << 6) + kk * 16 * 512;
                const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_p)(q));
                const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_p)(q + 4 * 512));
                typedef short i16x8 __attribute__((ext_vector_type(8)));
                const i16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                bv[s][j] = __builtin_bit_cast(bf16x8, both);
            } else {
                bv[s][j] = *reinterpret_cast<const bf16x8*>(base + ((b_rd0 ^ (kk * 32)) + j * 2048));
            }
        }
    };
    auto mma = [&](int s) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = mfma<IN>(av[s][i], bv[s][j], acc[i][j]);
    };

    const int nk = K / BKD;      // a multiple of 8: K is a multiple of 256
    const bf16_t* aux = EPI == EPI_POLY ? Mt.W[ops.a] : nullptr;
    const int gcol0 = tn * BT + wn * WCOLS;
    // the auxiliary operand of the polynomial's epilogue (G):
    // 16 bytes per lane and 8-column chunk of a 32-row block of this wave's tile.  The first two blocks are requested during
    // the last K tile, each later one while the block two before it is
    // being written, so that the epilogue does not wait for memory
    u32x4 ax[2][WCOLS / 16];
    auto aux_load = [&](int i) {
#pragma unroll
        for (int c = 0; c < WCOLS / 16; c++) {
            const int id = lane + 64 * c, row = id / (WCOLS / 8), c8 = id % (WCOLS / 8);
            ax[i & 1][c] = *(gvec_p)(aux + (size_t)(tm * BT + wm * (BT / 2) + i * 32 + row) * ldc + gcol0 + c8 * 8);
        }
    };
    // wait until at most n of this wave's loads are outstanding (vmcnt only; the other counters unconstrained)
#define SG_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | (((n) >> 4) << 14))
    dma_tile(0); dma_tile(1); dma_tile(2); dma_tile(3);
    SG_WAIT_VM(6 * LPT);
    __syncthreads();
    lds_load(0, 0, 0);
    // A K tile is two phases of 16 MFMAs.  Phase 0 multiplies k step 0 while the operands of k step 1 are read; then
    // the wave makes sure the next tile has landed (its loads were issued three tiles ago: only the two tiles after it
    // may still be in flight) and that its own reads of this stage are done, the workgroup meets, and the stage is
    // handed to the loads of the tile four ahead; phase 1 multiplies k step 1 while the first operands of the next
    // tile are read.
    // Phase 1 is written out as eight pairs of MFMAs, each followed by one load of the tile four ahead and one operand
    // read of the next tile: a burst of memory instructions would leave the matrix pipe idle while it issues.
    auto ktile = [&](int kt, auto dma_c, auto wait_c, auto next_c) {
        constexpr bool DMA = decltype(dma_c)::value != 0, NEXT = decltype(next_c)::value != 0;
        constexpr int WAIT = decltype(wait_c)::value;      // loads that may stay in flight once the next tile has landed
        const int stage = kt & (STAGES - 1), nstage = (kt + 1) & (STAGES - 1);
        __builtin_amdgcn_sched_barrier(0);
        lds_load(stage, 1, 1);
        mma(0);
        SG_MUON_SCHED_READS(NREADS, TM * TN);
        __builtin_amdgcn_sched_barrier(0);
        if (NEXT) SG_WAIT_VM(WAIT);
        __builtin_amdgcn_s_waitcnt(0xC07F);     // lgkmcnt(0): this wave's reads of the stage have returned
        __syncthreads();
        if (!NEXT && EPI == EPI_POLY) { aux_load(0); aux_load(1); }
        const unsigned char* nbase = lds + nstage * STAGE_BYTES;
        constexpr int MPG = TM * TN / 8;        // MFMAs per group
#pragma unroll
        for (int g = 0; g < 8; g++) {
            // operand reads of the next tile's k step 0: one fragment per group
            if (NEXT) {
                if (g < TM) av[0][g] = *reinterpret_cast<const bf16x8*>(nbase + a_rd0 + g * 2048);
                else if (g - TM >= TN) {}
                else if (!BKN) bv[0][g - TM] = *reinterpret_cast<const bf16x8*>(nbase + b_rd0 + (g - TM) * 2048);
                else {
                    const unsigned char* q = nbase + kn_rd0 + (((wn * TN + (g - TM)) ^ kn_sw) << 6);
                    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_p)(q));
                    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_p)(q + 4 * 512));
                    bv[0][g - TM] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                }
            }
#pragma unroll
            for (int m = MPG * g; m < MPG * (g + 1); m++)
                acc[m / TN][m % TN] = mfma<IN>(av[1][m / TN], bv[1][m % TN], acc[m / TN][m % TN]);
            __builtin_amdgcn_sched_barrier(0);
            if (DMA && g < 2 * LPT) dma_one(kt + 4, g);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using c0 = std::integral_constant<int, 0>;
    using c1 = std::integral_constant<int, 1>;
    int kt = 0;
    for (; kt + 4 < nk; kt++) ktile(kt, c1{}, std::integral_constant<int, 4 * LPT>{}, c1{});     // steady state
    ktile(kt, c0{}, std::integral_constant<int, 4 * LPT>{}, c1{});      // tiles nk-2 and nk-1 may still be in flight
    ktile(kt + 1, c0{}, std::integral_constant<int, 2 * LPT>{}, c1{});
    ktile(kt + 2, c0{}, std::integral_constant<int, 0>{}, c1{});
    ktile(kt + 3, c0{}, std::integral_constant<int, 0>{}, c0{});
#undef SG_WAIT_VM
    __syncthreads();        // the epilogue reuses the LDS stages: every wave is done reading them

    // ---- epilogue, staged through LDS (free after the last barrier) so that global memory sees
    // 16-byte accesses along rows.  Accumulator element e of MFMA tile (i,j) is
    // row 8*(e/4) + 4*(lane/32) + e%4, column lane%32.  One 32-row block of the wave's
    // tile at a time: fp32 block -> LDS, read back as 8-column chunks, combine with the auxiliary
    // operand, round to bf16 and store.  Off-diagonal tiles of the symmetric products also store
    // the transposed block: the rounded values go back into the staged block and are read down
    // its columns.  Every wave stages in its own LDS region and LDS executes a wave's
    // instructions in order, so no workgroup barrier is needed, only the compiler kept from
    // reordering (wave_barrier).
    constexpr int EP_ROW = WCOLS + 4;     // floats per staged row
    constexpr int RCH = WCOLS / 8;        // 8-column chunks per row
    constexpr int NC = 32 * RCH / 64;     // chunks per lane and 32-row block
    static_assert(GWAVES * 32 * EP_ROW * 4 <= GEMM_LDS_BYTES, "epilogue staging exceeds the GEMM's LDS");
    float* ep = reinterpret_cast<float*>(smem) + wave * (32 * EP_ROW);
    // uniform over the workgroup
    const bool mirror = EPI != EPI_APPLY && tm != tn;
    // first iteration: Y is the unnormalised momentum, so its Gram matrix carries 1/norm^2 and the applied Y 1/norm
    const float inv = Bt.inv_norm[mi];
    const bool diag_wave = EPI == EPI_POLY && tm == tn && wn / (GWN / 2) == wm;     // this wave's block meets the diagonal
    const bool first = (EPI == EPI_GRAM || EPI == EPI_APPLY) && (iter_flags & 2) != 0;       // (only they read Y)
    constexpr float factor = epi_factor<EPI, IN, OUT>();
    const float scale = first ? (EPI == EPI_GRAM ? inv * inv : inv) * factor : factor;
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int grow0 = tm * BT + wm * (BT / 2) + i * 32;
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int e = 0; e < 16; e++)
                ep[(8 * (e >> 2) + 4 * (lane >> 5) + (e & 3)) * EP_ROW + 32 * j + (lane & 31)] = acc[i][j][e];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int id = lane + 64 * c, row = id / RCH, c8 = id % RCH;
            f32x4* src = reinterpret_cast<f32x4*>(&ep[row * EP_ROW + c8 * 8]);
            const f32x4 lo = src[0], hi = src[1];
            float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            if (EPI == EPI_POLY) {
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    v[k] = polynomial<IN>(v[k], widen<IN>(ax[i & 1][c][k >> 1], k));
                }
                if (diag_wave) {        // H + a I: the apply step is then the single product (H + a I) Y
                    const int dk = (wm * (BT / 2) + i * 32 + row) - (wn * WCOLS + c8 * 8);
#pragma unroll
                    for (int k = 0; k < 8; k++) v[k] += (dk == k) ? diagonal<IN>() : 0.0f;
                }
            }
            if (EPI != EPI_POLY && (first || factor != 1.0f)) {      // uniform over the grid
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] *= scale;
            }
            u32x4 out;
#pragma unroll
            for (int k = 0; k < 4; k++) out[k] = round2<OUT>(v[2 * k], v[2 * k + 1]);
            *(gvec_w)(C + (size_t)(grow0 + row) * ldc + gcol0 + c8 * 8) = out;
            if (mirror) {   // rounded values (as bit patterns) back into the staged block
                u32x4 b0 = {out[0] & 0xffffu, out[0] >> 16, out[1] & 0xffffu, out[1] >> 16};
                u32x4 b1 = {out[2] & 0xffffu, out[2] >> 16, out[3] & 0xffffu, out[3] >> 16};
                reinterpret_cast<u32x4*>(src)[0] = b0;
                reinterpret_cast<u32x4*>(src)[1] = b1;
            }
        }
        if (EPI == EPI_POLY && i + 2 < TM) aux_load(i + 2);
        __builtin_amdgcn_wave_barrier();
        if (mirror) {
            const uint32_t* epb = reinterpret_cast<const uint32_t*>(ep);
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const int id = lane + 64 * c, col = id >> 2, r8 = id & 3;
                u32x4 t;
#pragma unroll
                for (int k = 0; k < 4; k++)
                    t[k] = epb[(r8 * 8 + 2 * k) * EP_ROW + col] | (epb[(r8 * 8 + 2 * k + 1) * EP_ROW + col] << 16);
                *(gvec_w)(CT + (size_t)(gcol0 + col) * ldct + grow0 + r8 * 8) = t;
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// ---- the same products on 64x64 output tiles, for calls whose 256x256 tiles leave most of the chip idle
// Four waves share a tile by splitting K: chunk c of 32 k goes to wave c % 4, which multiplies the whole tile and stages
// its operands in LDS of its own, one chunk ahead; the four partial tiles are added up through LDS.  So there is no barrier
// in the K loop and a chain of a quarter of K, and two workgroups fit a CU (one's epilogue under the other's products: eight
// waves on a tile were 0 to 5 % faster for calls of few tiles and 10 to 40 % slower for the rest; operands straight from
// memory into registers, 16 bytes a row, took up to twice as long).
// The apply step reads the transpose T of Y, which its own epilogue (and the momentum kernel) leaves beside Y: with it all
// three products have both operands K-contiguous.
// Bound by latency for few tiles (the operands come through memory, where other XCDs wrote them: 5 to 8 us a product, of
// which 4 are the launch), for many by what a CU gets from L2 (32 flop per byte: 0.6 PFLOP/s).
// Step over bf16 matrices, with k_gemm_nt alone and with choose_tiles between the two: 1 of 200 x 800 235 -> 116 us,
// 24 of 64 x 3000 368 -> 148, 1 of 1024 x 1024 413 -> 155, 2 of 1024 x 4096 621 -> 323, 24 of 512 x 2048 558 -> 457.
constexpr int NT64 = 64;
constexpr int KS_WAVES = 4, KS_THREADS = 64 * KS_WAVES;
constexpr int KS_ROW = NT64 + 4;                                                // floats per row of a partial tile
constexpr int KS_LDS_BYTES = KS_WAVES * NT64 * KS_ROW * 4;                      // 69,632 bytes
constexpr int KS_STAGE = 2 * NT64 * 32 * 2, KS_WAVE = 2 * KS_STAGE;             // two stages of 8 KB per wave
static_assert(KS_WAVES * KS_WAVE <= KS_LDS_BYTES, "the waves' stages fit where their partial tiles go");

// y_sel: as for k_gemm_nt; iter_flags: bit 1 = first iteration, bit 2 = last (no product reads T any more)
template <int EPI, int IN, int OUT>
__global__ __launch_bounds__(KS_THREADS) void k_gemm_64(Batch Bt, Ops ops, int y_sel, int iter_flags) {
    constexpr int W = KS_WAVES;
    extern __shared__ __attribute__((aligned(16))) float part[];
    __shared__ double sm[W];
    const int nblk = gridDim.x;
    int lb = blockIdx.x;
    if (nblk % 8 == 0) lb = (blockIdx.x % 8) * (nblk / 8) + blockIdx.x / 8;      // XCD-contiguous, as in k_gemm_nt
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const sg::cint_p prefix = sg::as_const(Bt.gtile_prefix[shape_of(EPI)]);
    if (EPI == EPI_MUL && ops.c2 >= 0 && lb >= nblk / 2) { lb -= nblk / 2; ops.a = ops.a2; ops.b = ops.b2; ops.c = ops.c2; }
    const int mi = sg::upper_seg(prefix, Bt.P, lb);
    const Mat& Mt = Bt.mats[mi];
    int tile = lb - prefix[mi];
    const bool first = (iter_flags & 2) != 0, last = (iter_flags & 4) != 0;      // uniform over the grid

    const bf16_t *A, *B;
    bf16_t *C, *CT;         // CT: where the transposed tile goes (NULL: nowhere)
    int K, ldc, ldct, tm, tn;
    if (EPI == EPI_APPLY) {
        A = Mt.W[ops.a]; B = y_sel ? Mt.T2 : Mt.T; C = y_sel ? Mt.Y : Mt.Y2; K = Mt.mp; ldc = Mt.np;
        CT = last ? nullptr : (y_sel ? Mt.T : Mt.T2); ldct = Mt.mp;
        const int ntm = Mt.mp / NT64;
        tm = tile % ntm;
        tn = tile / ntm;
    } else {
        C = Mt.W[ops.c];
        if (EPI == EPI_GRAM) { A = B = y_sel ? Mt.Y2 : Mt.Y; K = Mt.np; }
        else { A = Mt.W[ops.a]; B = Mt.W[ops.b]; K = Mt.mp; }
        ldc = ldct = Mt.mp;
        const int nt = Mt.mp / NT64;
        tm = 0;
        while (tile >= nt - tm) { tile -= nt - tm; tm++; }
        tn = tm + tile;
        CT = tm != tn ? C : nullptr;
    }
    const int r32 = lane & 31, kh = lane >> 5;
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;
    // a wave's stage: {A, B} rows of 32 k, in blocks of 16 rows with the swizzle of k_gemm_nt's [256 x 32 k] tiles
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) float*)part + (uint32_t)wave * KS_WAVE;
    const unsigned char* const mine = reinterpret_cast<const unsigned char*>(part) + wave * KS_WAVE;
    const uint32_t lane_off = (uint32_t)(((lane >> 2) * K + (((lane & 3) ^ ((lane >> 4) & 3)) * 8)) * 2);
    const char* const pa = reinterpret_cast<const char*>(A + (size_t)tm * NT64 * K);            // every operand's row stride is K
    const char* const pb = reinterpret_cast<const char*>(B + (size_t)tn * NT64 * K);
    auto fetch = [&](int s, int c) {
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const char* base = (q < 4 ? pa : pb) + ((size_t)(q & 3) * 16 * K + (size_t)c * 32) * 2;
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n"
                         : : "v"(lane_off), "s"(base), "s"(lds0 + (uint32_t)(s * KS_STAGE + q * 1024)) : "memory");
        }
    };
    // (the operands change places, so that a lane holds, of its row of the result, four times four consecutive columns)
    auto multiply = [&](int s, auto refill) {
        bf16x8 a[2][2], b[2][2];
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int r = 32 * i + r32, at = s * KS_STAGE + (r >> 4) * 1024 + (r & 15) * 64 + (((2 * u + kh) ^ ((r >> 2) & 3)) * 16);
                a[u][i] = *reinterpret_cast<const bf16x8*>(mine + at);
                b[u][i] = *reinterpret_cast<const bf16x8*>(mine + at + 4096);
            }
        refill();
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = mfma<IN>(b[u][j], a[u][i], acc[i][j]);
    };
    const int nk = K / 32;
    int c = wave, s = 0;
    if (c < nk) {
        fetch(0, c);
        if (c + W < nk) fetch(1, c + W);
#pragma unroll 1
        for (; c + W < nk; c += W) {
            asm volatile("s_waitcnt vmcnt(8)" ::: "memory");            // this chunk has landed, the next may be on its way
            multiply(s, [&] {
                if (c + 2 * W < nk) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage has been read
                    fetch(s, c + 2 * W);
                }
            });
            s ^= 1;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        multiply(s, [] {});
    }
    __syncthreads();                                            // the partial tiles overlay the stages
    constexpr int NR = 8 / W;                                   // eight elements each in this many rows of the tile per thread
    const int row0 = tid >> 3, c8 = tid & 7;
    u32x4 g[NR];
    if (EPI == EPI_POLY) {
#pragma unroll
        for (int h = 0; h < NR; h++) g[h] = *(gvec_p)(A + (size_t)(tm * NT64 + row0 + 8 * W * h) * ldc + tn * NT64 + 8 * c8);
    }
    // first iteration: Y is the unnormalised momentum, see k_momentum; the norm is added up from its tiles here
    constexpr float factor = epi_factor<EPI, IN, OUT>();
    float scale = factor;
    if ((EPI == EPI_GRAM || EPI == EPI_APPLY) && first) {
        double sq = 0.0;
        for (int k = Bt.ttile_prefix[mi] + tid; k < Bt.ttile_prefix[mi + 1]; k += 64 * W) sq += Bt.partials[k];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) sq += __shfl_down(sq, d, 64);
        if (lane == 0) sm[wave] = sq;
    }
    const int waves = min(nk, W);                               // those that have a partial tile
    if (wave < waves) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    *reinterpret_cast<f32x4*>(part + (wave * NT64 + 32 * i + r32) * KS_ROW + 32 * j + 8 * q + 4 * kh) =
                        f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    }
    __syncthreads();
    if ((EPI == EPI_GRAM || EPI == EPI_APPLY) && first) {
        const double tot = (sm[0] + sm[1]) + (sm[2] + sm[3]);
        const float inv = 1.0f / ((float)sqrt(tot) + 1e-7f);
        scale = (EPI == EPI_GRAM ? inv * inv : inv) * factor;
    }
    u32x4 out[NR];
#pragma unroll
    for (int h = 0; h < NR; h++) {
        const int row = row0 + 8 * W * h;
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = 0.0f;
        for (int w = 0; w < waves; w++) {
            const f32x4* src = reinterpret_cast<const f32x4*>(part + (w * NT64 + row) * KS_ROW + 8 * c8);
            const f32x4 lo = src[0], hi = src[1];
#pragma unroll
            for (int k = 0; k < 4; k++) { v[k] += lo[k]; v[4 + k] += hi[k]; }
        }
        if (EPI == EPI_POLY) {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                v[k] = polynomial<IN>(v[k], widen<IN>(g[h][k >> 1], k)) + (tm == tn && row == 8 * c8 + k ? diagonal<IN>() : 0.0f);
            }
        } else if (first || factor != 1.0f) {
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] *= scale;
        }
#pragma unroll
        for (int k = 0; k < 4; k++) out[h][k] = round2<OUT>(v[2 * k], v[2 * k + 1]);
        *(gvec_w)(C + (size_t)(tm * NT64 + row) * ldc + tn * NT64 + 8 * c8) = out[h];
    }
    if (CT) {       // uniform over the workgroup
        constexpr int TR = NT64 + 8;
        bf16_t* t = reinterpret_cast<bf16_t*>(part);
        __syncthreads();                                        // the partial tiles have been read
#pragma unroll
        for (int h = 0; h < NR; h++) *reinterpret_cast<u32x4*>(t + (row0 + 8 * W * h) * TR + 8 * c8) = out[h];
        __syncthreads();
#pragma unroll
        for (int h = 0; h < NR; h++) {
            const int row = row0 + 8 * W * h;
            u32x4 o;
#pragma unroll
            for (int k = 0; k < 4; k++) o[k] = (uint32_t)t[(8 * c8 + 2 * k) * TR + row] | ((uint32_t)t[(8 * c8 + 2 * k + 1) * TR + row] << 16);
            *(gvec_w)(CT + (size_t)(tn * NT64 + row) * ldct + tm * NT64 + 8 * c8) = o;
        }
    }
}

// ---- all iterations of one matrix in one workgroup: Y [mp x np] (mp 64 or 128) and G, then H in its place, stay in LDS.
// Eight waves.  G and G G: 32x32 tiles, those left of the diagonal mirrored; apply: strips of 32 columns, whose Y' replaces
// their Y (a strip is read by its own wave only).  Same roundings as the GEMM path: G, H and Y are bf16 between the
// products, the first step carries 1/norm^2 and 1/norm.
// Rows lie 16-byte chunk by chunk, chunk c of row r at c ^ ns_swizzle(r): a quarter wave's 16-byte reads of a chunk of
// consecutive rows and the transposing reads of four rows of four chunks both meet every bank once (with the row's low bits
// as they are, the transposing read took 8 cycles instead of 2.5).
// One CU per matrix.  Of an iteration of 128 x 512, the largest, about 15 400 cycles: matrix cores 7900, and the ends of
// three dependent products (operands on their way, conversion, LDS writes at 64 bytes a cycle, a barrier each).
// 41 us for five; 50 before the products' operand addresses were kept in registers, the reads dealt between the matrix
// instructions and half of the symmetric products left out; 180 as fifteen launches of k_gemm_nt.
constexpr int NS_THREADS = 512;
constexpr int NS_Y_ELEMS = 128 * 512;          // Y: 128 KB ...
constexpr int NS_LDS_BYTES = 2 * (NS_Y_ELEMS + 128 * 128);      // ... and G: 32 KB, all of a CU's 160 KB
inline bool fits_lds(int mp, int np) { return mp <= 128 && mp * np <= NS_Y_ELEMS; }
// of a row, its low bits dealt to the bits of a chunk's place; linear over exclusive or
__device__ __forceinline__ constexpr int ns_swizzle(int row, bool odd) { return odd ? ((row & 2) << 1) | ((row >> 2) & 3) : ((row & 3) << 2) | ((row >> 2) & 3); }

template <int MT>       // mp / 32
__device__ __forceinline__ void newton_schulz(const Mat& M, float inv, int steps, bf16_t* __restrict__ smem) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) unsigned char* lds_t;
    typedef __attribute__((address_space(3))) bf16x8* lds_op;
    typedef __attribute__((address_space(3))) u32x4* lds_vec;
    typedef __attribute__((address_space(3))) bf16_t* lds_b16;
    constexpr int mp = 32 * MT, WAVES = NS_THREADS / 64, GROW = 2 * mp;
    const int np = M.np, row = 2 * np, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool odd = np & 64;
    const lds_t Y = (lds_t)smem, G = Y + mp * row;
    // sixteen bytes of every chunk in order, a batch of them on their way at once (few for a small matrix: 54 x 112 has two a lane)
    const int chunks = np / 8, dr = NS_THREADS / chunks, dc = NS_THREADS % chunks;
    const bool few = mp * chunks <= 4 * NS_THREADS;
    auto stream = [&](auto batch, auto move) {
        constexpr int BATCH = decltype(batch)::value;
        int r = tid / chunks, c = tid % chunks;
        for (int i = tid; i < mp * chunks; i += BATCH * NS_THREADS) {
            int at[BATCH];
#pragma unroll
            for (int u = 0; u < BATCH; u++) {
                at[u] = r * row + ((c ^ ns_swizzle(r, odd)) << 4);
                r += dr;
                c += dc;
                if (c >= chunks) { c -= chunks; r++; }
            }
            move(i, at, min(BATCH, (mp * chunks - i + NS_THREADS - 1) / NS_THREADS));
        }
    };
    {
        const u32x4* __restrict__ src = reinterpret_cast<const u32x4*>(M.Y);
        auto load = [&](int i, const auto& at, int n) {
            constexpr int BATCH = std::extent_v<std::remove_reference_t<decltype(at)>>;
            u32x4 v[BATCH];
#pragma unroll
            for (int u = 0; u < BATCH; u++) if (u < n) v[u] = *(gvec_p)(src + i + u * NS_THREADS);
#pragma unroll
            for (int u = 0; u < BATCH; u++) if (u < n) *(lds_vec)(Y + at[u]) = v[u];
        };
        if (few) stream(std::integral_constant<int, 4>{}, load);
        else stream(std::integral_constant<int, 16>{}, load);
    }
    __syncthreads();
    // S S^T is symmetric: the tiles on and right of the diagonal, dealt so that the waves of a SIMD (w and w + 4) have at most
    // three; each reads the rows of its row of tiles rt and, with a tile off the diagonal, those of ct.  (Of two rows of tiles all
    // four are formed, a wave each: mirroring is longer than the product there.)
    const bool on = MT == 4 ? wave < 2 || wave == 4 || wave == 5 : wave < 2, off = MT == 4 ? wave != 4 && wave != 5 : wave == 2 || wave == 3;
    const int rt = MT == 4 ? (wave < 2 ? 2 * wave : wave == 4 ? 1 : wave == 5 ? 3 : wave & 1) : wave & 1;
    const int ct = MT == 4 ? (wave < 2 ? 2 * wave + 1 : wave < 4 ? 2 : 3) : 1 - rt;
#pragma unroll 1
    for (int it = 0; it < steps; it++) {
        int ln = lane;                       // keeps the address arithmetic in its phase: hoisted out of the loop it spills
        asm volatile("" : "+v"(ln));
        const int r32 = ln & 31, kh = ln >> 5;
        // a tile's 32 columns of a row, four of every eight in this lane (4 kh ..) and four in the lane 32 away: two exchanges give
        // each lane a whole chunk
        auto put_row = [&](lds_t at, u32x2 v, u32x2 w) {
            const auto x = __builtin_amdgcn_permlane32_swap(v[0], w[0], false, false);
            const auto y = __builtin_amdgcn_permlane32_swap(v[1], w[1], false, false);
            *(lds_vec)at = u32x4{x[0], y[0], x[1], y[1]};
        };
        f32x16 acc[2];                       // of the tile on the diagonal and of the one off it
        u32x2 g[2][4];                       // the same as bf16: four times four consecutive columns of a lane's row
        // the wave's tiles of S S^T, S [mp x width], in steps of 16 columns: four at a time, the next four on their way
        auto gram = [&](auto diag, auto side, lds_t s, int width, bool wodd) {
            constexpr bool D = decltype(diag)::value, O = decltype(side)::value;
            const int nk = width / 16;       // a multiple of four
            const int sw = ns_swizzle(r32, wodd) ^ kh, to_b = 64 * (ct - rt) * width;
            lds_t at[2][4];                  // of an even and an odd four: eight chunks on is a flipped bit or, with odd rows, 128 bytes
#pragma unroll
            for (int u = 0; u < 4; u++) {
                at[0][u] = s + (32 * rt + r32) * 2 * width + ((sw ^ (2 * u)) << 4);
                at[1][u] = s + (32 * rt + r32) * 2 * width + (wodd ? ((sw ^ (2 * u)) << 4) + 128 : (sw ^ (2 * u) ^ 8) << 4);
            }
            bf16x8 a[2][4], b[2][4];
            auto fetch = [&](auto set, int k) {          // k: of the even four
                constexpr int S = decltype(set)::value;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const lds_t p = at[S][u] + 32 * k;
                    a[S][u] = *(lds_op)p;
                    if (O) b[S][u] = *(lds_op)(p + to_b);
                }
            };
            auto multiply = [&](auto set) {
                constexpr int S = decltype(set)::value;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    if (D) acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[S][u], a[S][u], acc[0], 0, 0, 0);
                    if (O) acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[S][u], a[S][u], acc[1], 0, 0, 0);
                }
                // the reads between the products
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, O ? 2 : 1, 0);
                }
                if (D && O) __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            using Z0 = std::integral_constant<int, 0>;
            using Z1 = std::integral_constant<int, 1>;
            fetch(Z0{}, 0);
#pragma unroll 1
            for (int k = 0; k + 8 <= nk; k += 8) {       // (without branches around the reads: they would be waited for at once)
                fetch(Z1{}, k);
                multiply(Z0{});
                fetch(Z0{}, k + 8 < nk ? k + 8 : k);     // (after the last an operand that nobody uses)
                multiply(Z1{});
            }
            if (nk & 4) multiply(Z0{});
        };
        // a tile and, off the diagonal, its mirror image
        auto put = [&](auto side) {
            constexpr int J = decltype(side)::value;
            const int col = J ? ct : rt, sw = ns_swizzle(r32, mp & 64) ^ kh;
            const lds_t at = G + (32 * rt + r32) * GROW;
#pragma unroll
            for (int q = 0; q < 4; q += 2) put_row(at + ((sw ^ (4 * col + q)) << 4), g[J][q], g[J][q + 1]);
            if (J && MT == 4) {
                const lds_t mirror = G + (32 * col + 4 * kh) * GROW + 2 * (r32 & 7);
                const int place = (4 * rt + (r32 >> 3)) ^ ns_swizzle(4 * kh, mp & 64);
#pragma unroll
                for (int q = 0; q < 4; q++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        *(lds_b16)(mirror + ((place ^ ns_swizzle((8 * q + e) & 15, mp & 64)) << 4) + (8 * q + e) * GROW) = (bf16_t)(g[J][q][e >> 1] >> (16 * (e & 1)));
            }
        };
        using T = std::true_type;
        using F = std::false_type;
#pragma unroll 1
        for (int phase = 0; phase < 2; phase++) {
            const lds_t s = phase ? G : Y;               // G is symmetric
            const int width = phase ? mp : np;
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[j][e] = 0.0f;
            if (on && off) gram(T{}, T{}, s, width, width & 64);
            else if (on) gram(T{}, F{}, s, width, width & 64);
            else if (off) gram(F{}, T{}, s, width, width & 64);
            if (phase == 0) {
                const float scale = it == 0 ? inv * inv : 1.0f;
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    if (j ? !off : !on) continue;
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        g[j][q] = u32x2{bf16r2(acc[j][4 * q] * scale, acc[j][4 * q + 1] * scale), bf16r2(acc[j][4 * q + 2] * scale, acc[j][4 * q + 3] * scale)};
                }
            } else {                                     // H = a I + b G + c G G in place of G
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    if (j ? !off : !on) continue;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const u32x2 w = g[j][q];
                        float v[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const float x = sg_i2f((int32_t)((e & 1) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16)));
                            v[e] = sg_fma(NS_C, acc[j][4 * q + e], NS_B * x) + (j == 0 && r32 == 8 * q + 4 * kh + e ? NS_A : 0.0f);
                        }
                        g[j][q] = u32x2{bf16r2(v[0], v[1]), bf16r2(v[2], v[3])};
                    }
                }
                __syncthreads();
            }
            if (on) put(std::integral_constant<int, 0>{});
            if (off) put(std::integral_constant<int, 1>{});
            __syncthreads();
        }
        // Y' = H Y by strips of 32 columns
        for (int strip = wave; strip < np / 32; strip += WAVES) {
            f32x16 y[MT];
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int e = 0; e < 16; e++) y[i][e] = 0.0f;
            // transposing read (see k_gemm_nt): lane -> k row 8 (lane / 32) + (lane % 16) / 4, columns 16 ((lane / 16) % 2) + 4 (lane % 4)
            const int c0 = 4 * strip + 2 * ((ln >> 4) & 1) + ((ln & 3) >> 1), k0 = 8 * kh + ((ln & 15) >> 2);
            const lds_t t0 = Y + k0 * row + ((c0 ^ ns_swizzle(k0, odd)) << 4) + 8 * (ln & 1);
            const lds_t t4 = Y + (k0 + 4) * row + ((c0 ^ ns_swizzle(k0 + 4, odd)) << 4) + 8 * (ln & 1);
            const int hat = (ns_swizzle(r32, mp & 64) ^ kh) << 4;
            const lds_t hr = G + r32 * GROW;
            bf16x8 b[2], h[2][MT];
            auto fetch = [&](int k) {
                const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_p)(t0 + 16 * k * row));
                const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_p)(t4 + 16 * k * row));
                b[k & 1] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
                for (int i = 0; i < MT; i++) h[k & 1][i] = *(lds_op)(hr + (hat ^ (32 * k)) + 32 * i * GROW);
            };
            fetch(0);
#pragma unroll
            for (int k = 0; k < mp / 16; k++) {
                if (k + 1 < mp / 16) fetch(k + 1);
#pragma unroll
                for (int i = 0; i < MT; i++) y[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[k & 1], h[k & 1][i], y[i], 0, 0, 0);
                if (k + 1 < mp / 16) {
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_wave_barrier();
            if (it == 0)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int e = 0; e < 16; e++) y[i][e] *= inv;
            const int sw = ns_swizzle(r32, odd) ^ kh;
#pragma unroll
            for (int q = 0; q < 4; q += 2) {
                lds_t at = Y + r32 * row + ((sw ^ (4 * strip + q)) << 4);
#pragma unroll
                for (int i = 0; i < MT; i++, at += 32 * row)
                    put_row(at, u32x2{bf16r2(y[i][4 * q], y[i][4 * q + 1]), bf16r2(y[i][4 * q + 2], y[i][4 * q + 3])},
                            u32x2{bf16r2(y[i][4 * q + 4], y[i][4 * q + 5]), bf16r2(y[i][4 * q + 6], y[i][4 * q + 7])});
            }
        }
        __syncthreads();
    }
    u32x4* dst = reinterpret_cast<u32x4*>(steps & 1 ? M.Y2 : M.Y);
    auto store = [&](int i, const auto& at, int n) {
        constexpr int BATCH = std::extent_v<std::remove_reference_t<decltype(at)>>;
        u32x4 v[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; u++) if (u < n) v[u] = *(lds_vec)(Y + at[u]);
#pragma unroll
        for (int u = 0; u < BATCH; u++) if (u < n) *(gvec_w)(dst + i + u * NS_THREADS) = v[u];
    };
    if (few) stream(std::integral_constant<int, 4>{}, store);
    else stream(std::integral_constant<int, 16>{}, store);
}

__global__ __launch_bounds__(NS_THREADS) void k_newton_schulz(Batch B, int steps) {
    extern __shared__ __attribute__((aligned(16))) bf16_t smem[];
    const int mi = blockIdx.x;
    const Mat& M = B.mats[mi];
    // the norm, from the momentum kernel's tiles (a matrix has at most 16 of them): all read at once, then added in order
    const int t0 = B.ttile_prefix[mi], nt = B.ttile_prefix[mi + 1] - t0;
    const double mine = (int)(threadIdx.x & 63) < nt ? B.partials[t0 + (threadIdx.x & 63)] : 0.0;
    double part = 0.0;
    for (int k = 0; k < nt; k++) part += __shfl(mine, k);
    const float inv = 1.0f / ((float)sqrt(part) + 1e-7f);
    if (M.mp == 128) newton_schulz<4>(M, inv, steps, smem);
    else newton_schulz<2>(M, inv, steps, smem);
}

// p = (p - 0.2*lr*X) * (1 - lr*wd).  X lies in the wide orientation; one 64x64 tile of the parameter's own
// orientation per workgroup (the grid of k_momentum), a tall parameter's tile of X is transposed through LDS.
// scale_inv: no iteration ran, X is still the unnormalised momentum; type: what X is held in
__global__ __launch_bounds__(256) void k_update(Batch B, float lr, float decay, int y_sel, int scale_inv, int type) {
    __shared__ bf16_t t[64][66];
    const int mi = sg::upper_seg(B.ttile_prefix, B.P, blockIdx.x);
    const Mat& M = B.mats[mi];
    const bf16_t* X = y_sel ? M.Y2 : M.Y;         // [mp x np]
    const int C = M.wide ? M.np : M.mp;           // padded columns of the parameter's orientation
    const int tile = (int)blockIdx.x - B.ttile_prefix[mi];
    const int tc = C / 64, tr0 = (tile / tc) * 64, tc0 = (tile % tc) * 64;
    if (tr0 >= M.rows || tc0 >= M.cols) return;   // padding only (uniform over the workgroup)
    // the reference's scalar arithmetic (csrc/ops.cpp:729-734)
    const float max_dim = (float)max(M.rows, M.cols);
    const float scale_factor = 0.2f * sqrtf(max_dim);
    const float neg_lr_scale = -lr * scale_factor / sqrtf(max_dim);
    const float xs = scale_inv ? B.inv_norm[mi] : type == T_F16 ? F16_UNSCALE : 1.0f;
    const int dtype = type == T_F16 ? SG_F16 : SG_BF16;
    const bool full = tr0 + 64 <= M.rows && tc0 + 64 <= M.cols && M.vec8;
    const int lr_ = threadIdx.x >> 2, c0 = (threadIdx.x & 3) * 16;
    if (!M.wide) {
        // X tile: rows = the parameter's columns tc0.., columns = its rows tr0.. (the padded buffer covers all of it)
        const SG_GLOBAL u32x4* src = (const SG_GLOBAL u32x4*)(X + (size_t)(tc0 + lr_) * M.np + tr0 + c0);
        const u32x4 w0 = src[0], w1 = src[1];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            t[lr_][c0 + 2 * q] = (bf16_t)(w0[q] & 0xffffu);
            t[lr_][c0 + 2 * q + 1] = (bf16_t)(w0[q] >> 16);
            t[lr_][c0 + 8 + 2 * q] = (bf16_t)(w1[q] & 0xffffu);
            t[lr_][c0 + 8 + 2 * q + 1] = (bf16_t)(w1[q] >> 16);
        }
        __syncthreads();
    }
    if (full) {
        // interior tile: a lane moves 16 consecutive elements of a row
        const size_t at = (size_t)(tr0 + lr_) * M.cols + tc0 + c0;
        float o[16], p[16];
        if (M.wide) {
            load8(X, dtype, (size_t)(tr0 + lr_) * M.np + tc0 + c0, o);
            load8(X, dtype, (size_t)(tr0 + lr_) * M.np + tc0 + c0 + 8, o + 8);
        } else {
#pragma unroll
            for (int e = 0; e < 16; e++) o[e] = type == T_F16 ? widen<T_F16>(t[c0 + e][lr_], 0) : sg::bf16_bits_to_f(t[c0 + e][lr_]);
        }
        load8(M.param, M.dtype, at, p);
        load8(M.param, M.dtype, at + 8, p + 8);
#pragma unroll
        for (int e = 0; e < 16; e++) {
            o[e] *= xs;
            if (M.dtype == SG_F16) o[e] = __half2float(__float2half_rn(o[e]));     // X.to(p.dtype)
            p[e] = sg_fma(neg_lr_scale, o[e], p[e]) * decay;
        }
        store8(M.param, M.dtype, at, p);
        store8(M.param, M.dtype, at + 8, p + 8);
        return;
    }
    for (int k = threadIdx.x; k < 64 * 64; k += 256) {
        const int r = tr0 + (k >> 6), c = tc0 + (k & 63);
        if (r >= M.rows || c >= M.cols) continue;
        const bf16_t x = M.wide ? X[(size_t)r * M.np + c] : t[k & 63][k >> 6];
        float o = (type == T_F16 ? widen<T_F16>(x, 0) : sg::bf16_bits_to_f(x)) * xs;
        if (M.dtype == SG_F16) o = __half2float(__float2half_rn(o));
        const int64_t i = (int64_t)r * M.cols + c;
        const float p = sg::load_elem(M.param, M.dtype, i);
        sg::store_elem(M.param, M.dtype, i, sg_fma(neg_lr_scale, o, p) * decay);
    }
}

inline int round_up(int x, int a) { return (x + a - 1) / a * a; }

struct Layout {
    int P;
    std::vector<Mat> mats;
    bool small;                    // every matrix fits k_newton_schulz
    bool may_share;                // some number of iterations runs in fewer stages than iterations
    bool fine[3];                  // products that go to k_gemm_64
    double time[3];                // and what count_stages takes each to cost, in microseconds
    std::vector<int> pre_g[3], pre_t;
    size_t off_mats, off_pre, off_partials, off_inv, bytes;
};

// Which products of a call take 64x64 tiles (k_gemm_64): those that a fit to the measured times says are faster so.  A product
// on 256x256 tiles takes, in microseconds, 7 + 0.0165 K for each round of 256 tiles (one per CU); on 64x64 tiles 5, and the
// longer of the chain of one tile (0.003 K) and what all tiles take together (3 ns and 14 ps per k each).  Over 18 sets from
// 1 x 200 x 800 to 6 x 1024 x 4096 the choice so made was within 8 % of the best.
// fine_pad: what the matrices would be padded to for k_gemm_64 (64, or 256 where another product keeps its large tiles)
// time: what the chosen form costs one of many products in a row.  Rounds that fill the chip are held at the rate that the part's
// power allows, 1.1 PFLOP/s (a tile's K at 0.12 ns; 24 of 1024 x 1024 take 43 to 55 us for the symmetric products, the fit 24).
void choose_tiles(int P, const SgMuonMatrix* in, int fine_pad, bool fine[3], double time[3]) {
    double tiles[3] = {}, each[3] = {}, chain[3] = {}, k_max[3] = {}, work[3] = {};
    for (int i = 0; i < P; i++) {
        const double m = (double)std::min(in[i].rows, in[i].cols), n = (double)std::max(in[i].rows, in[i].cols);
        auto up = [](double x, int a) { return std::ceil(x / a) * a; };
        for (int e = 0; e < 3; e++) {
            auto count = [&](int pad, int size) {
                const double tm = up(m, pad) / size, tn = up(n, pad) / size;
                return e == EPI_APPLY ? tm * tn : tm * (tm + 1) / 2;
            };
            const double k256 = up(e == EPI_GRAM ? n : m, BT);
            tiles[e] += count(BT, BT);
            work[e] += count(BT, BT) * k256;
            k_max[e] = std::max(k_max[e], k256);
            const double k = up(e == EPI_GRAM ? n : m, fine_pad);
            each[e] += count(fine_pad, NT64) * (0.003 + 14e-6 * k);
            chain[e] = std::max(chain[e], 0.003 * k);
        }
    }
    for (int e = 0; e < 3; e++) {
        const double rounds = std::ceil(tiles[e] / 256.0);
        const double small = 5.0 + std::max(chain[e], each[e]), large = rounds * (7.0 + 0.0165 * k_max[e]);
        fine[e] = small < large;
        time[e] = fine[e] ? small : std::max(large, 12.0 * rounds + 1.2e-4 * work[e]);
    }
}

// In how many stages the iterations run (see the head of the file): at most three iterations a stage, or one a stage (the Gram
// matrix from Y every time, in bf16), which near squares and in calls that wait for launches more than for products is
// faster.  By the products' costs.  Over 80 sets of 1 to 60 matrices with sides of 130 to 8192, ratios of 1 to 30 and 2 to 7
// iterations, the measured ratio tracked / each was 0.89-1.07 of the expected one where all products take 64x64 tiles, 1.0-1.24
// where some do and 1.07-1.20 where none does, hence three lines.  They keep out what would be slower for it (tracked is at most
// 0.99 of each where they choose it), and with that some calls that would be up to 10 % faster.  Five iterations, each /
// tracked, expected: 24 of 1024 x 1024 822 / 933 us (1.05), 12 of 1536 x 1920 1434 / 1513 (0.91), 24 of 768 x 1152 670 / 694
// (0.92), 12 of 1536 x 2304 1538 / 1563 (0.88), 24 of 1024 x 2048 1262 / 1169 (0.81), 24 of 1024 x 4096 2243 / 1683 (0.63); 16 of
// 512 x 2048 367 / 341 (0.82), 6 of 1024 x 2048 465 / 463 (0.94); 12 of 300 x 1200 234 / 200 (0.93), 1 of 200 x 800 116 / 119 (1.13).
int count_stages(const Layout& L, int ns_steps) {
    if (!L.may_share) return ns_steps;
    const int stages = (ns_steps + 2) / 3;
    const double ends = L.time[EPI_GRAM] + L.time[EPI_APPLY], poly = L.time[EPI_POLY];
    const double tracked = stages * ends + (4.0 * ns_steps - 3.0 * stages) * poly, each = ns_steps * (ends + poly);
    const int fine = L.fine[EPI_GRAM] + L.fine[EPI_POLY] + L.fine[EPI_APPLY];
    return tracked < (fine == 3 ? 0.95 : fine > 0 ? 0.9 : 0.86) * each ? stages : ns_steps;
}

int make_layout(int P, const SgMuonMatrix* in, Layout* L) {
    L->P = P;
    L->mats.resize(P);
    for (int k = 0; k < 3; k++) L->pre_g[k].assign(P + 1, 0);
    L->pre_t.assign(P + 1, 0);
    size_t o = 0;
    auto take = [&](size_t b) { size_t r = o; o = sg::align_up(o + b, 256); return r; };
    L->off_mats = take(sizeof(Mat) * (size_t)P);
    L->off_pre = L->off_mats + sizeof(Mat) * (size_t)P;      // right behind the records: one upload
    o = sg::align_up(L->off_pre + 4 * sizeof(int) * (size_t)(P + 1), 256);
    // One workgroup per matrix does its five iterations in 50 us at most (128 x 512), fifteen products of small matrices take
    // ten to fourteen each; next to matrices that need the products anyway the small ones come along in their launches.
    L->small = true;
    for (int i = 0; i < P; i++) {
        const int64_t m = std::min(in[i].rows, in[i].cols), n = std::max(in[i].rows, in[i].cols);
        L->small = L->small && m > 0 && m <= 128 && n <= NS_Y_ELEMS && fits_lds(round_up((int)m, 64), round_up((int)n, 64));
    }
    auto all_fine = [&] { return L->fine[EPI_GRAM] && L->fine[EPI_POLY] && L->fine[EPI_APPLY]; };
    choose_tiles(P, in, NT64, L->fine, L->time);
    if (!all_fine()) choose_tiles(P, in, BT, L->fine, L->time);
    const int pad = L->small || all_fine() ? 64 : BT;
    // (sharing costs least, beside one Gram matrix an iteration, where every stage has its three iterations)
    L->may_share = !L->small;
    L->may_share = count_stages(*L, 3) < 3;
    for (int i = 0; i < P; i++) {
        const SgMuonMatrix& s = in[i];
        if (s.rows <= 0 || s.cols <= 0 || s.rows * s.cols > 0x7fffffff) return sg::fail("matrix %d: bad shape %lld x %lld", i, (long long)s.rows, (long long)s.cols);
        if (s.dtype != SG_F32 && s.dtype != SG_F16 && s.dtype != SG_BF16) return sg::fail("matrix %d: bad dtype %d", i, s.dtype);
        Mat& M = L->mats[i];
        M.param = s.param; M.grad = s.grad; M.buf = s.buf;
        M.rows = (int)s.rows; M.cols = (int)s.cols; M.dtype = s.dtype;
        M.wide = s.rows <= s.cols;
        M.vec8 = (s.cols % 8 == 0) && ((((uintptr_t)s.param | (uintptr_t)s.grad | (uintptr_t)s.buf) & 15u) == 0);
        M.m = (int)std::min(s.rows, s.cols); M.n = (int)std::max(s.rows, s.cols);
        M.mp = round_up(M.m, pad); M.np = round_up(M.n, pad);

        for (int e = 0; e < 3; e++) {
            const int size = L->fine[e] ? NT64 : BT, nt = M.mp / size;
            // symmetric products: tiles on or above the diagonal
            L->pre_g[e][i + 1] = L->pre_g[e][i] + (e == EPI_APPLY ? nt * (M.np / size) : nt * (nt + 1) / 2);
        }
        L->pre_t[i + 1] = L->pre_t[i] + (M.mp / 64) * (M.np / 64);
    }
    int64_t ttiles = 0;
    for (int i = 0; i < P; i++) ttiles += (int64_t)(L->mats[i].mp / 64) * (L->mats[i].np / 64);
    L->off_partials = take(sizeof(double) * (size_t)(ttiles + 1));
    L->off_inv = take(sizeof(float) * (size_t)P);
    for (int i = 0; i < P; i++) {
        Mat& M = L->mats[i];
        // offsets for now; turned into pointers once the workspace base is known
        M.Y = (bf16_t*)take(2 * (size_t)M.mp * M.np);
        M.Y2 = (bf16_t*)take(2 * (size_t)M.mp * M.np);
        M.T = M.T2 = nullptr;
        for (auto& w : M.W) w = nullptr;
        if (L->small) continue;
        if (L->fine[EPI_APPLY]) {
            M.T = (bf16_t*)take(2 * (size_t)M.mp * M.np);
            M.T2 = (bf16_t*)take(2 * (size_t)M.mp * M.np);
        }
        for (int k = 0; k < (L->may_share ? 5 : 2); k++) M.W[k] = (bf16_t*)take(2 * (size_t)M.mp * M.mp);
    }
    L->bytes = o;
    return 0;
}

// The products, on tiles of either size.
struct Product {
    int epi, in, out;
    void (*k256)(Batch, Ops, int, int);
    void (*k64)(Batch, Ops, int, int);
};
#define SG_PRODUCT(E, I, O) {E, I, O, k_gemm_nt<E, I, O>, k_gemm_64<E, I, O>}
const Product products[] = {
    SG_PRODUCT(EPI_GRAM, T_BF16, T_BF16),  SG_PRODUCT(EPI_POLY, T_BF16, T_BF16),  SG_PRODUCT(EPI_APPLY, T_BF16, T_BF16),
    SG_PRODUCT(EPI_GRAM, T_BF16, T_F16),   SG_PRODUCT(EPI_GRAM, T_F16, T_F16),    SG_PRODUCT(EPI_POLY, T_F16, T_F16),
    SG_PRODUCT(EPI_MUL, T_F16, T_F16),     SG_PRODUCT(EPI_MUL, T_F16, T_BF16),
    SG_PRODUCT(EPI_APPLY, T_BF16, T_F16),  SG_PRODUCT(EPI_APPLY, T_F16, T_F16),
};
#undef SG_PRODUCT

}  // namespace
}  // namespace sgmu

extern "C" {

size_t sg_muon_workspace_bytes(int num_matrices, const SgMuonMatrix* mats) {
    if (num_matrices <= 0 || !mats) return 0;
    sgmu::Layout L;
    if (sgmu::make_layout(num_matrices, mats, &L)) return 0;
    return L.bytes;
}

int sg_muon_stages_for(int num_matrices, const SgMuonMatrix* mats, int ns_steps) {
    sgmu::Layout L;
    if (num_matrices <= 0 || ns_steps < 0 || !mats) return sg::fail("no matrices, or ns_steps below 0"), -1;
    if (sgmu::make_layout(num_matrices, mats, &L)) return -1;
    return sgmu::count_stages(L, ns_steps);
}

int sg_muon_tiles_for(int num_matrices, const SgMuonMatrix* mats, int tiles[3]) {
    sgmu::Layout L;
    if (num_matrices <= 0 || !mats || !tiles) return sg::fail("no matrices, or nowhere to write");
    if (sgmu::make_layout(num_matrices, mats, &L)) return 1;
    for (int e = 0; e < 3; e++) tiles[e] = L.small ? 0 : L.fine[e] ? sgmu::NT64 : sgmu::BT;
    return 0;
}

int sg_muon_step(int num_matrices, const SgMuonMatrix* mats, float momentum, float lr, float wd, int ns_steps, void* workspace,
                 size_t workspace_bytes, void* stream) {
    using namespace sgmu;
    if (num_matrices <= 0) return 0;
    if (!mats) return sg::fail("NULL argument");
    if (ns_steps < 0) return sg::fail("ns_steps must be >= 0");
    for (int i = 0; i < num_matrices; i++)
        if (!mats[i].param || !mats[i].grad || !mats[i].buf) return sg::fail("matrix %d: NULL pointer", i);
    Layout L;
    if (make_layout(num_matrices, mats, &L)) return 1;
    if (!workspace || workspace_bytes < L.bytes) return sg::fail("workspace too small: need %zu bytes, got %zu", L.bytes, workspace_bytes);
    if (((uintptr_t)workspace & 255u) != 0) return sg::fail("workspace must be 256-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    unsigned char* ws = static_cast<unsigned char*>(workspace);
    const int P = L.P;
    for (auto& M : L.mats) {
        M.Y = (bf16_t*)(ws + (size_t)M.Y); M.Y2 = (bf16_t*)(ws + (size_t)M.Y2);
        for (auto& w : M.W) if (w) w = (bf16_t*)(ws + (size_t)w);
        if (M.T) { M.T = (bf16_t*)(ws + (size_t)M.T); M.T2 = (bf16_t*)(ws + (size_t)M.T2); }
    }
    // per-call tables: through kernel arguments (no host-to-device copy, nothing blocks the host), records and tile prefixes
    // one after the other
    Batch B;
    {
        std::vector<uint32_t> w((sizeof(Mat) * (size_t)P) / 4 + 4 * (size_t)(P + 1));
        memcpy(w.data(), L.mats.data(), sizeof(Mat) * (size_t)P);
        uint32_t* pre = w.data() + sizeof(Mat) * (size_t)P / 4;
        static_assert(sizeof(Mat) % 4 == 0, "records in words");
        for (int k = 0; k < 4; k++) memcpy(pre + (size_t)k * (P + 1), (k < 3 ? L.pre_g[k] : L.pre_t).data(), sizeof(int) * (size_t)(P + 1));
        if (sg::upload_words(ws + L.off_mats, w.data(), 4 * w.size(), st)) return 1;
    }
    B.mats = reinterpret_cast<const Mat*>(ws + L.off_mats);
    const int* pre = reinterpret_cast<const int*>(ws + L.off_pre);
    for (int k = 0; k < 3; k++) B.gtile_prefix[k] = pre + (size_t)k * (P + 1);
    B.ttile_prefix = pre + 3 * (size_t)(P + 1);
    B.P = P;
    for (int k = 0; k < 3; k++) B.gtiles[k] = L.pre_g[k][P];
    B.ttiles = L.pre_t[P];
    B.partials = reinterpret_cast<double*>(ws + L.off_partials);
    B.inv_norm = reinterpret_cast<float*>(ws + L.off_inv);

    {   // the GEMM needs more LDS than the default per-kernel limit: raise it once per device
        static bool raised[64] = {};
        int dev = 0;
        SG_HIP_CHECK(hipGetDevice(&dev));
        if (dev < 0 || dev >= 64) return sg::fail("device index %d out of range", dev);
        if (!raised[dev]) {
            for (const Product& p : products)
                for (int fine = 0; fine < 2; fine++)
                    SG_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(fine ? p.k64 : p.k256), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     fine ? KS_LDS_BYTES : GEMM_LDS_BYTES));
            SG_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_newton_schulz), hipFuncAttributeMaxDynamicSharedMemorySize, NS_LDS_BYTES));
            raised[dev] = true;
        }
    }

    hipLaunchKernelGGL(k_momentum, dim3(B.ttiles), dim3(256), 0, st, B, momentum);
    // k_newton_schulz and k_gemm_64 add the norm up themselves
    if (ns_steps == 0 || (!L.small && !(L.fine[EPI_GRAM] && L.fine[EPI_APPLY]))) hipLaunchKernelGGL(k_norm, dim3(P), dim3(256), 0, st, B);
    SG_LAUNCH_CHECK("muon prologue");
    if (L.small && ns_steps > 0) {
        size_t lds = 0;
        for (const auto& M : L.mats) lds = std::max(lds, 2 * ((size_t)M.mp * M.np + (size_t)M.mp * M.mp));
        hipLaunchKernelGGL(k_newton_schulz, dim3(P), dim3(NS_THREADS), lds, st, B, ns_steps);
        SG_LAUNCH_CHECK("k_newton_schulz");
    }
    bool missing = false;
    auto launch = [&](int epi, int in, int out, Ops ops, int sel, int flags) {
        const int e = shape_of(epi);
        const dim3 grid(B.gtiles[e] * (ops.c2 >= 0 ? 2 : 1));
        const Product* p = std::find_if(std::begin(products), std::end(products), [&](const Product& q) { return q.epi == epi && q.in == in && q.out == out; });
        if (p == std::end(products)) missing = true;
        else if (L.fine[e]) hipLaunchKernelGGL(p->k64, grid, dim3(KS_THREADS), KS_LDS_BYTES, st, B, ops, sel, flags);
        else hipLaunchKernelGGL(p->k256, grid, dim3(GTHREADS), GEMM_LDS_BYTES, st, B, ops, sel, flags);
    };
    const int stages = count_stages(L, ns_steps);
    const bool tracked = stages < ns_steps;
    for (int j = 0, left = ns_steps; !L.small && j < stages; j++) {
        const int n = left / (stages - j);               // iterations of this stage: the later ones take one more where they differ
        left -= n;
        const int sel = j & 1, flags = (j == 0 ? 2 : 0) | (j + 1 == stages ? 4 : 0);     // iter_flags
        if (!tracked) {
            launch(EPI_GRAM, T_BF16, T_BF16, Ops{0, 0, 0, 0, 0, -1}, sel, flags);
            launch(EPI_POLY, T_BF16, T_BF16, Ops{0, 0, 1, 0, 0, -1}, sel, flags);
            launch(EPI_APPLY, T_BF16, T_BF16, Ops{1, 0, 0, 0, 0, -1}, sel, flags);
        } else {
            // W[0] the Gram matrix, W[q] the product of the polynomials so far; the other three hold what a step forms
            const int in = j == 0 ? T_BF16 : T_F16;      // the last product of a stage becomes what Y is held in
            launch(EPI_GRAM, in, T_F16, Ops{0, 0, 0, 0, 0, -1}, sel, flags);
            int q = -1, free[4] = {1, 2, 3, 4};
            for (int k = 0; k < n; k++) {
                // P = a I + b G + c G^2, then S = P G and Q <- P Q together, then G <- S P
                const int p = free[0], s = free[1], to = free[2];
                launch(EPI_POLY, T_F16, T_F16, Ops{0, 0, p, 0, 0, -1}, sel, flags);
                if (k + 1 < n) {
                    launch(EPI_MUL, T_F16, T_F16, k == 0 ? Ops{p, 0, s, 0, 0, -1} : Ops{p, 0, s, p, q, to}, sel, flags);
                    launch(EPI_MUL, T_F16, T_F16, Ops{s, p, 0, 0, 0, -1}, sel, flags);
                } else if (k > 0) {
                    launch(EPI_MUL, T_F16, in, Ops{p, q, to, 0, 0, -1}, sel, flags);
                }
                if (k == 0) {
                    q = p; free[0] = 4;                  // of 1..4
                } else {
                    std::swap(q, free[2]);
                }
            }
            launch(EPI_APPLY, in, T_F16, Ops{q, 0, 0, 0, 0, -1}, sel, flags);
        }
        SG_LAUNCH_CHECK("muon newton-schulz");
        if (missing) return sg::fail("internal: a product of these types has no kernel");
    }
    hipLaunchKernelGGL(k_update, dim3(B.ttiles), dim3(256), 0, st, B, lr, 1.0f - lr * wd, stages & 1, ns_steps == 0 ? 1 : 0, tracked ? T_F16 : T_BF16);
    SG_LAUNCH_CHECK("k_update");
    return 0;
}

}  // extern "C"
