// Segmented, stable, ascending LSD radix sort of (|grad| bits, element index)
// for all parameter tensors at once.  One segment per tensor.
//
// Stands in for the reference's input_proj_sort_kernel key generation
// (csrc/supergrok2_mamba_peer_kernels.cu:92-117) and its
// cub::DeviceSegmentedRadixSort::SortPairs call (:1860-1879).  Non-negative
// floats order like their bit patterns, so the keys are sorted as uint32.
//
// Small calls sort runs of 4096 keys in LDS and merge a tensor's runs (k_sort_runs, k_merge_runs); the others:
// Four passes of 8 bits (two where all gradients are 16-bit, see key_bits) over tiles of 8192 keys (512 lanes x 16), or of
// 2048 where the call is small.  Per pass:
//   hist     per-tile digit counts -> spine[segment][digit][tile]  (first pass: counted while the keys are made)
//   scan     exclusive prefix over the whole spine (2 small kernels).  Because
//            the spine is laid out segment-major, the global prefix of entry
//            (seg, d, tile) is exactly: keys in earlier segments + keys of this
//            segment with a smaller digit + keys with digit d in earlier tiles
//            = destination of the first such key of this tile.
//            Calls whose tensors have few tiles each, and small calls, have no scan: a
//            scatter workgroup adds up the counts of its own segment itself.
//   scatter  stable rank inside the tile (each wave owns a contiguous quarter
//            of the tile; match-any ballots give the rank among equal digits)
//            and write to destination; the last pass of a small call also takes
//            the sharpness along into sorted order (large ones: a kernel of its own).
// Calls whose tensors all fit one tile (see sort_tile_for) are sorted by one launch, a workgroup per
// tensor that keeps its keys in LDS for all passes.
#include <type_traits>

#include "sg2_compose_block.hpp"
#include "sg2_internal.hpp"

namespace sg2 {
namespace {

constexpr int SORT_THREADS = 512;
constexpr int WAVES = SORT_THREADS / 64;
static_assert(SORT_THREADS >= 256 && SORT_THREADS % 64 == 0 && SORT_TILE_SMALL % SORT_THREADS == 0, "one thread per digit at least");

struct TileRef {
    int base;        // index of the tile's first key in the packed arrays
    int cnt;         // keys in the tile
    int spine0;      // index of spine entry (digit 0) for this tile
    int stride;      // spine stride between digits
    int tiles;       // tiles of the segment
    int seg;         // the segment
    int tile;        // tile within the segment
    int seg_off;     // index of the segment's first key
};
// SELF: the spine is laid out [segment][tile][digit], else [segment][digit][tile] (see k_scatter)
template <bool SELF>
__device__ __forceinline__ TileRef tile_ref(const Plan& pl, int tile) {
    const sg::Seg seg = sg::find_seg(sg::as_const(pl.sort_tile_prefix), pl.P, tile);
    const int t0 = seg.first, nt = seg.end - seg.first;
    const TensorDev& T = pl.tensors[seg.i];
    TileRef r;
    r.seg = seg.i;
    r.base = T.off + (tile - t0) * pl.sort_tile;
    r.cnt = min(pl.sort_tile, T.numel - (tile - t0) * pl.sort_tile);
    r.spine0 = SELF ? 256 * tile : 256 * t0 + (tile - t0);
    r.stride = SELF ? 1 : nt;
    r.tiles = nt;
    r.tile = tile - t0;
    r.seg_off = T.off;
    return r;
}


// ---- digit counts of the first pass, straight from the gradients ----------------------
// One sort tile per workgroup.  The keys themselves are never written in element order: the first scatter pass
// forms them again from the gradients (key_of / payload_of) while it moves them.
// key = |g| bits; the sign rides in bit 31 of the payload so that the sorted (key, payload) pair gives back g
// exactly and the scan never has to gather gradients from element order
__device__ __forceinline__ uint32_t key_of(float g) { return (uint32_t)sg_f2i(sg_abs(g)); }
__device__ __forceinline__ int32_t payload_of(float g, int index) { return index | (sg_f2i(g) & (int32_t)0x80000000); }
// What the passes order a key by.  The magnitude of a 16-bit gradient has at most 16 significant bits, so a call (a tensor,
// where one workgroup sorts it) of such gradients only takes two passes: bfloat16 is the upper half of the key; a float16
// that is not zero has its ten mantissa bits at 13 .. 22 and an exponent field from 103 (subnormals) to 142, so the key >> 13
// less 102 << 10 fits 16 bits and orders like the key.  Arrays, payloads and whatever is read from them stay as they are.
// (3.1 M bfloat16 elements: 65 us less, two scatters of 17, two counts of 9 and four scans of 5 us less.)
struct KeyBits {
    int shift, bias;
};
template <bool HALF>
__device__ __forceinline__ KeyBits key_bits(int dtype) {
    return HALF ? (dtype == SG_F16 ? KeyBits{13, 102 << 10} : KeyBits{16, 0}) : KeyBits{0, 0};
}
template <bool HALF>
__device__ __forceinline__ uint32_t order_of(uint32_t key, KeyBits b) {
    return HALF ? (uint32_t)max((int)(key >> b.shift) - b.bias, 0) : key;
}

// Without SAM the sharpness of every element is 0 (the optimizer's initial state): remember per tensor whether anything
// else was seen, so that the gather into sorted order can be skipped for such tensors.  (plain store, and only while the
// flag still reads 0: every writer stores the same value; called by the whole workgroup)
__device__ __forceinline__ void note_sharpness(const Plan& pl, int seg, bool nz) {
    if (__syncthreads_or(nz) && threadIdx.x == 0) {
        volatile int* flag = pl.sharp_nonzero + seg;
        if (*flag == 0) *flag = 1;
    }
}

// Factor of the tensor's gradients in a clipping call: the workgroup adds up the tensor's norm tiles (k_tables) itself, in
// the order of a 256-lane reduction; `keep` stores it for the later kernels.
__device__ __forceinline__ float clip_factor(const Plan& pl, int ti, bool keep) {
    if (!pl.gscale) return 1.0f;
    __shared__ double sm[4];
    double part = 0.0;
    if (threadIdx.x < 256)
        for (int k = pl.norm_tile_prefix[ti] + (int)threadIdx.x; k < pl.norm_tile_prefix[ti + 1]; k += 256) part += pl.norm_partials[k];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) part += __shfl_down(part, d, 64);
    if (threadIdx.x < 256 && (threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = part;
    __syncthreads();
    // a NaN norm compares false (no clip); an infinite one gives factor 0, and what 0 * inf leaves counts as non-finite
    const float norm = (float)sqrt((sm[0] + sm[1]) + (sm[2] + sm[3]));
    const float gs = norm > pl.max_norm ? pl.max_norm / (norm + 1e-12f) : 1.0f;
    if (keep && threadIdx.x == 0) pl.gscale[ti] = gs;
    return gs;
}

// Workgroup 0 derives the scan's coefficients (compose_block); workgroup 1 + t counts tile t.
template <class G, int TILE, bool SELF, bool HALF>
__global__ __launch_bounds__(SORT_THREADS) void k_keys(Plan pl) {
    if (blockIdx.x == 0) {
        compose_block<G>(pl, SORT_THREADS);
        return;
    }
    constexpr int ITEMS = TILE / SORT_THREADS;
    // lane-selected copies of the counters, as in k_hist: gradients that came from a 16-bit format have one value of digit 0
    constexpr int HCOPY = 8, HSTRIDE = 256 + 8;
    __shared__ uint32_t hc[HCOPY * HSTRIDE];
    const int tile = (int)blockIdx.x - 1;
    const TileRef tr = tile_ref<SELF>(pl, tile);
    const int seg = tr.seg;
    const TensorDev& T = pl.tensors[seg];
    const int start = tr.base - T.off;
    for (int k = threadIdx.x; k < HCOPY * HSTRIDE; k += SORT_THREADS) hc[k] = 0;
    uint32_t* const h = hc + (threadIdx.x & (HCOPY - 1)) * HSTRIDE;
    bool nz = false;
    const float* gp = static_cast<const float*>(T.grad) + start;
    const float* sp = static_cast<const float*>(T.sharp) + start;
    // everything is requested before the clip factor is waited for
    if (!HALF && T.dtype == SG_F32 && tr.cnt == TILE && ((((uintptr_t)gp) | ((uintptr_t)sp)) & 15u) == 0) {
        // whole fp32 tile on a 16-byte boundary: 16 bytes per lane and load
        constexpr int VR = TILE / (4 * SORT_THREADS);
        typedef float vf4 __attribute__((ext_vector_type(4)));
        vf4 g[VR], sh[VR];
#pragma unroll
        for (int r = 0; r < VR; r++) g[r] = ((const SG_GLOBAL vf4*)gp)[r * SORT_THREADS + (int)threadIdx.x];
#pragma unroll
        for (int r = 0; r < VR; r++) sh[r] = ((const SG_GLOBAL vf4*)sp)[r * SORT_THREADS + (int)threadIdx.x];
        const float gs = clip_factor(pl, seg, tr.tile == 0);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < VR; r++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                atomicAdd(&h[key_of(clipped(g[r][e], gs, SG_F32)) & 255u], 1u);
                nz = nz || sh[r][e] != 0.0f;
            }
    } else {
        float g[ITEMS];
#pragma unroll
        for (int r = 0; r < ITEMS; r++) {
            const int k = r * SORT_THREADS + (int)threadIdx.x;
            g[r] = (k < tr.cnt) ? sg::load_elem(T.grad, T.dtype, start + k) : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < ITEMS; r++) {
            const int k = r * SORT_THREADS + (int)threadIdx.x;
            if (k < tr.cnt) nz = nz || sharp_rounded(T, start + k) != 0.0f;
        }
        const float gs = clip_factor(pl, seg, tr.tile == 0);
        const KeyBits bits = key_bits<HALF>(T.dtype);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; r++) {
            const int k = r * SORT_THREADS + (int)threadIdx.x;
            if (k < tr.cnt) atomicAdd(&h[order_of<HALF>(key_of(clipped(g[r], gs, T.dtype)), bits) & 255u], 1u);
        }
    }
    note_sharpness(pl, seg, nz);
    if (threadIdx.x < 256) {
        uint32_t tot = 0;
#pragma unroll
        for (int c = 0; c < HCOPY; c++) tot += hc[c * HSTRIDE + threadIdx.x];
        pl.spine[tr.spine0 + (int)threadIdx.x * tr.stride] = tot;
    }
}

// ---- per-tile histogram ---------------------------------------------------------
template <bool SELF, bool HALF>
__global__ __launch_bounds__(SORT_THREADS) void k_hist(Plan pl, int src, int shift) {
    // HCOPY copies of the counters, chosen by lane: a pass whose digit takes few values (the exponent byte of the
    // magnitudes) would otherwise queue most of a wave's lanes on a dozen counters.  Copies start 8 banks apart.
    constexpr int HCOPY = 8, HSTRIDE = 256 + 8;
    __shared__ uint32_t hc[HCOPY * HSTRIDE];
    const TileRef tr = tile_ref<SELF>(pl, blockIdx.x);
    for (int k = threadIdx.x; k < HCOPY * HSTRIDE; k += SORT_THREADS) hc[k] = 0;
    uint32_t* const h = hc + (threadIdx.x & (HCOPY - 1)) * HSTRIDE;
    __syncthreads();
    const uint32_t* __restrict__ keys = pl.keys[src] + tr.base;
    const KeyBits bits = key_bits<HALF>(pl.tensors[tr.seg].dtype);
    // 16 bytes per lane where the tile starts on a 16-byte boundary (tensor offsets are arbitrary); the ragged end by single keys
    const int vec = ((tr.base & 3) == 0) ? (tr.cnt & ~3) : 0;
    for (int k = threadIdx.x * 4; k < vec; k += SORT_THREADS * 4) {
        const uint4 q = *reinterpret_cast<const uint4*>(keys + k);
        atomicAdd(&h[(order_of<HALF>(q.x, bits) >> shift) & 255u], 1u);
        atomicAdd(&h[(order_of<HALF>(q.y, bits) >> shift) & 255u], 1u);
        atomicAdd(&h[(order_of<HALF>(q.z, bits) >> shift) & 255u], 1u);
        atomicAdd(&h[(order_of<HALF>(q.w, bits) >> shift) & 255u], 1u);
    }
    for (int k = vec + threadIdx.x; k < tr.cnt; k += SORT_THREADS) atomicAdd(&h[(order_of<HALF>(keys[k], bits) >> shift) & 255u], 1u);
    __syncthreads();
    if (threadIdx.x < 256) {
        uint32_t tot = 0;
#pragma unroll
        for (int c = 0; c < HCOPY; c++) tot += hc[c * HSTRIDE + threadIdx.x];
        pl.spine[tr.spine0 + (int)threadIdx.x * tr.stride] = tot;
    }
}

// ---- exclusive scan of the spine -------------------------------------------------
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(v, d, 64);
        if (lane >= d) v += o;
    }
    return v;
}
// exclusive scan over the 256 threads of a block; *total receives the block sum
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* smem /*[4]*/, uint32_t* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t inc = wave_incl_scan(v);
    if (lane == 63) smem[w] = inc;
    __syncthreads();
    uint32_t base = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t s = smem[k];
        if (k < w) base += s;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return base + inc - v;
}

__global__ __launch_bounds__(256) void k_spine_reduce(const uint32_t* __restrict__ spine, uint32_t* blocksums, int n) {
    __shared__ uint32_t sm[4];
    const int base = blockIdx.x * SCAN_BLOCK_ITEMS;
    uint32_t s = 0;
    for (int k = threadIdx.x; k < SCAN_BLOCK_ITEMS; k += 256)
        if (base + k < n) s += spine[base + k];
    uint32_t tot;
    block_excl_scan(s, sm, &tot);
    if (threadIdx.x == 0) blocksums[blockIdx.x] = tot;
}
// Every workgroup adds up the block sums before its own by itself (a few hundred values for tens of millions of
// elements; 16 K on average at the 2^31-element limit, still small beside that step): no launch for a scan of them.
__global__ __launch_bounds__(256) void k_spine_down(uint32_t* spine, const uint32_t* __restrict__ blocksums, int n) {
    __shared__ uint32_t sm[4];
    constexpr int PER = SCAN_BLOCK_ITEMS / 256;
    uint32_t before;
    {
        uint32_t part = 0;
        for (int k = threadIdx.x; k < (int)blockIdx.x; k += 256) part += blocksums[k];
        block_excl_scan(part, sm, &before);
    }
    const int base = blockIdx.x * SCAN_BLOCK_ITEMS + threadIdx.x * PER;
    uint32_t v[PER], s = 0;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        v[k] = (base + k < n) ? spine[base + k] : 0u;
        s += v[k];
    }
    uint32_t tot;
    uint32_t run = before + block_excl_scan(s, sm, &tot);
#pragma unroll
    for (int k = 0; k < PER; k++) {
        if (base + k < n) spine[base + k] = run;
        run += v[k];
    }
}

// ---- stable scatter ---------------------------------------------------------------
// What a tile's keys are ranked with in LDS, and where its digits' runs start.
struct RankLds {
    uint32_t cnt[WAVES][256];     // running digit counts of each wave; later: positions of each wave's first key of a digit
    uint32_t lbase[256], wsum[4];
};
// Stable rank of every key of the tile among the keys of its digit, wave by wave; ROUNDS rounds of 64 keys per wave, wave
// w holds keys w * ROUNDS * 64 ... .  Returns in rank[r] the number of equal digits before it in its wave's part and leaves
// the waves' counts in L.cnt.  live(r): whether this lane's key of round r exists.
template <bool HALF, int ROUNDS, class Live>
__device__ __forceinline__ void rank_keys(RankLds& L, const uint32_t (&key)[ROUNDS], uint32_t (&rank)[ROUNDS], KeyBits bits, int shift, Live live) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        const bool ok = live(r);
        const uint32_t d = (order_of<HALF>(key[r], bits) >> shift) & 255u;       // 0 for a lane past the end (its key reads as 0)
        // lanes of the wave with the same digit: for every bit, keep the lanes whose bit equals this lane's.  With
        // rep = the lane's bit spread over a word, that is m & ~(ballot ^ rep): one three-input bit operation per
        // half (truth table 0x90 = a & ~(b ^ c)).  Lanes past the end hold no set bit and are outside the initial mask.
        const uint64_t m0 = __ballot(ok);
        uint32_t mlo = (uint32_t)m0, mhi = (uint32_t)(m0 >> 32);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const int32_t rep_b = __builtin_amdgcn_sbfe((int32_t)d, b, 1);
            const uint64_t bal = __ballot(rep_b != 0);
            mlo = __builtin_amdgcn_bitop3_b32(mlo, (uint32_t)bal, (uint32_t)rep_b, 0x90);
            mhi = __builtin_amdgcn_bitop3_b32(mhi, (uint32_t)(bal >> 32), (uint32_t)rep_b, 0x90);
        }
        const uint64_t m = ((uint64_t)mhi << 32) | mlo;
        if (ok) {
            const uint32_t before = __popcll(m & lt);
            const uint32_t prev = L.cnt[w][d];
            rank[r] = prev + before;
            if (before == 0) L.cnt[w][d] = prev + (uint32_t)__popcll(m);
        }
    }
}
// Digit d = threadIdx.x: total of the tile, start of the digit in the tile's digit-sorted order (lbase) and position of
// each wave's first key of it there (cnt).  Called by the whole workgroup after a barrier; ends without one.
__device__ __forceinline__ void digit_starts(RankLds& L) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int d = threadIdx.x & 255;       // (threads beyond the 256 digits repeat the first ones' work and store nothing)
    const bool own = threadIdx.x < 256;
    uint32_t tot = 0;
#pragma unroll
    for (int k = 0; k < WAVES; k++) tot += L.cnt[k][d];
    const uint32_t inc = wave_incl_scan(tot);     // over the 64 digits of this wave, then across the 4 waves
    if (lane == 63 && own) L.wsum[w] = inc;
    __syncthreads();
    uint32_t before = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) before += (k < (d >> 6)) ? L.wsum[k] : 0u;
    if (own) {
        uint32_t run = before + inc - tot;
        L.lbase[d] = run;
#pragma unroll
        for (int k = 0; k < WAVES; k++) {
            const uint32_t c = L.cnt[k][d];
            L.cnt[k][d] = run;
            run += c;
        }
    }
}

// FIRST: the pass over digit 0 takes its keys and payloads from the tensor's gradients (element order) instead of
// the key / payload arrays, which nothing has written yet.  LAST (small calls): the sharpness of an element goes with it.  SELF: the
// spine holds plain counts: digit d of the tile starts after the segment's keys of smaller digits and those of digit d in
// earlier tiles, added up here (a count per digit and tile of the segment, at most 256 of them, two lanes a digit); a scan kernel between the
// counting and the scatter of each pass costs a small call 5 us and another gap.
template <int TILE, bool FIRST, bool LAST, bool SELF, bool HALF>
__global__ __launch_bounds__(SORT_THREADS) void k_scatter(Plan pl, int src, int shift) {
    constexpr int ITEMS = TILE / SORT_THREADS;      // rounds per wave
    constexpr int WAVE_ITEMS = TILE / WAVES;        // contiguous keys per wave
    __shared__ RankLds L;
    __shared__ uint32_t gdelta[256], wtot[4];
    __shared__ uint2 half2[SELF ? 256 : 1];
    __shared__ uint32_t skey[TILE];
    __shared__ int32_t sval[TILE];
    const TileRef tr = tile_ref<SELF>(pl, blockIdx.x);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int k = threadIdx.x; k < WAVES * 256; k += SORT_THREADS) (&L.cnt[0][0])[k] = 0;
    // this tile's start in every digit's run of the segment, before the keys are looked at (its loads pass under theirs)
    uint32_t seg_total = 0, seg_before = 0;
    if (SELF) {
        // lanes 0-255 take the even tiles of their digit, lanes 256-511 the odd ones: coalesced rows of 256 counts
        static_assert(SORT_THREADS == 512, "two lanes per digit");
        const uint32_t* col = pl.spine + (tr.spine0 - 256 * tr.tile) + (threadIdx.x & 255);
#pragma unroll 4
        for (int k = threadIdx.x >> 8; k < tr.tiles; k += 2) {
            const uint32_t c = col[256 * k];
            seg_total += c;
            seg_before += k < tr.tile ? c : 0u;
        }
        if (threadIdx.x >= 256) { half2[threadIdx.x & 255] = make_uint2(seg_total, seg_before); }
    }
    __syncthreads();

    // a whole tile (all but the last tile of a tensor) needs no bounds tests: the body exists in both forms
    auto body = [&](auto full_c) {
    constexpr bool FULL = decltype(full_c)::value;
    const uint32_t* __restrict__ keys = pl.keys[src] + tr.base;
    const int32_t* __restrict__ vals = pl.vals[src] + tr.base;
    const int seg = tr.seg;
    const KeyBits bits = key_bits<HALF>(pl.tensors[seg].dtype);

    uint32_t key[ITEMS], rank[ITEMS];
    int32_t val[ITEMS];
    if (FIRST) {
        const TensorDev& T = pl.tensors[seg];
        const int start = tr.base - T.off, dtype = T.dtype;
        const float gs = grad_scale(pl, seg);
        float g[ITEMS];
#pragma unroll
        for (int r = 0; r < ITEMS; r++) {
            const int i = w * WAVE_ITEMS + r * 64 + lane;
            g[r] = (FULL || i < tr.cnt) ? sg::load_elem(T.grad, dtype, start + i) : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < ITEMS; r++) {
            const int i = w * WAVE_ITEMS + r * 64 + lane;
            const bool ok = FULL || i < tr.cnt;
            const float v = clipped(g[r], gs, dtype);
            key[r] = ok ? key_of(v) : 0u;
            val[r] = ok ? payload_of(v, start + i) : 0;
        }
    } else {
#pragma unroll
        for (int r = 0; r < ITEMS; r++) {
            const int i = w * WAVE_ITEMS + r * 64 + lane;
            const bool ok = FULL || i < tr.cnt;
            key[r] = ok ? keys[i] : 0u;
            val[r] = ok ? vals[i] : 0;
        }
    }
    rank_keys<HALF>(L, key, rank, bits, shift, [&](int r) { return FULL || w * WAVE_ITEMS + r * 64 + lane < tr.cnt; });
    __syncthreads();
    digit_starts(L);
    __syncthreads();
    if (SELF) {
        // exclusive scan of the segment's totals over the digits (lanes beyond the 256 digits store nothing)
        const int d = threadIdx.x & 255;
        const uint2 odd = half2[d];
        seg_total += odd.x;
        seg_before += odd.y;
        const uint32_t inc = wave_incl_scan(seg_total);
        if (lane == 63 && w < 4) wtot[w] = inc;
        __syncthreads();
        uint32_t smaller = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) smaller += k < (d >> 6) ? wtot[k] : 0u;
        if (threadIdx.x < 256) gdelta[d] = tr.seg_off + smaller + inc - seg_total + seg_before - L.lbase[d];
    } else if (threadIdx.x < 256) {
        gdelta[threadIdx.x] = pl.spine[tr.spine0 + (int)threadIdx.x * tr.stride] - L.lbase[threadIdx.x];     // global destination = gdelta[d] + local position (mod 2^32)
    }
    // reorder through LDS so that global stores go out in digit-sorted order: consecutive lanes then write
    // consecutive addresses within each digit's run instead of 4-byte pieces all over the tile's 256 runs
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int i = w * WAVE_ITEMS + r * 64 + lane;
        if (FULL || i < tr.cnt) {
            const uint32_t lp = L.cnt[w][(order_of<HALF>(key[r], bits) >> shift) & 255u] + rank[r];
            skey[lp] = key[r];
            sval[lp] = val[r];
        }
    }
    __syncthreads();
    uint32_t* __restrict__ kout = pl.keys[src ^ 1];
    int32_t* __restrict__ vout = pl.vals[src ^ 1];
    const bool gather = LAST && SELF && pl.sharp_nonzero[seg] != 0;      // all-zero sharpness: no sorted copy is made, every reader tests the same flag
    const TensorDev& T = pl.tensors[seg];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int lp = r * SORT_THREADS + threadIdx.x;
        if (FULL || lp < tr.cnt) {
            const uint32_t kk = skey[lp];
            const int32_t v = sval[lp];
            const uint32_t dst = gdelta[(order_of<HALF>(kk, bits) >> shift) & 255u] + (uint32_t)lp;
            kout[dst] = kk;
            vout[dst] = v;
            if (LAST && SELF && gather) pl.ssorted[dst] = sharp_of(T, v & 0x7fffffff);
        }
    }
    };
    if (tr.cnt == TILE) body(std::true_type{});
    else body(std::false_type{});
}

// All passes over n keys in LDS, by the whole workgroup after a barrier; ends with one.  ROUNDS rounds of 64 keys per wave cover them.
template <int ROUNDS, bool HALF>
__device__ __forceinline__ void sort_in_lds(RankLds& L, uint32_t* skey, int32_t* sval, int n, KeyBits bits) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t key[ROUNDS], rank[ROUNDS];
    int32_t val[ROUNDS];
    auto at = [&](int r) { return (w * ROUNDS + r) * 64 + lane; };
    for (int shift = 0; shift < (HALF ? 16 : 32); shift += 8) {
        for (int k = threadIdx.x; k < WAVES * 256; k += SORT_THREADS) (&L.cnt[0][0])[k] = 0;
#pragma unroll
        for (int r = 0; r < ROUNDS; r++) {
            key[r] = at(r) < n ? skey[at(r)] : 0u;
            val[r] = at(r) < n ? sval[at(r)] : 0;
        }
        __syncthreads();
        rank_keys<HALF>(L, key, rank, bits, shift, [&](int r) { return at(r) < n; });
        __syncthreads();
        digit_starts(L);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ROUNDS; r++)
            if (at(r) < n) {
                const uint32_t lp = L.cnt[w][(order_of<HALF>(key[r], bits) >> shift) & 255u] + rank[r];
                skey[lp] = key[r];
                sval[lp] = val[r];
            }
        __syncthreads();
    }
}

// ---- every tensor fits one tile: keys, four passes and the sharpness in one launch ----------------------------------
// Workgroup 0 derives the scan's coefficients; workgroup 1 + i sorts tensor i.  The keys stay in LDS between the passes:
// the launches of the general sort (12 for 8 tensors of at most 255 elements, 48 us) carry next to no work there.
template <class G>
__global__ __launch_bounds__(SORT_THREADS) void k_sort_tile(Plan pl) {
    if (blockIdx.x == 0) {
        compose_block<G>(pl, SORT_THREADS);
        return;
    }
    constexpr int ITEMS = SORT_TILE / SORT_THREADS;
    __shared__ RankLds L;
    __shared__ uint32_t skey[SORT_TILE];
    __shared__ int32_t sval[SORT_TILE];
    const int seg = (int)blockIdx.x - 1;
    const TensorDev& T = pl.tensors[seg];
    const int n = T.numel, dtype = T.dtype;
    if (n == 0) return;
    const float gs = clip_factor(pl, seg, true);
    bool nz = false;
    for (int i = threadIdx.x; i < n; i += SORT_THREADS) {
        const float v = clipped(sg::load_elem(T.grad, dtype, i), gs, dtype);
        skey[i] = key_of(v);
        sval[i] = payload_of(v, i);
        nz = nz || sharp_rounded(T, i) != 0.0f;
    }
    note_sharpness(pl, seg, nz);
    const bool gather = __syncthreads_or(nz);
    const int rounds = (n + SORT_THREADS - 1) / SORT_THREADS;
    auto with = [&](auto half_c) {
        constexpr bool HALF = decltype(half_c)::value;
        const KeyBits bits = key_bits<HALF>(dtype);
        if (rounds <= 1) sort_in_lds<1, HALF>(L, skey, sval, n, bits);
        else if (rounds <= 4) sort_in_lds<4, HALF>(L, skey, sval, n, bits);
        else sort_in_lds<ITEMS, HALF>(L, skey, sval, n, bits);
    };
    if (dtype == SG_F32) with(std::false_type{});
    else with(std::true_type{});
    for (int i = threadIdx.x; i < n; i += SORT_THREADS) {
        const int32_t v = sval[i];
        pl.keys[0][T.off + i] = skey[i];
        pl.vals[0][T.off + i] = v;
        if (gather) pl.ssorted[T.off + i] = sharp_of(T, v & 0x7fffffff);
    }
}

// ---- small calls: runs of RUN keys sorted by themselves, then all runs of a tensor merged at once --------------------------
// Two launches instead of the eight of the radix passes, which are bound by their latency and the gaps between them in
// such calls (14 tensors of 0.42 M elements: 57 us and as much again for 15 000).  A key's place in the tensor is its
// place in its own run plus, for every other run, the number of that run's keys before it: smaller ones, and equal ones
// where the run lies earlier (stable, as the passes are).  The runs pass through LDS two at a time while the next two are on
// their way, and a workgroup looks its 2048 keys up by halving steps.
// Bound by the vector ALU (three instructions a step, 13 steps a key and run) where a tensor has many runs: runs of 4096
// instead of 2048 halve that and add 6 us of sorting.  0.42 M elements: 21 + 26 us for 57; 15 000 elements in 6 tensors and
// 30 000 in 5 take 21 and 17 us less, one tensor of 60 000 10.
constexpr int RUN_TILES = 2, RUN = RUN_TILES * SORT_TILE_SMALL;
template <class G, bool HALF>
__global__ __launch_bounds__(SORT_THREADS) void k_sort_runs(Plan pl) {
    if (blockIdx.x == 0) {
        compose_block<G>(pl, SORT_THREADS);
        return;
    }
    constexpr int ITEMS = RUN / SORT_THREADS;
    __shared__ RankLds L;
    __shared__ uint32_t skey[RUN];
    __shared__ int32_t sval[RUN];
    const TileRef tr = tile_ref<true>(pl, (int)blockIdx.x - 1);
    if (tr.tile % RUN_TILES != 0) return;
    const TensorDev& T = pl.tensors[tr.seg];
    const int start = tr.base - T.off, dtype = T.dtype, cnt = min(RUN, T.numel - start);
    float g[ITEMS];
    bool nz = false;
    // everything is requested before the clip factor is waited for
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int k = r * SORT_THREADS + (int)threadIdx.x;
        g[r] = k < cnt ? sg::load_elem(T.grad, dtype, start + k) : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int k = r * SORT_THREADS + (int)threadIdx.x;
        if (k < cnt) nz = nz || sharp_rounded(T, start + k) != 0.0f;
    }
    const float gs = clip_factor(pl, tr.seg, tr.tile == 0);
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int k = r * SORT_THREADS + (int)threadIdx.x;
        const float v = clipped(g[r], gs, dtype);
        if (k < cnt) {
            skey[k] = key_of(v);
            sval[k] = payload_of(v, start + k);
        }
    }
    note_sharpness(pl, tr.seg, nz);              // (its barrier covers the keys)
    sort_in_lds<ITEMS, HALF>(L, skey, sval, cnt, key_bits<HALF>(dtype));
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int k = r * SORT_THREADS + (int)threadIdx.x;
        if (k < cnt) {
            pl.keys[1][tr.base + k] = skey[k];
            pl.vals[1][tr.base + k] = sval[k];
        }
    }
}

template <bool HALF>
__global__ __launch_bounds__(SORT_THREADS) void k_merge_runs(Plan pl) {
    constexpr int ITEMS = SORT_TILE_SMALL / SORT_THREADS, PARTS = RUN / SORT_THREADS, GROUP = 2;
    static_assert((RUN & (RUN - 1)) == 0, "binary search by halving steps");
    __shared__ uint32_t run[2][GROUP][RUN];
    // a tensor's tiles next to each other on an XCD: their keys fall between each other, into the same lines of its L2
    const int nb = gridDim.x, tile = nb % 8 == 0 ? ((int)blockIdx.x % 8) * (nb / 8) + (int)blockIdx.x / 8 : (int)blockIdx.x;
    const TileRef tr = tile_ref<true>(pl, tile);
    const TensorDev& T = pl.tensors[tr.seg];
    const KeyBits bits = key_bits<HALF>(T.dtype);
    uint32_t key[ITEMS], at[ITEMS], place[ITEMS], next[GROUP][PARTS];
    int32_t val[ITEMS];
    const int mine = tr.tile / RUN_TILES, others = (tr.tiles - 1) / RUN_TILES;
    auto other = [&](int j) { return j < mine ? j : j + 1; };      // the j-th of the other runs
    auto request = [&](int j0) {
#pragma unroll
        for (int u = 0; u < GROUP; u++) {
            const int first = other(j0 + u) * RUN, n = j0 + u < others ? T.numel - first : 0;
#pragma unroll
            for (int r = 0; r < PARTS; r++) {
                const int k = r * SORT_THREADS + (int)threadIdx.x;
                next[u][r] = k < n ? order_of<HALF>(pl.keys[1][tr.seg_off + first + k], bits) : 0xffffffffu;       // (beyond every key)
            }
        }
    };
    request(0);
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int k = r * SORT_THREADS + (int)threadIdx.x;
        key[r] = k < tr.cnt ? pl.keys[1][tr.base + k] : 0u;
        val[r] = k < tr.cnt ? pl.vals[1][tr.base + k] : 0;
        at[r] = order_of<HALF>(key[r], bits);
        place[r] = (uint32_t)(tr.seg_off + (tr.tile % RUN_TILES) * SORT_TILE_SMALL + k);      // in its own run
    }
    int turn = 0;
    for (int j = 0; j < others; j += GROUP, turn ^= 1) {
#pragma unroll
        for (int u = 0; u < GROUP; u++)
#pragma unroll
            for (int r = 0; r < PARTS; r++) run[turn][u][r * SORT_THREADS + (int)threadIdx.x] = next[u][r];
        __syncthreads();                             // (a wave is at most one group ahead: the other buffer)
        if (j + GROUP < others) request(j + GROUP);
        // (pointers instead of indexes: the halving steps fit the reads' offsets)
        typedef const __attribute__((address_space(3))) uint32_t* lds_keys;
        lds_keys from[GROUP][ITEMS];
        uint32_t limit[GROUP][ITEMS];
#pragma unroll
        for (int u = 0; u < GROUP; u++)
#pragma unroll
            for (int r = 0; r < ITEMS; r++) {
                from[u][r] = (lds_keys)run[turn][u];
                limit[u][r] = at[r] + (j + u < mine ? 1u : 0u);
            }
#pragma unroll
        for (int step = RUN / 2; step > 0; step >>= 1)
#pragma unroll
            for (int u = 0; u < GROUP; u++)
#pragma unroll
                for (int r = 0; r < ITEMS; r++) from[u][r] += from[u][r][step - 1] < limit[u][r] ? step : 0;
#pragma unroll
        for (int u = 0; u < GROUP; u++)
#pragma unroll
            for (int r = 0; r < ITEMS; r++) place[r] += (uint32_t)(from[u][r] - (lds_keys)run[turn][u]) + (*from[u][r] < limit[u][r] ? 1u : 0u);
    }
    const bool gather = pl.sharp_nonzero[tr.seg] != 0;       // all-zero sharpness: no sorted copy is made, every reader tests the same flag
#pragma unroll
    for (int r = 0; r < ITEMS; r++)
        if (r * SORT_THREADS + (int)threadIdx.x < tr.cnt) {
            pl.keys[0][place[r]] = key[r];
            pl.vals[0][place[r]] = val[r];
            if (gather) pl.ssorted[place[r]] = sharp_of(T, val[r] & 0x7fffffff);
        }
}

// Sharpness into sorted order for large calls (one random read per element, once, instead of one per scan pass and
// direction).  In the last scatter these reads have two workgroups per CU to hide behind (3.1 M elements: 37 us more
// there, 17 us here); small calls save the launch instead.
constexpr int GATHER_PARTS = 4;      // workgroups per sort tile
__global__ __launch_bounds__(SORT_THREADS) void k_gather_sharpness(Plan pl) {
    constexpr int ITEMS = SORT_TILE / SORT_THREADS / GATHER_PARTS;
    const TileRef tr = tile_ref<false>(pl, blockIdx.x / GATHER_PARTS);
    if (pl.sharp_nonzero[tr.seg] == 0) return;          // nothing to gather: every reader tests the same flag
    const TensorDev& T = pl.tensors[tr.seg];
    const int k0 = (blockIdx.x % GATHER_PARTS) * (SORT_TILE / GATHER_PARTS) + (int)threadIdx.x;
    float s[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int k = k0 + r * SORT_THREADS;
        s[r] = k < tr.cnt ? sharp_raw(T, pl.vals[0][tr.base + k] & 0x7fffffff) : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int k = k0 + r * SORT_THREADS;
        if (k < tr.cnt) pl.ssorted[tr.base + k] = sharp_value(T, s[r]);
    }
}

// the plain permutation, for inspection
__global__ __launch_bounds__(256) void k_permutation(Plan pl, int32_t* __restrict__ dbg_perm) {
    const int tile = blockIdx.x;
    const int ti = sg::upper_seg(sg::as_const(pl.elem_tile_prefix), pl.P, tile);
    const TensorDev& T = pl.tensors[ti];
    const int start = (tile - pl.elem_tile_prefix[ti]) * ELEM_TILE;
    const int cnt = min(ELEM_TILE, T.numel - start);
    for (int k = threadIdx.x; k < cnt; k += 256) dbg_perm[T.off + start + k] = pl.vals[0][T.off + start + k] & 0x7fffffff;
}

template <class G, int TILE, bool SELF, bool HALF>
int launch_passes(const Plan& pl, hipStream_t st) {
    hipLaunchKernelGGL((k_keys<G, TILE, SELF, HALF>), dim3(1 + pl.sort_tiles), dim3(SORT_THREADS), 0, st, pl);
    SG_LAUNCH_CHECK("k_keys");
    const int n = 256 * pl.sort_tiles;
    const int nb = (n + SCAN_BLOCK_ITEMS - 1) / SCAN_BLOCK_ITEMS;
    constexpr int PASSES = HALF ? 2 : 4;         // an even number: the last one leaves its output in keys[0] / vals[0]
    for (int pass = 0; pass < PASSES; pass++) {
        const int src = pass & 1, shift = 8 * pass;
        if (pass > 0) hipLaunchKernelGGL((k_hist<SELF, HALF>), dim3(pl.sort_tiles), dim3(SORT_THREADS), 0, st, pl, src, shift);     // the first pass's counts come from k_keys
        if (!SELF) {
            hipLaunchKernelGGL(k_spine_reduce, dim3(nb), dim3(256), 0, st, pl.spine, pl.blocksums, n);
            hipLaunchKernelGGL(k_spine_down, dim3(nb), dim3(256), 0, st, pl.spine, pl.blocksums, n);
        }
        const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(pl.sort_tiles), dim3(SORT_THREADS), 0, st, pl, src, shift); };
        if (pass == 0) go(k_scatter<TILE, true, false, SELF, HALF>);
        else if (pass == PASSES - 1 && SELF) go(k_scatter<TILE, false, SELF, SELF, HALF>);
        else go(k_scatter<TILE, false, false, SELF, HALF>);
        SG_LAUNCH_CHECK("radix pass");
    }
    if (!SELF) {
        hipLaunchKernelGGL(k_gather_sharpness, dim3(GATHER_PARTS * pl.sort_tiles), dim3(SORT_THREADS), 0, st, pl);
        SG_LAUNCH_CHECK("k_gather_sharpness");
    }
    return 0;
}

template <class G, bool HALF>
int launch_sort_geo(const Plan& pl, hipStream_t st) {
    switch (sort_form(pl.sort_tile, pl.sort_tiles, pl.sort_widest, HALF)) {
        case SG2_SORT_RUNS:
            hipLaunchKernelGGL((k_sort_runs<G, HALF>), dim3(1 + pl.sort_tiles), dim3(SORT_THREADS), 0, st, pl);
            SG_LAUNCH_CHECK("k_sort_runs");
            hipLaunchKernelGGL(k_merge_runs<HALF>, dim3(pl.sort_tiles), dim3(SORT_THREADS), 0, st, pl);
            SG_LAUNCH_CHECK("k_merge_runs");
            return 0;
        case SG2_SORT_TENSORS:
            hipLaunchKernelGGL(k_sort_tile<G>, dim3(1 + pl.P), dim3(SORT_THREADS), 0, st, pl);
            SG_LAUNCH_CHECK("k_sort_tile");
            return 0;
        case SG2_SORT_SMALL_PASSES: return launch_passes<G, SORT_TILE_SMALL, true, HALF>(pl, st);
        case SG2_SORT_PASSES: return launch_passes<G, SORT_TILE, true, HALF>(pl, st);
        default: return launch_passes<G, SORT_TILE, false, HALF>(pl, st);
    }
}

}  // namespace

// Tiles of the largest tensor up to which runs are merged.  The merge's work grows with the square of a tensor's length and the
// passes' with the length; 16-bit gradients have two passes only.  What runs change against passes over small tiles: four
// fp32 tensors of 20 000 -17 us, one of 60 000 -9, of 80 000 0, of 130 000 +7, sixteen of 60 000 -12, thirty +3 (hence the
// product); bfloat16, one of 8000 -9, four of 20 000 +3, one of 60 000 +24.
constexpr int MERGE_TILES = 40, MERGE_WORK = 20000, HALF_MERGE_TILES = 4;
int sort_form(int sort_tile, int sort_tiles, int sort_widest, bool half) {
    if (sort_tile == SORT_TILE_SMALL) {
        const bool merges = sort_widest <= (half ? HALF_MERGE_TILES : MERGE_TILES) && (int64_t)sort_tiles * sort_widest <= MERGE_WORK;
        return merges ? SG2_SORT_RUNS : SG2_SORT_SMALL_PASSES;
    }
    if (sort_widest <= 1) return SG2_SORT_TENSORS;
    return sort_widest <= SELF_SCAN_TILES ? SG2_SORT_PASSES : SG2_SORT_SCANNED_PASSES;
}

int launch_sort(const Plan& pl, int32_t* dbg_perm, hipStream_t st) {
    if (pl.total == 0) return 0;
    const int bad = pl.geo == GEO_LARGE ? (pl.half_grads ? launch_sort_geo<GeoLarge, true>(pl, st) : launch_sort_geo<GeoLarge, false>(pl, st))
                                        : (pl.half_grads ? launch_sort_geo<GeoDefault, true>(pl, st) : launch_sort_geo<GeoDefault, false>(pl, st));
    if (bad) return 1;
    // result in keys[0] / vals[0]
    if (dbg_perm) {
        hipLaunchKernelGGL(k_permutation, dim3(pl.elem_tiles), dim3(256), 0, st, pl, dbg_perm);
        SG_LAUNCH_CHECK("k_permutation");
    }
    return 0;
}

}  // namespace sg2
