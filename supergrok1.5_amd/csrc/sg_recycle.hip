// Expert recycling: dead experts become noisy clones of a sampled one, keys that only dead experts share are drawn anew
// (_recycle_dead_experts, grokking_optimizers/mamba3_peer_metanet.py:437-491 of the reference).
// A few hundred draws of a few values each: as library calls they are a launch apiece, 3.5 ms of host time in an event with
// 144 dead experts (35 us a step at one event in 100 steps, a third of the step of a small model).  Here they are two launches.
//
// The draws are those of the framework's device generator (torch's normal_ on the GPU), to rounding: Philox4x32-10 (Salmon
// et al., "Parallel random numbers: as easy as 1, 2, 3", 2011) with the generator's seed as key, counter = (offset / 4,
// element), and Box-Muller (1958) on the first two words.  A draw of up to 256 values per CU moves the generator's offset by
// 4.  Which words and counters a draw takes is observed, not documented: the caller compares both once per device
// (generator_is_known in ops_group.cpp) and leaves these kernels where they differ.
#include "sg_common.hpp"

#include <cstring>
#include <vector>

namespace sgrc {
namespace {

__device__ __forceinline__ float normal(uint64_t seed, uint64_t block, uint32_t element) {
    uint32_t c0 = (uint32_t)block, c1 = (uint32_t)(block >> 32), c2 = element, c3 = 0;
    uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
#pragma unroll
    for (int r = 0; r < 10; r++) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        c0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
        c1 = (uint32_t)p1;
        c2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        c3 = (uint32_t)p0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    // (0, 1] from 32 bits; the angle in half turns
    const float u = sg_fma((float)c0, 0x1p-32f, 0x1p-33f), v = sg_fma((float)c1, 0x1p-31f, 0x1p-32f);
    return sqrtf(-2.0f * logf(u)) * sinpif(v);
}

struct Experts {
    float* t[4];
    int row[4];             // values per expert
    int group0[5];          // first workgroup of each tensor
};

// dead: {expert, draw number of its first tensor} each.  A workgroup takes 16 values of every dead expert's row of one
// tensor, so that it alone reads the sampled expert's values and may write them.
__global__ __launch_bounds__(256) void k_clone_experts(Experts X, const int2* dead, int num_dead, int top, uint64_t seed, uint64_t block) {
    int which = 0;
    while ((int)blockIdx.x >= X.group0[which + 1]) which++;
    const int j = ((int)blockIdx.x - X.group0[which]) * 16 + (threadIdx.x & 15), n = X.row[which];
    float* t = X.t[which];
    const bool mine = j < n;
    float base = mine ? t[(size_t)top * n + j] : 0.0f, base_after = base;
    int at = num_dead;              // the sampled expert may be dead itself: those after it clone its new values
    for (int k = 0; k < num_dead; k++)
        if (dead[k].x == top) at = k;
    if (at < num_dead) base_after = base + 0.01f * normal(seed, block + (uint64_t)(dead[at].y + which), (uint32_t)j);
    __syncthreads();                // the old values have been read
    if (!mine) return;
    for (int k = (int)(threadIdx.x >> 4); k < num_dead; k += 16)
        t[(size_t)dead[k].x * n + j] = (k > at ? base_after : base) + 0.01f * normal(seed, block + (uint64_t)(dead[k].y + which), (uint32_t)j);
}

struct Key {
    float* row;
    int n, draw;
};

__global__ __launch_bounds__(64) void k_redraw_keys(const Key* keys, uint64_t seed, uint64_t block) {
    const Key K = keys[blockIdx.x];
    for (int j = threadIdx.x; j < K.n; j += 64) K.row[j] = 0.02f * normal(seed, block + (uint64_t)K.draw, (uint32_t)j);
}

}  // namespace
}  // namespace sgrc

extern "C" int sg_recycle_experts(const SgRecycle* r, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace sgrc;
    if (!r || r->num_dead < 0 || r->num_keys < 0) return sg::fail("recycle: NULL or negative argument");
    static_assert(sizeof(Key) == 16 && sizeof(int2) == 8, "table records");
    const size_t need = sizeof(Key) * (size_t)r->num_keys + sizeof(int2) * (size_t)r->num_dead;
    if (need == 0) return 0;
    if ((r->num_dead > 0 && (!r->dead || !r->draw)) || (r->num_keys > 0 && (!r->key_rows || !r->key_lengths || !r->key_draws)))
        return sg::fail("recycle: NULL argument");
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 15u) != 0) return sg::fail("recycle: needs a 16-byte aligned workspace of %zu bytes", need);
    if (r->offset % 4 != 0) return sg::fail("recycle: the generator's offset must be a multiple of 4");
    Experts X;
    X.group0[0] = 0;
    for (int k = 0; k < 4; k++) {
        X.t[k] = r->tensors[k];
        X.row[k] = r->row[k];
        if (r->num_dead > 0 && (!X.t[k] || X.row[k] <= 0)) return sg::fail("recycle: bad expert tensor %d", k);
        X.group0[k + 1] = X.group0[k] + (X.row[k] + 15) / 16;
    }
    for (int k = 0; k < r->num_dead; k++)
        if (r->dead[k] < 0 || r->dead[k] >= r->num_experts) return sg::fail("recycle: expert %d out of range", r->dead[k]);
    if (r->num_dead > 0 && (r->top < 0 || r->top >= r->num_experts)) return sg::fail("recycle: expert %d out of range", r->top);
    for (int k = 0; k < r->num_keys; k++)
        if (!r->key_rows[k] || r->key_lengths[k] <= 0) return sg::fail("recycle: bad key %d", k);
    hipStream_t st = (hipStream_t)stream;
    std::vector<uint32_t> w(need / 4);
    Key* keys = reinterpret_cast<Key*>(w.data());
    for (int k = 0; k < r->num_keys; k++) {
        const Key K = {r->key_rows[k], r->key_lengths[k], r->key_draws[k]};
        memcpy(keys + k, &K, sizeof(K));
    }
    uint32_t* d = w.data() + 4 * (size_t)r->num_keys;
    for (int k = 0; k < r->num_dead; k++) { d[2 * k] = (uint32_t)r->dead[k]; d[2 * k + 1] = (uint32_t)r->draw[k]; }
    if (sg::upload_words(workspace, w.data(), need, st)) return 1;
    const Key* keys_dev = static_cast<const Key*>(workspace);
    const int2* dead_dev = reinterpret_cast<const int2*>(keys_dev + r->num_keys);
    const uint64_t block = r->offset / 4;
    if (r->num_dead > 0) hipLaunchKernelGGL(k_clone_experts, dim3(X.group0[4]), dim3(256), 0, st, X, dead_dev, r->num_dead, r->top, r->seed, block);
    if (r->num_keys > 0) hipLaunchKernelGGL(k_redraw_keys, dim3(r->num_keys), dim3(64), 0, st, keys_dev, r->seed, block);
    SG_LAUNCH_CHECK("expert recycling");
    return 0;
}
