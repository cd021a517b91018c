// pull.hpp -- delivery of a grouped population's recurrent spikes from the
// target's side, for the groups that fire densely.
//
// The fold (fold_ring_body) pushes every event into its target's segment with
// scattered atomics and stores, and the update kernel sorts the segment.  Where
// many sources fire it is cheaper to read every synapse: each target walks its incoming list, which is kept in delivery
// order (delay, source, position in the source's row), and tests the source's
// bit in a bitmap of the spikes of each delay's update, staged in LDS.  The
// events that are due are added to the conductance as they come: no atomics,
// no sorting, 8 coalesced bytes per synapse.
//
// Each group takes the cheaper way in each update, by the share of its
// neurons that fired over the delays' updates (pull_dense): the push fold
// skips the spikes of pulled groups, the pull kernel the others.
//
// 512 AdEx networks (2.9M neurons, in-degree 100, 330 Hz on average, some at
// 1.6 kHz and many silent), per step: pull 201 us, fold 33 us, update 49 us;
// with every event pushed the fold takes 1,047 us and the update, which sorts,
// 464 us.  The pull is bound by the 8 bytes per synapse of the dense groups.
#pragma once
#include "device_common.hpp"

namespace edl {

constexpr int kPullBlock = 512;         // neurons and threads of a pull workgroup
constexpr int kPullLanesMax = 2048;     // longest incoming list (sorted in LDS at set-up)
constexpr int kPullLdsMax = 96 << 10;   // largest bitmap of a group over all delays
// An incoming synapse: type << 31 | bit of its source in the group's bitmap,
// counted over 32-bit words, delay by delay.
constexpr uint32_t kPullType = 0x80000000u;

struct PullBlock {
    int32_t first, n;        // neurons of this block (one group's)
    int32_t group;
    int32_t gstart, words;   // first neuron of the group, 32-bit words of its bitmap
    int32_t gn;              // its neurons
};

struct PullArgs {
    const PullBlock *blocks;
    int n_blocks;               // the grid
    int groups, max_delay, ring;
    const uint32_t *ent;        // per 64-neuron slice: its lists interleaved, padded to the longest
    const float *w;
    const int64_t *slice;       // [slices + 1] first entry row (64 entries each)
    const uint32_t *bits;       // [ring][words_all]: one bit per neuron, by update slot
    int64_t words_all;
    uint32_t *count;            // [ring][groups]: spikes per group, by update slot
    uint8_t *mode;              // [2][groups] by update parity: 1 pulled
    const int32_t *gsize;       // [groups]
    float *g_exc, *g_inh;
    StepRef step;
};

// A pulled group reads 8 bytes of every synapse (1.6 ps at the rate of a large
// copy), a pushed event costs about 0.16 ns with the sorting: by those they meet
// at one neuron in 100 firing per update.  Sweeps, us per step, by the line:
//
//   networks, in-degree    1/30   1/100   1/300   1/1,000   1/3,000
//   512, 25                 124     128     126       115       108
//   512, 100                344     308     307       306       306
//   256, 250                610     609     609       608       610
//
// From one in 100 down the line hardly matters at in-degree 100 and above (few
// groups lie between), so 300 stands anywhere on that flat; sparse wiring gains
// up to 15% from a lower one, as a quiet group's walk is short.
__device__ __forceinline__ bool pull_dense(uint32_t spikes, int32_t n, int delays) {
    return (uint64_t)spikes * 300ull >= (uint64_t)n * (uint64_t)delays;
}

// Update k: adds the due events of the pulled groups to their conductances,
// decides every group's way for update k + 1, whose spikes (updates k - D to
// k - 1) are known, and clears update k's spike counts.
__global__ __launch_bounds__(kPullBlock) void k_pull(PullArgs a) {
    extern __shared__ uint32_t s_bits[];
    const int32_t k = a.step.get();
    for (int g = (int)(blockIdx.x * kPullBlock + threadIdx.x); g < a.groups; g += (int)gridDim.x * kPullBlock) {
        uint32_t c = 0;
        for (int d = 1; d <= a.max_delay; d++) {
            const int32_t s = k - d;
            if (s >= 1) c += a.count[(int64_t)(s % a.ring) * a.groups + g];
        }
        a.mode[(int64_t)((k + 1) & 1) * a.groups + g] = pull_dense(c, a.gsize[g], a.max_delay) ? 1 : 0;
        a.count[(int64_t)(k % a.ring) * a.groups + g] = 0u;
    }
    const PullBlock B = a.blocks[blockIdx.x];
    if (!a.mode[(int64_t)(k & 1) * a.groups + B.group]) return;
    for (int d = 1; d <= a.max_delay; d++) {
        const int32_t s = k - 1 - d;
        const uint32_t *src = a.bits + (int64_t)((s < 1 ? 0 : s) % a.ring) * a.words_all + B.gstart / 32;
        for (int q = threadIdx.x; q < B.words; q += kPullBlock) s_bits[(d - 1) * B.words + q] = s < 1 ? 0u : src[q];
    }
    if (threadIdx.x == 0) s_bits[a.max_delay * B.words] = 0u;   // read by the padding entries
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1);
    if ((int)threadIdx.x - lane >= B.n) return;   // whole waves: n is a multiple of kGroupAlign
    const int i = B.first + (int)threadIdx.x;
    const int64_t r0 = a.slice[i / kWave], r1 = a.slice[i / kWave + 1];
    float ge = a.g_exc[i], gi = a.g_inh[i];
    const uint32_t *ent = a.ent + r0 * kWave + lane;
    const float *w = a.w + r0 * kWave + lane;
    auto apply = [&](uint32_t e, float x) {
        const uint32_t word = s_bits[(e & ~kPullType) >> 5];
        const bool hit = (word >> (e & 31u)) & 1u;
        const bool inh = (e & kPullType) != 0u;
        const float te = ge + x, ti = gi + x;
        ge = (hit && !inh) ? te : ge;
        gi = (hit && inh) ? ti : gi;
    };
    constexpr int U = 8;   // entries in flight per lane
    int64_t r = r0;
    for (; r + U <= r1; r += U) {
        uint32_t e[U];
        float x[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            e[u] = ent[u * kWave];
            x[u] = w[u * kWave];
        }
        ent += U * kWave;
        w += U * kWave;
#pragma unroll
        for (int u = 0; u < U; u++) apply(e[u], x[u]);
    }
    for (; r < r1; r++) {
        apply(*ent, *w);
        ent += kWave;
        w += kWave;
    }
    a.g_exc[i] = ge;
    a.g_inh[i] = gi;
}

// ---- set-up -----------------------------------------------------------------
struct PullBuild {
    const int64_t *row_ptr;      // [n * max_delay + 1]
    const uint32_t *tgt_type;
    const float *w;
    int64_t n;                   // neurons of the index space (sources and targets)
    int max_delay;
    const uint32_t *chunk_group;
    const int32_t *gstart;       // [groups]
    const int32_t *gsize;
    uint32_t *deg;               // [stride] incoming synapses, then fill cursors
    const int64_t *slice;
    uint64_t *key;               // interleaved like ent: delay - 1 << 56 | source row position (below)
    uint32_t *ent;
    float *w_out;
    uint32_t *bad;               // set when a synapse cannot be pulled
};

// Sorting key of an incoming synapse: delivery order (delay, source, position
// in the source's row), from which its place in the rows follows.
constexpr int kPullSrcBits = 24, kPullPosBits = 30;
__device__ __forceinline__ uint64_t pull_key(int d, int64_t src, int64_t pos) {
    return ((uint64_t)(d - 1) << (kPullSrcBits + kPullPosBits)) | ((uint64_t)src << kPullPosBits) | (uint64_t)pos;
}

// Counts (FILL false) or places (true) every synapse with its target.
template <bool FILL>
__global__ __launch_bounds__(kBlock) void k_pull_scatter(PullBuild b) {
    const int64_t rows = b.n * b.max_delay;
    for (int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x; r < rows; r += (int64_t)gridDim.x * kBlock) {
        const int64_t q0 = b.row_ptr[r], q1 = b.row_ptr[r + 1];
        if (q0 == q1) continue;
        const int64_t src = r / b.max_delay;
        const int d = (int)(r % b.max_delay) + 1;
        const uint32_t g = b.chunk_group[src / kGroupAlign];
        const int64_t local = src - b.gstart[g];
        for (int64_t q = q0; q < q1; q++) {
            const uint32_t tt = b.tgt_type[q];
            const uint32_t t = tt & 0x3fffffffu;
            if ((tt >> 30) > 1u || (int64_t)t >= b.n || b.chunk_group[t / kGroupAlign] != g || local < 0 ||
                local >= (1ll << kPullSrcBits) || q - q0 >= (1ll << kPullPosBits)) {
                *b.bad = 1u;
                continue;
            }
            const uint32_t at = atomicAdd(&b.deg[t], 1u);
            if (FILL)
                b.key[(b.slice[t / kWave] + at) * kWave + t % kWave] = pull_key(d, local, q - q0);
        }
    }
}

// Longest list of each 64-neuron slice.
__global__ __launch_bounds__(kBlock) void k_pull_slices(const uint32_t *deg, int64_t stride, uint32_t *len) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    uint32_t m = i < stride ? deg[i] : 0u;
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const uint32_t x = (uint32_t)__shfl_xor((int)m, o, kWave);
        m = x > m ? x : m;
    }
    if (i < stride && (threadIdx.x & (kWave - 1)) == 0) len[i / kWave] = m;
}

// One wave per target: its keys sorted in LDS (bitonic, P a power of two), and
// the entries and weights written in that order.
__global__ __launch_bounds__(kBlock) void k_pull_sort(PullBuild b, int64_t stride, int P) {
    extern __shared__ uint64_t s_key[];
    const int lane = threadIdx.x & (kWave - 1);
    uint64_t *k = s_key + (int)(threadIdx.x / kWave) * P;
    const int64_t waves = (int64_t)gridDim.x * kWavesPerBlock;
    for (int64_t t = (int64_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; t < stride; t += waves) {
        const int64_t r0 = b.slice[t / kWave], len = b.slice[t / kWave + 1] - r0;
        const int m = t < b.n ? (int)b.deg[t] : 0;
        const int64_t at = r0 * kWave + t % kWave;
        int pow2 = 1;
        while (pow2 < m) pow2 *= 2;
        for (int j = lane; j < pow2; j += kWave) k[j] = j < m ? b.key[at + (int64_t)j * kWave] : ~0ull;
        for (int size = 2; size <= pow2; size *= 2)
            for (int step = size / 2; step > 0; step /= 2) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                for (int j = lane; j < pow2 / 2; j += kWave) {
                    const int lo = (j / step) * 2 * step + j % step, hi = lo + step;
                    const bool up = (lo & size) == 0;
                    const uint64_t x = k[lo], y = k[hi];
                    if ((x > y) == up) {
                        k[lo] = y;
                        k[hi] = x;
                    }
                }
            }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        int64_t gstart = 0, words = 0;
        if (m > 0) {
            const uint32_t g = b.chunk_group[t / kGroupAlign];
            gstart = b.gstart[g];
            words = (b.gsize[g] + 31) / 32;
        }
        for (int64_t j = lane; j < len; j += kWave) {
            uint32_t e = 0u;
            float x = 0.0f;
            if (j < m) {
                const uint64_t key = k[j];
                const int d = (int)(key >> (kPullSrcBits + kPullPosBits)) + 1;
                const int64_t src = (int64_t)((key >> kPullPosBits) & ((1ull << kPullSrcBits) - 1ull));
                const int64_t q = b.row_ptr[(gstart + src) * b.max_delay + d - 1] +
                                  (int64_t)(key & ((1ull << kPullPosBits) - 1ull));
                e = (uint32_t)(((d - 1) * words + src / 32) * 32 + src % 32) | ((b.tgt_type[q] >> 30) ? kPullType : 0u);
                x = b.w[q];
            } else {
                // padding: the word of zeros after the group's bitmap
                const uint32_t g = b.chunk_group[t / kGroupAlign];
                e = (uint32_t)((int64_t)b.max_delay * ((b.gsize[g] + 31) / 32)) * 32u;
            }
            b.ent[at + j * kWave] = e;
            b.w_out[at + j * kWave] = x;
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Spike bits and counts of the updates in the ring lists (lists built while a
// run is under way).
__global__ __launch_bounds__(kBlock) void k_pull_history(const int32_t *ring_idx, const int32_t *ring_cnt,
                                                         int64_t slot_len, int ring, const uint32_t *chunk_group,
                                                         uint32_t *bits, int64_t words_all, uint32_t *count,
                                                         int groups) {
    for (int s = 0; s < ring; s++) {
        const int32_t m = ring_cnt[s];
        for (int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x; j < m; j += (int64_t)gridDim.x * kBlock) {
            const int32_t id = ring_idx[(int64_t)s * slot_len + j];
            atomicOr(&bits[(int64_t)s * words_all + id / 32], 1u << (id % 32));
            atomicAdd(&count[(int64_t)s * groups + chunk_group[id / kGroupAlign]], 1u);
        }
    }
}

}  // namespace edl
