// kernels.hpp -- the per-step kernels of the time-driven neuron update path.
//
//   k_update     one step of every neuron: optional external drive, ODE step,
//                conductance decay, threshold/reset, NaN reset and ordered
//                spike compaction (one fused pass over the SoA state).
//   k_step_*     a step's Poisson devices, trains, lists, folds and learning, launched together.
//   k_fold_*     ordered conductance accumulation of a step's input events.
#pragma once
#include <type_traits>
#include "device_common.hpp"
#include "device_models.hpp"
#include "event_list.hpp"
#include "eventq.hpp"

namespace edl {

// kBif*: the GPU Bifixed methods -- UpdateArgs::n_sub steps of the base
// method (INTEG - kBifixed) per update, at the sub-step's dt.
enum Integ { kEuler = 0, kRK2 = 1, kRK4 = 2, kBifEuler = 3, kBifRK2 = 4, kBifRK4 = 5 };
constexpr int kBifixed = 3;

// ---------------------------------------------------------------------------
// Ordered conductance accumulation.
//
// Every input event of a step is (key = type*stride + target, order, w); the
// CPU reference adds them one by one into the state, in `order`.  The fold
// reproduces that sequence exactly, for any event density, in one pass over
// the events and a tail in the update kernel:
//
//   events   network mode: each event takes the next free entry of its key's
//            fixed segment of the event buffer; plug-in mode (any number of
//            events per key): event q becomes node q of its key's list.  The
//            target's tile is flagged.
//   update   in flagged tiles each neuron brings its keys' events into order
//            and adds them to the conductance one by one before integrating,
//            then clears the key
//
// The event buffer can hold every event of a step (one per synapse) in the
// network mode, so it cannot overflow there.
// ---------------------------------------------------------------------------
constexpr int kItems = 4;                    // neurons per thread in the update kernels
constexpr int kUpdTile = kBlock * kItems;    // neurons per update tile (kItems per thread)
constexpr int kFlagTile = 512;               // neurons per fold flag (smallest update tile)
constexpr int kBdfBlock = 512;               // threads, and neurons, of a BDF update tile

// One queued event of the fold: its order key and weight in one 16-byte
// entry, so that scattering an event writes one line.
struct FoldEntry {
    uint64_t ord;
    float w;
    uint32_t pad;
};

struct FoldTarget {
    float *state;
    int64_t stride;
    int ndiff;
    uint32_t n_node;     // plug-in mode: the step's events
    uint32_t *fill;      // network mode, per key: events this step
    uint32_t *tile_flag; // per kFlagTile neurons: some key there has an event
    int par;             // parity of this step, unless par_by_step
    int par_by_step;     // parity = update index & 1 (network mode)
    FoldEntry *b_ent;    // network mode: event buffer (order key, weight)
    uint32_t *head;      // plug-in mode, per key: 1 + its last listed event (0: none)
    FoldNode *node;      // plug-in mode: list nodes of the step's events
    // network mode: fixed segment of each key (prefix of the keys' synapse
    // counts; a synapse carries at most one event per step), null otherwise
    const uint64_t *seg_off;
    // network mode with the event queue's order: the rank tables (null:
    // canonical order)
    const struct RankTab *rtab;
};

// Rank of each group of the window that update k consumes, per source,
// [2][delays][cmax] by the parity of k (device memory, one per network).
struct RankTab {
    const uint32_t *rank[4];
    int32_t cmax[4];
    int32_t delays;
};

// Network-mode order key of an event: delay, source, chunk (the group of 1,024
// spiking sources it belongs to, or the input spike's position in its update),
// synapse position.  Sorting by it gives the canonical order (delay, source,
// spiking index, synapse); the event queue's order replaces (delay, source,
// chunk) by the group's rank in its window.
constexpr int kOrdSynBits = 36;
constexpr uint64_t kOrdSynMask = (1ull << kOrdSynBits) - 1ull;
constexpr int kOrdChunkBits = 18;
__host__ __device__ __forceinline__ uint64_t ord_key(int d, int p, uint32_t c, uint64_t q) {
    return ((uint64_t)(d - 1) << 56) | ((uint64_t)p << 54) | ((uint64_t)c << kOrdSynBits) | q;
}

__device__ __forceinline__ float *g_ptr(const FoldTarget &t, uint64_t key) {
    const uint64_t type = key / (uint64_t)t.stride;
    const uint64_t tgt = key - type * (uint64_t)t.stride;
    return t.state + (int64_t)(t.ndiff + (int)type) * t.stride + (int64_t)tgt;
}

// Network mode: the key's fixed segment, next free entry.
__device__ __forceinline__ void fold_event(const FoldTarget &t, uint64_t key, uint64_t ord, float w) {
    const uint32_t pos = atomicAdd(&t.fill[key], 1u);
    const uint64_t at = t.seg_off[key] + pos;
    t.b_ent[at] = FoldEntry{ord, w, 0u};
    if (pos == 0u) t.tile_flag[(key % (uint64_t)t.stride) / kFlagTile] = 1u;
}

// The group rank of an order key, in the window of the update of parity par.
__device__ __forceinline__ uint32_t key_rank(const RankTab *rt, int par, uint64_t o) {
    const int d = (int)(o >> 56) + 1;
    const int p = (int)((o >> 54) & 3u);
    const uint32_t c = (uint32_t)((o >> kOrdSynBits) & ((1u << kOrdChunkBits) - 1u));
    return rt->rank[p][((int64_t)par * rt->delays + (d - 1)) * rt->cmax[p] + c];
}

// A sorting network's exchange of two events.
__device__ __forceinline__ void fold_exchange(uint64_t &ka, float &wa, uint64_t &kb, float &wb) {
    const bool x = kb < ka;
    const uint64_t k = x ? ka : kb;
    const float w = x ? wa : wb;
    ka = x ? kb : ka;
    wa = x ? wb : wa;
    kb = k;
    wb = w;
}

// Adds the m >= 2 events of one key, its segment's first entries e, to g in
// order.  Dependent memory accesses bound it, so every load that can be is
// issued before any is used: up to four events are loaded together, take
// their ranks together and are sorted in registers; more of them take their
// ranks eight at a time (written back) and leave in passes that each find the
// next four.  An insertion sort in place, where each entry waits for its
// predecessor's store, made the update kernel of 1,000 LIF neurons with
// Poisson inputs 14.8 us (now 9.2), of 800 plastic AdEx neurons 19.2 us
// (13.1), of a million AdEx neurons 13.4 us (12.0).
__device__ __attribute__((noinline)) float fold_sorted(FoldEntry *ent, const RankTab *rt, int par, uint32_t m,
                                                       float g) {
    EQ_GLOBAL FoldEntry *e = eq_g(ent);
    // (delay, source, chunk) -> the group's rank in the event queue's window
    const EQ_GLOBAL uint32_t *rank[4] = {nullptr, nullptr, nullptr, nullptr};
    int64_t first[4] = {0, 0, 0, 0};
    int32_t cm[4] = {0, 0, 0, 0};
    if (rt) {
        const EQ_GLOBAL RankTab *t = eq_g(rt);
        const int64_t delays = t->delays;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            rank[p] = eq_g(t->rank[p]);
            cm[p] = t->cmax[p];
            first[p] = (int64_t)par * delays * cm[p];
        }
    }
    auto order = [&](uint64_t o) -> uint64_t {
        if (!rt) return o;
        const int p = (int)((o >> 54) & 3u);
        const int64_t c = (int64_t)((o >> kOrdSynBits) & ((1u << kOrdChunkBits) - 1u));
        const EQ_GLOBAL uint32_t *r = p < 2 ? (p == 0 ? rank[0] : rank[1]) : (p == 2 ? rank[2] : rank[3]);
        const int64_t f = p < 2 ? (p == 0 ? first[0] : first[1]) : (p == 2 ? first[2] : first[3]);
        const int32_t n = p < 2 ? (p == 0 ? cm[0] : cm[1]) : (p == 2 ? cm[2] : cm[3]);
        return ((uint64_t)r[f + (int64_t)(o >> 56) * n + c] << kOrdSynBits) | (o & kOrdSynMask);
    };
    if (m <= 4u) {
        uint64_t k[4];
        float w[4];
#pragma unroll
        for (uint32_t u = 0; u < 4u; u++) {
            const uint32_t j = u < m ? u : 0u;   // entry 0 stands in for the missing ones
            k[u] = e[j].ord;
            w[u] = e[j].w;
        }
#pragma unroll
        for (uint32_t u = 0; u < 4u; u++) k[u] = order(k[u]);
#pragma unroll
        for (uint32_t u = 2; u < 4u; u++) k[u] = u < m ? k[u] : ~0ull;
        fold_exchange(k[0], w[0], k[1], w[1]);
        fold_exchange(k[2], w[2], k[3], w[3]);
        fold_exchange(k[0], w[0], k[2], w[2]);
        fold_exchange(k[1], w[1], k[3], w[3]);
        fold_exchange(k[1], w[1], k[2], w[2]);
        g = g + w[0];
        g = g + w[1];
        if (m > 2u) g = g + w[2];
        if (m > 3u) g = g + w[3];
        return g;
    }
    if (rt) {
        for (uint32_t j0 = 0; j0 < m; j0 += 8u) {
            uint64_t k[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; u++) k[u] = e[j0 + u < m ? j0 + u : 0u].ord;
            // entry 0 may hold its rank already: only for missing ones, unused
#pragma unroll
            for (uint32_t u = 0; u < 8u; u++) k[u] = j0 + u < m ? order(k[u]) : 0ull;
#pragma unroll
            for (uint32_t u = 0; u < 8u; u++)
                if (j0 + u < m) e[j0 + u].ord = k[u];
        }
    }
    // the events after (lk, lj) in the order of key and entry, four a pass
    uint64_t lk = 0;
    uint32_t lj = ~0u;   // none yet
    for (uint32_t done = 0; done < m;) {
        uint64_t b[4] = {~0ull, ~0ull, ~0ull, ~0ull};
        uint32_t bj[4] = {~0u, ~0u, ~0u, ~0u};
        for (uint32_t j0 = 0; j0 < m; j0 += 8u) {
            uint64_t k[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; u++) k[u] = e[j0 + u < m ? j0 + u : 0u].ord;
#pragma unroll
            for (uint32_t u = 0; u < 8u; u++) {
                const uint32_t j = j0 + u;
                const bool left = j < m && (lj == ~0u || k[u] > lk || (k[u] == lk && j > lj));
                // entries come in ascending j, so an equal key stays behind
                if (left && (bj[3] == ~0u || k[u] < b[3])) {
                    b[3] = k[u];
                    bj[3] = j;
#pragma unroll
                    for (int q = 3; q > 0; q--) {
                        const bool x = bj[q - 1] == ~0u || b[q] < b[q - 1];
                        const uint64_t tb = b[q - 1];
                        const uint32_t tj = bj[q - 1];
                        b[q - 1] = x ? b[q] : b[q - 1];
                        bj[q - 1] = x ? bj[q] : bj[q - 1];
                        b[q] = x ? tb : b[q];
                        bj[q] = x ? tj : bj[q];
                    }
                }
            }
        }
        float w[4];
#pragma unroll
        for (int q = 0; q < 4; q++) w[q] = bj[q] != ~0u ? e[bj[q]].w : 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (bj[q] == ~0u) continue;
            g = g + w[q];
            lk = b[q];
            lj = bj[q];
            done++;
        }
    }
    return g;
}

// Plug-in mode: adds the events listed from `hd` to g in the order of their
// numbers, or leaves a long list for fold_list_long.
struct FoldSum {
    float g;
    uint32_t end;   // ListEnd
};
__device__ __attribute__((noinline)) FoldSum fold_list(FoldNode *node, uint32_t n_node, uint32_t hd, float g) {
    const uint32_t end = event_list_add(eq_g(node), n_node, hd, g);
    return FoldSum{g, end};
}
__device__ __attribute__((noinline)) FoldSum fold_list_long(FoldNode *node, uint32_t n_node, uint32_t hd, float g) {
    const uint32_t end = event_list_add_long(eq_g(node), n_node, hd, g);
    return FoldSum{g, end};
}

struct ExtDrive {
    uint64_t seed;
    uint32_t thr[16];  // cumulative thresholds, decreasing
    int n_thr;
    float w;
};

// Grouped populations (many independent networks in one index space): group
// g owns neurons [start, start + n) and its own model parameters.  Groups
// start on multiples of kGroupAlign, so every wave's span of a tile lies in
// one group and the group's parameters are wave-uniform (scalar loads).
struct GroupInfo {
    ModelParams mp;
    int32_t start;
    int32_t n;
};
struct GroupTable {
    const GroupInfo *tab;
    const uint32_t *chunk_group;   // group of each kGroupAlign-neuron chunk
};

struct UpdateArgs {
    float *state;          // SoA, row stride `stride`
    int64_t stride;
    int n;                 // neurons
    int n_tiles;
    StepRef step;          // update index k (>= 1)
    ModelParams mp;
    StepConsts k;
    const float *chan;     // channel-rate table (HH, granule, Purkinje)
    const float *exp_lut;
    const float *nmda_lut;
    const float *refr;
    int refr_len;
    int32_t *last_spike;   // LIF, Purkinje: update (Bifixed: sub-step) index of the last spike
    int n_sub;             // Bifixed kernels: sub-steps per update
    BdfState bdf;          // BDF integrator history
    ExtDrive ext;
    TileOut out;
    FoldTarget fold;       // ordered input fold of this step (multi-event keys)
    GroupTable grp;        // grouped populations only
    // grouped populations that can pull (pull.hpp): spike bits and counts per
    // group by update slot (null: none)
    uint64_t *spk_bits;    // [ring][stride / 64]
    uint32_t *spk_count;   // [ring][groups]
    int ring, groups;
    // timed runs: every workgroup stores its start and end on the device
    // wall clock at clk[((step - clk_first) * gridDim.x + block) * 2 + {0,1}]
    // for steps in [clk_first, clk_first + clk_count) (clk null: untimed)
    unsigned long long *clk;
    int32_t clk_first;
    int32_t clk_count;
};

__device__ __forceinline__ unsigned long long *clock_slot(const UpdateArgs &a, int32_t step) {
    const int32_t k = step - a.clk_first;
    if (!a.clk || k < 0 || k >= a.clk_count) return nullptr;
    return a.clk + ((size_t)k * gridDim.x + blockIdx.x) * 2;
}
__device__ __forceinline__ void clock_begin(const UpdateArgs &a, int32_t step) {
    unsigned long long *c = clock_slot(a, step);
    if (c && threadIdx.x == 0) c[0] = (unsigned long long)wall_clock64();
}
__device__ __forceinline__ void clock_finish(const UpdateArgs &a, int32_t step) {
    unsigned long long *c = clock_slot(a, step);
    if (c) {
        __syncthreads();
        if (threadIdx.x == 0) c[1] = (unsigned long long)wall_clock64();
    }
}

// Reads (and clears) the fold flags covering a tile of T neurons.
template <int T>
__device__ __forceinline__ uint32_t take_tile_flag(uint32_t *flags, int tile) {
    constexpr int F = T / kFlagTile;
    uint32_t f = 0;
#pragma unroll
    for (int q = 0; q < F; q++) f |= flags[tile * F + q];
    return f;
}
template <int T>
__device__ __forceinline__ void clear_tile_flag(uint32_t *flags, int tile) {
    constexpr int F = T / kFlagTile;
#pragma unroll
    for (int q = 0; q < F; q++) flags[tile * F + q] = 0u;
}

// The queued events of a thread's ITEMS neurons, kWave apart from neuron i0,
// added to their conductances g[type] in order.  The fill counts of all keys
// are loaded together, then for each type the segments and the first events
// of all neurons; keys with one event, nearly all of a sparse step's, end
// there.  Each lane then takes its own next key with more, whichever type and
// neuron that is, so a wave calls fold_sorted as often as its busiest lane
// has such keys, not once for every type and neuron that any lane has.  In
// plug-in mode the lanes' listed keys are taken the same way (an update of 1,000
// LIF cells with 125 events 36.4 us; 40.0 us with a call for every type and
// neuron).
template <unsigned MASK, int ITEMS>
__device__ __forceinline__ void fold_keys(const UpdateArgs &a, int32_t step, uint32_t i0, const bool (&live)[ITEMS],
                                          float (&g)[3][ITEMS]) {
    const FoldTarget &t = a.fold;
    uint32_t m[3][ITEMS];
    if (!t.seg_off) {
        uint32_t more = 0u;   // keys with events, by ty * ITEMS + n
#pragma unroll
        for (int ty = 0; ty < 3; ty++)
#pragma unroll
            for (int n = 0; n < ITEMS; n++) {
                m[ty][n] = 0u;
                if (((MASK >> ty) & 1u) && live[n]) m[ty][n] = (t.head + (int64_t)ty * a.stride)[i0 + n * kWave];
            }
#pragma unroll
        for (int q = 0; q < 3 * ITEMS; q++)
            if (m[q / ITEMS][q % ITEMS]) more |= 1u << q;
        while (more) {
            const int x = __builtin_ctz(more);
            more &= more - 1u;
            const uint64_t key = (uint64_t)(x / ITEMS) * (uint64_t)a.stride + (uint64_t)(i0 + (x % ITEMS) * kWave);
            float gx = 0.0f;
            uint32_t hd = 0u;
#pragma unroll
            for (int q = 0; q < 3 * ITEMS; q++) {
                gx = x == q ? g[q / ITEMS][q % ITEMS] : gx;
                hd = x == q ? m[q / ITEMS][q % ITEMS] : hd;
            }
            FoldSum s = fold_list(t.node, t.n_node, hd, gx);
            if (s.end == kListLong) s = fold_list_long(t.node, t.n_node, hd, gx);
            if (s.end != kListDone) atomicOr(a.bdf.err, 4u);
            t.head[key] = 0u;
#pragma unroll
            for (int q = 0; q < 3 * ITEMS; q++) g[q / ITEMS][q % ITEMS] = x == q ? s.g : g[q / ITEMS][q % ITEMS];
        }
        return;
    }
#pragma unroll
    for (int ty = 0; ty < 3; ty++)
#pragma unroll
        for (int n = 0; n < ITEMS; n++) {
            m[ty][n] = 0u;
            if (((MASK >> ty) & 1u) && live[n]) m[ty][n] = (t.fill + (int64_t)ty * a.stride)[i0 + n * kWave];
        }
    uint32_t more = 0u;   // keys of several events, by ty * ITEMS + n
#pragma unroll
    for (int ty = 0; ty < 3; ty++) {
        if (!((MASK >> ty) & 1u)) continue;
        uint64_t b[ITEMS];
        float w[ITEMS];
#pragma unroll
        for (int n = 0; n < ITEMS; n++) {
            b[n] = 0;
            if (m[ty][n] == 1u) b[n] = (t.seg_off + (int64_t)ty * a.stride)[i0 + n * kWave];
        }
#pragma unroll
        for (int n = 0; n < ITEMS; n++) {
            w[n] = 0.0f;
            if (m[ty][n] == 1u) w[n] = t.b_ent[b[n]].w;
        }
#pragma unroll
        for (int n = 0; n < ITEMS; n++) {
            if (m[ty][n] == 1u) {
                (t.fill + (int64_t)ty * a.stride)[i0 + n * kWave] = 0u;
                g[ty][n] = g[ty][n] + w[n];
            }
            if (m[ty][n] > 1u) more |= 1u << (ty * ITEMS + n);
        }
    }
    while (more) {
        const int x = __builtin_ctz(more);
        more &= more - 1u;
        const uint64_t key = (uint64_t)(x / ITEMS) * (uint64_t)a.stride + (uint64_t)(i0 + (x % ITEMS) * kWave);
        float gx = 0.0f;
        uint32_t mx = 0u;
#pragma unroll
        for (int q = 0; q < 3 * ITEMS; q++) {
            gx = x == q ? g[q / ITEMS][q % ITEMS] : gx;
            mx = x == q ? m[q / ITEMS][q % ITEMS] : mx;
        }
        gx = fold_sorted(t.b_ent + t.seg_off[key], t.rtab, step & 1, mx, gx);
        t.fill[key] = 0u;
#pragma unroll
        for (int q = 0; q < 3 * ITEMS; q++) g[q / ITEMS][q % ITEMS] = x == q ? gx : g[q / ITEMS][q % ITEMS];
    }
}

// One tile = kBlock*ITEMS neurons in the wave-major layout of tile_neuron:
// each lane handles ITEMS neurons kWave apart (each item is one coalesced row
// access per wave).  All loads are issued first, the ITEMS neurons are
// integrated stage-major, and the stores come last, so every thread keeps
// ITEMS independent dependency chains in flight.  GROUPED takes the model
// parameters, the live range and the drive seed from the wave's group.
template <class M, int INTEG, unsigned MASK, bool EXT, int ITEMS, bool GROUPED>
__global__ __launch_bounds__(kBlock) void k_update(UpdateArgs a) {
    constexpr int T = kBlock * ITEMS;
    static_assert(T % kFlagTile == 0, "update tiles cover whole fold flags");
    static_assert(kGroupAlign % (ITEMS * kWave) == 0, "a wave's span lies in one group");
    const int tile = blockIdx.x;
    const int32_t step = a.step.get();
    clock_begin(a, step);
    __shared__ uint32_t s_flag;
    // the tile's fold flag is read alongside the state loads (the barrier
    // that publishes it comes after them)
    uint32_t flag = 0;
    if (threadIdx.x == 0) flag = take_tile_flag<T>(a.fold.tile_flag, tile);
    ModelParams gmp;
    int32_t gstart = 0, gn = a.n;
    uint64_t dseed = a.ext.seed;
    if (GROUPED) {
        const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
        const int first = tile * T + wid * ITEMS * kWave;
        const uint32_t g = a.grp.chunk_group[first / kGroupAlign];
        gmp = a.grp.tab[g].mp;
        gstart = a.grp.tab[g].start;
        gn = a.grp.tab[g].n;
        dseed = a.ext.seed + g;
    }
    const ModelParams &mp = GROUPED ? gmp : a.mp;
    // one row pointer per state variable (uniform), 32-bit neuron offsets
    float *__restrict__ row[M::NV];
#pragma unroll
    for (int j = 0; j < M::NV; j++) row[j] = a.state + (int64_t)j * a.stride;
    const uint32_t step_key = EXT ? drive_step_key(dseed, step) : 0u;
    int idx[ITEMS];
    bool live[ITEMS];
    float s[ITEMS][M::NV];
    RhsCtx c[ITEMS];
#pragma unroll
    for (int n = 0; n < ITEMS; n++) {
        idx[n] = tile_neuron<ITEMS>(tile, n);
        live[n] = idx[n] - gstart < gn;
        // rows are padded to a multiple of kUpdTile, so the loads stay in bounds
        const uint32_t i = (uint32_t)idx[n];
#pragma unroll
        for (int j = 0; j < M::ND; j++) s[n][j] = row[j][i];
        s[n][M::EXC] = (MASK & 1u) ? row[M::EXC][i] : 0.0f;
        s[n][M::INH] = (MASK & 2u) ? row[M::INH][i] : 0.0f;
        s[n][M::NMDA] = (MASK & 4u) ? row[M::NMDA][i] : 0.0f;
        s[n][M::EXT] = (MASK & 8u) ? row[M::EXT][i] : 0.0f;
        c[n].chan = a.chan;
        c[n].exp_lut = a.exp_lut;
        c[n].nmda_lut = a.nmda_lut;
        c[n].refr = a.refr;
        c[n].refr_len = a.refr_len;
        c[n].since_spike = a.last_spike ? (step - 1 - a.last_spike[i]) : (1 << 30);
    }
    if (threadIdx.x == 0) {
        s_flag = flag;
        if (flag) clear_tile_flag<T>(a.fold.tile_flag, tile);
    }
    __syncthreads();
    if (s_flag) {
        // the step's input events, in delivery order
        float g[3][ITEMS];
#pragma unroll
        for (int n = 0; n < ITEMS; n++)
#pragma unroll
            for (int ty = 0; ty < 3; ty++) g[ty][n] = s[n][M::EXC + ty];
        fold_keys<MASK, ITEMS>(a, step, (uint32_t)idx[0], live, g);
#pragma unroll
        for (int n = 0; n < ITEMS; n++)
#pragma unroll
            for (int ty = 0; ty < 3; ty++) s[n][M::EXC + ty] = g[ty][n];
    }
    if (EXT) {
        // External drive events of this interval, after the recurrent ones;
        // the hash takes the neuron's index within its group.  The event
        // count is #{j : u < thr[j]} (thresholds decrease); the loop walks
        // the thresholds in wave-uniform order and stops once no lane hits.
        uint32_t u[ITEMS];
        int cnt[ITEMS];
#pragma unroll
        for (int n = 0; n < ITEMS; n++) {
            u[n] = drive_hash_keyed(step_key, (uint32_t)(idx[n] - gstart));
            cnt[n] = 0;
        }
        for (int j = 0; j < a.ext.n_thr; j++) {
            const uint32_t t = a.ext.thr[j];
            bool hit = false;
#pragma unroll
            for (int n = 0; n < ITEMS; n++) {
                const bool h = u[n] < t;
                cnt[n] += h ? 1 : 0;
                hit = hit || h;
            }
            if (!__any(hit)) break;
        }
#pragma unroll
        for (int n = 0; n < ITEMS; n++)
            for (int q = 0; q < cnt[n]; q++) s[n][M::EXC] += a.ext.w;
    }
    // Fixed methods take one step.  The Bifixed methods take n_sub steps of
    // the base method, each followed by the spike condition, and report a
    // neuron once per update (Bifixed_RK4_GPU2.cuh:100-150); their spike clock
    // counts sub-steps, numbered from 1 over the run (update k covers
    // (k-1)*n_sub+1 .. k*n_sub), and the clock tables are built for the
    // sub-step.
    constexpr bool SUB = INTEG >= kBifixed;
    constexpr int BASE = SUB ? INTEG - kBifixed : INTEG;
    const int n_sub = SUB ? a.n_sub : 1;
    const int32_t g0 = SUB ? (step - 1) * n_sub : step - 1;
    bool spk[ITEMS];
    int32_t last[ITEMS];
#pragma unroll
    for (int n = 0; n < ITEMS; n++) {
        spk[n] = false;
        last[n] = (SUB && a.last_spike) ? a.last_spike[(uint32_t)idx[n]] : 0;
    }
    for (int it = 0; it < n_sub; it++) {
        const int32_t g = g0 + it + 1;
        float prev_v[ITEMS];
#pragma unroll
        for (int n = 0; n < ITEMS; n++) {
            if (SUB && a.last_spike) c[n].since_spike = g - 1 - last[n];
            prev_v[n] = s[n][0];
        }
        if (BASE == kEuler) integrate_euler<M, MASK, ITEMS>(mp, c, a.k, s);
        else if (BASE == kRK2) integrate_rk2<M, MASK, ITEMS>(mp, c, a.k, s);
        else integrate_rk4<M, MASK, ITEMS>(mp, c, a.k, s);
#pragma unroll
        for (int n = 0; n < ITEMS; n++) {
            const bool f = live[n] && M::spike(mp, prev_v[n], s[n]);
            if constexpr (M::kClockOverride)
                if (live[n]) M::clock_override(c[n], f, s[n]);
            if (f) {
                spk[n] = true;
                last[n] = g;
            }
        }
    }

#pragma unroll
    for (int n = 0; n < ITEMS; n++) {
        const uint32_t i = (uint32_t)idx[n];
        if (!live[n]) continue;
        if (spk[n] && a.last_spike) a.last_spike[i] = last[n];
        if (s[n][0] != s[n][0]) {
            // TimeDrivenNeuronModel.cpp:75-88: NaN -> whole state to initial.
#pragma unroll
            for (int j = 0; j < M::NV; j++) row[j][i] = M::init(mp, j);
        } else {
            // non-temporal stores: the next reader is the next step's
            // update, so the rows need not stay in L2 (and the end-of-kernel
            // write-back has less to do): 13.7 us per 1M-neuron AdEx launch
            // against 14.0 us with ordinary stores
#pragma unroll
            for (int j = 0; j < M::ND; j++) __builtin_nontemporal_store(s[n][j], &row[j][i]);
            if (MASK & 1u) __builtin_nontemporal_store(s[n][M::EXC], &row[M::EXC][i]);
            if (MASK & 2u) __builtin_nontemporal_store(s[n][M::INH], &row[M::INH][i]);
            if (MASK & 4u) __builtin_nontemporal_store(s[n][M::NMDA], &row[M::NMDA][i]);
        }
    }
    if (GROUPED && a.spk_bits) {
        const int slot = step % a.ring;
        uint32_t total = 0;
#pragma unroll
        for (int n = 0; n < ITEMS; n++) {
            const uint64_t m = __ballot(spk[n]);
            total += (uint32_t)__popcll(m);
            if ((threadIdx.x & (kWave - 1)) == 0) a.spk_bits[slot * (a.stride / kWave) + idx[n] / kWave] = m;
        }
        if ((threadIdx.x & (kWave - 1)) == 0 && total)
            atomicAdd(&a.spk_count[(int64_t)slot * a.groups + a.grp.chunk_group[idx[0] / kGroupAlign]], total);
    }
    tile_spikes<ITEMS>(a.out, tile, spk, idx);
    clock_finish(a, step);
}


// Loads the state of neuron i at the start of a BDF step into sf: the row
// values, the ordered fold of its multi-event keys when its tile's fold flag
// is set, and the external drive.
template <class M, unsigned MASK, bool EXT>
__device__ __forceinline__ void bdf_load(const UpdateArgs &a, float *__restrict__ const *row, int32_t step,
                                         uint32_t step_key, uint32_t flag, uint32_t i, float *sf) {
#pragma unroll
    for (int j = 0; j < M::ND; j++) sf[j] = row[j][i];
    sf[M::EXC] = (MASK & 1u) ? row[M::EXC][i] : 0.0f;
    sf[M::INH] = (MASK & 2u) ? row[M::INH][i] : 0.0f;
    sf[M::NMDA] = (MASK & 4u) ? row[M::NMDA][i] : 0.0f;
    sf[M::EXT] = (MASK & 8u) ? row[M::EXT][i] : 0.0f;
    if (flag) {
        const bool live[1] = {true};
        float g[3][1];
#pragma unroll
        for (int ty = 0; ty < 3; ty++) g[ty][0] = sf[M::EXC + ty];
        fold_keys<MASK, 1>(a, step, i, live, g);
#pragma unroll
        for (int ty = 0; ty < 3; ty++) sf[M::EXC + ty] = g[ty][0];
    }
    if (EXT) {
        const uint32_t u = drive_hash_keyed(step_key, i);
        int cnt = 0;
        while (cnt < a.ext.n_thr && u < a.ext.thr[cnt]) cnt++;
        for (int q = 0; q < cnt; q++) sf[M::EXC] += a.ext.w;
    }
}

// Stores neuron i's state after the step (TimeDrivenNeuronModel.cpp:75-88:
// a NaN membrane potential puts the whole state back to its initial values).
template <class M, unsigned MASK>
__device__ __forceinline__ void bdf_store(const UpdateArgs &a, float *__restrict__ const *row, uint32_t i,
                                          const float *out) {
    if (out[0] != out[0]) {
#pragma unroll
        for (int j = 0; j < M::NV; j++) row[j][i] = M::init(a.mp, j);
    } else {
#pragma unroll
        for (int j = 0; j < M::ND; j++) row[j][i] = out[j];
        if (MASK & 1u) row[M::EXC][i] = out[M::EXC];
        if (MASK & 2u) row[M::INH][i] = out[M::INH];
        if (MASK & 4u) row[M::NMDA][i] = out[M::NMDA];
    }
}

// BDF update: one neuron per thread (the Newton iteration is a serial chain of
// data-dependent length, so a second neuron on the thread doubles the kernel
// wherever the population leaves SIMDs idle).  T = double runs the whole BDF
// step in double (FP64 Newton mode); the state is stored back in float.
// 4,099 HH cells, FP64 Newton: 41 us per launch; with four neurons on each of 256
// threads 109 us.
template <class M, unsigned MASK, bool EXT, typename T>
__global__ __launch_bounds__(kBdfBlock) void k_update_bdf(UpdateArgs a) {
    constexpr int TILE = kBdfBlock;
    static_assert(TILE % kFlagTile == 0, "update tiles cover whole fold flags");
    const int tile = blockIdx.x;
    const int32_t step = a.step.get();
    clock_begin(a, step);
    __shared__ uint32_t s_flag;
    if (threadIdx.x == 0) {
        s_flag = take_tile_flag<TILE>(a.fold.tile_flag, tile);
        if (s_flag) clear_tile_flag<TILE>(a.fold.tile_flag, tile);
    }
    __syncthreads();
    float *__restrict__ row[M::NV];
#pragma unroll
    for (int j = 0; j < M::NV; j++) row[j] = a.state + (int64_t)j * a.stride;
    const int64_t ld = a.stride;
    const uint32_t step_key = EXT ? drive_step_key(a.ext.seed, step) : 0u;
    const int idx = tile * TILE + (int)threadIdx.x;
    bool spk = false;
    if (idx < a.n) {
        const uint32_t i = (uint32_t)idx;
        float sf[M::NV];
        bdf_load<M, MASK, EXT>(a, row, step, step_key, s_flag, i, sf);
        T S[M::NV];
#pragma unroll
        for (int j = 0; j < M::NV; j++) S[j] = sf[j];
        const T prev = S[0];
        RhsCtx c;
        c.chan = a.chan;
        c.exp_lut = a.exp_lut;
        c.nmda_lut = a.nmda_lut;
        c.refr = a.refr;
        c.refr_len = a.refr_len;
        c.since_spike = a.last_spike ? (step - 1 - a.last_spike[i]) : (1 << 30);
        int st = a.bdf.st[i];
        integrate_bdf<M, MASK, T>(a.mp, c, (T)a.k.dt, a.bdf, ld, i, st, S);
        spk = M::spike(a.mp, prev, S);
        if constexpr (M::kClockOverride) M::clock_override(c, spk, S);
        if (spk && M::kResetsIntegrator) st = 0;
        a.bdf.st[i] = st;
        if (spk && a.last_spike) a.last_spike[i] = step;
        float out[M::NV];
#pragma unroll
        for (int j = 0; j < M::NV; j++) out[j] = (float)S[j];
        bdf_store<M, MASK>(a, row, i, out);
    }
    tile_spikes<1, kBdfBlock>(a.out, tile, &spk, &idx);
    clock_finish(a, step);
}

// ---------------------------------------------------------------------------
// Poisson generator device (PoissonGeneratorDeviceVector.cpp:56-70): per
// source, if rate > 0 draw the next frand() of its LCG
// (RandomGenerator.h:61-107) and fire when rate*step (double) exceeds it.
// ---------------------------------------------------------------------------
struct PoissonArgs {
    uint32_t *lcg;
    int n;
    int n_tiles;
    float rate;             // frequency of every generator (Hz) when rates is null
    const float *rates;     // per-generator frequencies (PoissonGeneratorDeviceVector)
    double step_s;          // time-driven step (s)
    TileOut out;
};

__device__ __forceinline__ void poisson_body(const PoissonArgs &a, int tile) {
    bool spk[1] = {false};
    int idx[1] = {tile * kBlock + (int)threadIdx.x};
    const int i = idx[0];
    const float f = (i < a.n && a.rates) ? a.rates[i] : a.rate;
    if (i < a.n && f > 0.0f) {
        uint32_t x = a.lcg[i];
        x = (uint32_t)(((uint64_t)x * 1103515245ull + 12345ull) & 0x7fffffffull);
        a.lcg[i] = x;
        const float u = ((float)x) / 2147483647.0f;
        spk[0] = (double)f * a.step_s > (double)u;
    }
    tile_spikes<1>(a.out, tile, spk, idx);
}

// ---------------------------------------------------------------------------
// Spike-train source: input neurons (InputSpikeNeuronModel driven by
// FileInputSpikeDriver.cpp:45-85 or Simulation_API::AddExternalSpikeActivity)
// whose spikes the host has placed on update steps.  Update k copies its
// ascending, duplicate-free list idx[ptr[k-1] .. ptr[k]) into ring slot
// k % ring; steps past the train have no spikes.
// ---------------------------------------------------------------------------
struct TrainArgs {
    const int64_t *ptr;     // [n_steps + 1]
    const int32_t *idx;
    int64_t n_steps;
    int32_t *ring_idx;      // [ring][n_src]
    int32_t *ring_cnt;      // [ring]
    int64_t n_src;
    int ring;
    StepRef step;
};

__device__ __forceinline__ void train_body(const TrainArgs &a, int bid, int nb) {
    const int32_t k = a.step.get();
    const int slot = k % a.ring;
    int64_t b = 0, e = 0;
    if (k >= 1 && (int64_t)k <= a.n_steps) {
        b = a.ptr[k - 1];
        e = a.ptr[k];
    }
    int32_t *out = a.ring_idx + (int64_t)slot * a.n_src;
    for (int64_t j = b + (int64_t)bid * kBlock + threadIdx.x; j < e; j += (int64_t)nb * kBlock) out[j - b] = a.idx[j];
    if (bid == 0 && threadIdx.x == 0) a.ring_cnt[slot] = (int32_t)(e - b);
}

// Events pushed by the host (read from its pinned buffer) or handed over in
// device memory: order = position in the list.  They are checked here (target
// in range, synapse type enabled); one that fails is dropped and sets err bit
// 8 (the host's own were checked when they were queued).
struct PushEvents {
    const int32_t *tgt;
    const uint8_t *type;
    const float *w;
    int n;
    int32_t n_tgt;
    uint32_t mask;       // enabled synapse types taking spikes (bits 0-2)
    uint32_t *err;
};

__global__ __launch_bounds__(kBlock) void k_fold_push(FoldTarget t, PushEvents e) {
    for (int q = blockIdx.x * kBlock + threadIdx.x; q < e.n; q += gridDim.x * kBlock) {
        const int32_t tg = e.tgt[q];
        const uint32_t ty = e.type[q];
        const float w = e.w[q];
        if ((uint32_t)tg >= (uint32_t)e.n_tgt || ty > 2u || !((e.mask >> ty) & 1u)) {
            atomicOr(e.err, 256u);
            continue;
        }
        const uint32_t prev = atomicExch(&t.head[(uint64_t)ty * (uint64_t)t.stride + (uint64_t)tg], (uint32_t)q + 1u);
        t.node[q] = FoldNode{prev, w};
        t.tile_flag[(uint32_t)tg / (uint32_t)kFlagTile] = 1u;
    }
}

// Events generated on the device from the spike rings of the sources.
constexpr int kMaxSources = 4;
constexpr int kMaxDelay = 256;
// Additive STDP on the synapses of a source (STDPWeightChange / STDPState):
// per synapse a presynaptic and a postsynaptic trace and the time of its
// last update; weights change in place.
struct StdpSyn {
    float *pre;
    float *post;
    double *last;
    float a_plus, a_minus;           // max_LTP, max_LTD
    float inv_tau_plus, inv_tau_minus;
    float w_max;
};

struct RingSource {
    const int32_t *ring_idx;   // [ring][n_src]
    const int32_t *ring_cnt;   // [ring]
    const int64_t *row_ptr;    // [n_src*max_delay+1]
    const uint32_t *tgt_type;  // target | type << 30
    float *w;
    int64_t n_src;
    int stdp;                  // plastic synapses (StdpSyn below)
    StdpSyn syn;
    // groups of 1,024 spiking sources (the reference's PropagatedSpikeGroup):
    // the chunk of a list entry is its position / 1024 unless bnd_on[slot],
    // then the number of chunks whose last member comes before it
    // (bnd [ring][max_delay][cmax]); a spike train's events are one per spike
    int train;
    const int32_t *bnd;
    const uint8_t *bnd_on;
    int32_t cmax;
    int poisson;               // a Poisson device: its groups' times are on its own clock
};
struct RingEvents {
    RingSource src[kMaxSources];
    int n_sources;
    int max_delay;
    int ring;
    StepRef step;              // update index about to run
    // STDP only: update time of each ring slot (populations; Poisson
    // devices on their own 0.1 ms clock), delay of d steps in seconds
    const double *time_ring;   // [ring]
    const double *time_ring_p; // [ring]
    const double *delay_s;     // [max_delay + 1]
    const float *exp_lut;
    // a run that stops inside a window delivers the groups ranked before its
    // stop event at its end (rank_hi) and the rest with the next update:
    // that update's fold skips the groups ranked below skip[1] when the
    // update is skip[0] (device memory, set by the host); rtab null: all
    const RankTab *rtab;
    const uint32_t *skip;
    uint32_t rank_hi;
    // groups whose events are pulled (pull.hpp), [2][groups] by update parity,
    // and the group of each kGroupAlign-neuron chunk (null: none)
    const uint8_t *pulled;
    const uint32_t *chunk_group;
    int groups;
};

// STDPState::SetNewUpdateTime (STDPState.cpp:74-82): both traces decay by
// ExponentialTable factors of the float elapsed time.
__device__ __forceinline__ void stdp_decay(const StdpSyn &s, const float *exp_lut, int64_t q, double t) {
    const float elapsed = (float)(t - s.last[q]);
    s.pre[q] = s.pre[q] * lut_exp(exp_lut, -elapsed * s.inv_tau_plus);
    s.post[q] = s.post[q] * lut_exp(exp_lut, -elapsed * s.inv_tau_minus);
    s.last[q] = t;
}
// Interconnection::IncrementWeight (Interconnection.h:400-409)
__device__ __forceinline__ void stdp_increment(const StdpSyn &s, float *w, int64_t q, float inc) {
    float x = w[q] + inc;
    if (x > s.w_max) x = s.w_max;
    else if (x < 0.0f) x = 0.0f;
    w[q] = x;
}

// Work item = one spike of one source at emission step k-1-d; a group of
// LANES lanes walks its synapses of delay d.  Items are enumerated in
// (d, source, rank) order from a prefix over the per-(d, source) counts.
// The order key (ord_key) holds delay, source, chunk and synapse position;
// within a group the synapse position rises with the source index and then
// the target index, which is the reference's delivery order in a group.
// PULL: a wave looks 64 items up at once and leaves out the pulled groups'.
// FIXED lanes (a power of two) or, where it is 0, `lanes`.
struct FoldLds {
    int64_t pref[kMaxDelay * kMaxSources + 1];
    int slot[kMaxDelay * kMaxSources];
};
__device__ __forceinline__ FoldLds &fold_lds() {
    __shared__ FoldLds s;
    return s;
}
template <int FIXED, bool PULL>
__device__ __forceinline__ void fold_ring_body(const FoldTarget &t, const RingEvents &r, int bid, int nb,
                                               int lanes = FIXED) {
    const int LANES = FIXED > 0 ? FIXED : lanes;
    const int shift = __builtin_ctz((unsigned)LANES);
    int64_t *const s_pref = fold_lds().pref;
    int *const s_slot = fold_lds().slot;
    const int nseg = r.max_delay * r.n_sources;
    const int32_t step = r.step.get();
    const uint32_t rank_lo = (r.rtab && r.skip && r.skip[0] == (uint32_t)step) ? r.skip[1] : 0u;
    for (int g = threadIdx.x; g < nseg; g += kBlock) {
        const int d = g / r.n_sources + 1;
        const int p = g % r.n_sources;
        const int64_t s = (int64_t)step - 1 - d;
        int slot = 0, c = 0;
        if (s >= 1) {
            slot = (int)(s % r.ring);
            c = r.src[p].ring_cnt[slot];
        }
        s_slot[g] = slot;
        s_pref[g + 1] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        s_pref[0] = 0;
        for (int g = 0; g < nseg; g++) s_pref[g + 1] += s_pref[g];
    }
    __syncthreads();
    const int64_t n_items = s_pref[nseg];
    if (PULL) {
        // a grouped population's own spikes in the canonical order (a single
        // source, no STDP)
        const RingSource &src = r.src[0];
        const uint8_t *pulled = r.pulled + (int64_t)(step & 1) * r.groups;
        const int wl = threadIdx.x & (kWave - 1);
        const int64_t wave = (int64_t)bid * kWavesPerBlock + threadIdx.x / kWave;
        for (int64_t it0 = wave * kWave; it0 < n_items; it0 += (int64_t)nb * kBlock) {
            const int64_t it = it0 + wl;
            int64_t b = 0, e = 0;
            uint64_t ord = 0;
            if (it < n_items) {
                int lo = 0, hi = nseg - 1;
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (s_pref[mid] <= it) lo = mid;
                    else hi = mid - 1;
                }
                const int64_t rank = it - s_pref[lo];
                const int32_t id = src.ring_idx[(int64_t)s_slot[lo] * src.n_src + rank];
                if (!pulled[r.chunk_group[id / kGroupAlign]]) {
                    b = src.row_ptr[(int64_t)id * r.max_delay + lo];
                    e = src.row_ptr[(int64_t)id * r.max_delay + lo + 1];
                    ord = ord_key(lo + 1, 0, s_pref[lo + 1] - s_pref[lo] >= 1024 ? (uint32_t)(rank >> 10) : 0u, 0);
                }
            }
            uint64_t live = __ballot(b < e);
            while (live) {
                // one item per group of LANES lanes
                int from = -1;
                for (int u = 0; u < (kWave >> shift) && live; u++) {
                    if ((wl >> shift) == u) from = __builtin_ctzll(live);
                    live &= live - 1ull;
                }
                const int f = from < 0 ? 0 : from;
                const int64_t fb = __shfl(b, f), fe = __shfl(e, f);
                const uint64_t fo = __shfl(ord, f);
                for (int64_t q = fb + (wl & (LANES - 1)); from >= 0 && q < fe; q += LANES) {
                    const uint32_t tt = src.tgt_type[q];
                    fold_event(t, (uint64_t)(tt >> 30) * (uint64_t)t.stride + (uint64_t)(tt & 0x3fffffffu),
                               fo | (uint64_t)q, src.w[q]);
                }
            }
        }
        return;
    }
    const int lane = (int)threadIdx.x & (LANES - 1);
    const int64_t group = (int64_t)(bid * kBlock + (int)threadIdx.x) >> shift;
    const int64_t n_groups = (int64_t)nb * kBlock >> shift;
    for (int64_t it = group; it < n_items; it += n_groups) {
        // last segment g with s_pref[g] <= it (segments may be empty)
        int lo = 0, hi = nseg - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (s_pref[mid] <= it) lo = mid;
            else hi = mid - 1;
        }
        const int g = lo;
        const int d = g / r.n_sources + 1;
        const int p = g % r.n_sources;
        const RingSource &src = r.src[p];
        const int64_t rank = it - s_pref[g];
        const int32_t id = src.ring_idx[(int64_t)s_slot[g] * src.n_src + rank];
        const int64_t b = src.row_ptr[(int64_t)id * r.max_delay + d - 1];
        const int64_t e = src.row_ptr[(int64_t)id * r.max_delay + d];
        uint32_t chunk = 0;
        if (src.train) {
            chunk = (uint32_t)rank;
        } else if (s_pref[g + 1] - s_pref[g] >= 1024) {
            const int slot = s_slot[g];
            if (src.bnd_on && src.bnd_on[slot]) {
                const int32_t *bd = src.bnd + ((int64_t)slot * r.max_delay + (d - 1)) * src.cmax;
                while ((int32_t)chunk < src.cmax && bd[chunk] < rank) chunk++;
            } else {
                chunk = (uint32_t)(rank >> 10);
            }
        }
        const uint64_t ord_hi = ord_key(d, p, chunk, 0);
        if (rank_lo > 0u || r.rank_hi != 0xffffffffu) {
            const uint32_t rk = key_rank(r.rtab, step & 1, ord_hi);
            if (rk < rank_lo || rk >= r.rank_hi) continue;
        }
        double t_arr = 0.0;
        if (src.stdp)
            t_arr = (src.poisson ? r.time_ring_p[s_slot[g]] : r.time_ring[s_slot[g]]) + r.delay_s[d];
        for (int64_t q = b + lane; q < e; q += LANES) {
            const uint32_t tt = src.tgt_type[q];
            const uint64_t key =
                (uint64_t)(tt >> 30) * (uint64_t)t.stride + (uint64_t)(tt & 0x3fffffffu);
            fold_event(t, key, ord_hi | (uint64_t)q, src.w[q]);
            if (src.stdp) {
                // STDPWeightChange::ApplyPreSynapticSpike (STDPWeightChange.cpp:43-55),
                // after the event used the weight (PropagatedSpikeGroup.cpp:76-97).
                // A synapse carries at most one event per step: no other lane
                // touches q.
                stdp_decay(src.syn, r.exp_lut, q, t_arr);
                src.syn.pre[q] = src.syn.pre[q] + 1.0f;
                stdp_increment(src.syn, src.w, q, -src.syn.a_minus * src.syn.post[q]);
            }
        }
    }
}

template <int LANES, bool PULL = false>
__global__ __launch_bounds__(kBlock) void k_fold_ring(FoldTarget t, RingEvents r) {
    fold_ring_body<LANES, PULL>(t, r, blockIdx.x, gridDim.x);
}

// Compaction of update k's spikes and the fold of the events update k + 1
// consumes, in one launch (network mode without STDP): the fold reads the
// spike lists of updates <= k - 1 only, and the fold buffers it fills were
// drained by update k.  Workgroups [0, nb_compact) compact, the rest fold.
template <int LANES, bool PULL = false>
__global__ __launch_bounds__(kBlock) void k_compact_fold(CompactArgs c, FoldTarget t, RingEvents r,
                                                         int nb_compact) {
    clock_next_kernel(c);
    if ((int)blockIdx.x < nb_compact) compact_body(c, blockIdx.x, nb_compact);
    else fold_ring_body<LANES, PULL>(t, r, blockIdx.x - nb_compact, gridDim.x - nb_compact);
}

// The same with the event-queue replay of update k's window in the first
// workgroup (its chain of dependent steps is the longest): it reads update
// k's spikes from the update kernel's tiles, so it depends on nothing the
// other workgroups write and runs beside them.
template <int LANES, int ITEMS>
__global__ __launch_bounds__(kBlock) void k_compact_fold_eq(CompactArgs c, FoldTarget t, RingEvents r,
                                                            int nb_compact, EqArgs q) {
    clock_next_kernel(c);
    const int b = (int)blockIdx.x - 1;
    if (b < 0) eq_body<ITEMS, kEqFusedDelays>(q);
    else if (b < nb_compact) compact_body(c, b, nb_compact);
    else fold_ring_body<LANES, false>(t, r, b - nb_compact, (int)gridDim.x - 1 - nb_compact);
}

// Synapses per (type, target) key of one source, for the fixed segments of
// the network-mode fold.
__global__ __launch_bounds__(kBlock) void k_key_degree(const uint32_t *tgt_type, int64_t nsyn, int64_t stride,
                                                       uint32_t *deg) {
    for (int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x; q < nsyn; q += (int64_t)gridDim.x * kBlock) {
        const uint32_t tt = tgt_type[q];
        atomicAdd(&deg[(uint64_t)(tt >> 30) * (uint64_t)stride + (tt & 0x3fffffffu)], 1u);
    }
}

// ---------------------------------------------------------------------------
// Post-synaptic STDP (STDPWeightChange::ApplyPostSynapticSpike,
// STDPWeightChange.cpp:57-76, called for every neuron that fired at update k,
// TimeDrivenInternalSpike.cpp:94-103): every plastic input synapse of a
// spiking neuron decays to the update time, gains a postsynaptic trace unit
// and potentiates by max_LTP times its presynaptic trace (in_syn lists
// synapse positions by target).
// ---------------------------------------------------------------------------
struct StdpPostArgs {
    const int32_t *spk_idx;    // own spike ring, slot k % ring
    const int32_t *spk_cnt;
    int64_t slot_len;
    int ring;
    StepRef step;
    const int64_t *in_ptr;     // [n_tgt + 1]
    const int64_t *in_syn;     // synapse positions grouped by target
    int chunks;                // kWave-synapse chunks of the longest list
    float *w;
    StdpSyn syn;
    const double *time_ring;
    const float *exp_lut;
};

// Post-synaptic learning of the neurons that fired at update k: every
// incoming synapse of each of them.  A work
// item is one wave-sized chunk of one neuron's list, so a neuron with 2,000
// inputs is spread over 32 waves rather than walked by one; the synapses are
// distinct, so the order of their updates does not matter.
__device__ __forceinline__ void stdp_post_body(const StdpPostArgs &a, int bid, int nb) {
    const int32_t step = a.step.get();
    const int slot = step % a.ring;
    const int64_t n = a.spk_cnt[slot];
    const int32_t *ids = a.spk_idx + (int64_t)slot * a.slot_len;
    const double tk = a.time_ring[slot];
    const int lane = threadIdx.x % kWave;
    const int64_t wave = (int64_t)(bid * kBlock + (int)threadIdx.x) / kWave;
    const int64_t n_waves = (int64_t)nb * kBlock / kWave;
    for (int64_t it = wave; it < n * a.chunks; it += n_waves) {
        const int32_t i = ids[it / a.chunks];
        const int64_t x = a.in_ptr[i] + (it % a.chunks) * kWave + lane;
        if (x < a.in_ptr[i + 1]) {
            const int64_t q = a.in_syn[x];
            stdp_decay(a.syn, a.exp_lut, q, tk);
            a.syn.post[q] = a.syn.post[q] + 1.0f;
            stdp_increment(a.syn, a.w, q, a.syn.a_plus * a.syn.pre[q]);
        }
    }
}

// Update time of step k: t_k = t_{k-1} + double(float dt), kept per ring slot
// (TimeEventUpdateNeurons.cpp:78), for plastic networks.  The Poisson devices'
// clock advances by their own step in a second ring.
struct TickArgs {
    double *time_ring;     // [ring]
    double *time_ring_p;
    int ring;
    double dt, dt_p;
};

__device__ __forceinline__ void tick_body(const TickArgs &a, int32_t k) {
    if (threadIdx.x == 0) {
        a.time_ring[k % a.ring] = a.time_ring[(k - 1) % a.ring] + a.dt;
        a.time_ring_p[k % a.ring] = a.time_ring_p[(k - 1) % a.ring] + a.dt_p;
    }
}

// ---------------------------------------------------------------------------
// The launches around the update kernels, shared by every network of a step.
// Each of these roles takes 1-3 us of one or a few workgroups, but about
// 4.6 us as a kernel of its own in a replayed graph, so a step of a circuit
// spent most of its small kernels on launches.  Roles that do not read each
// other's results share one:
//
// k_step_head, before the updates of step k: the clocks, spike trains and
// Poisson devices of k and the folds of plastic networks (they read spike
// lists of updates <= k - 2, weights of update k - 1 and the times of those
// spikes; the ring has max_delay + 2 slots, so slot k is not among them).
//
// k_step_tail, after them: every list of k (populations' and Poisson tiles),
// the folds of step k + 1 of networks without plastic synapses (they read
// lists of updates <= k - 1) and, in the first workgroup, the event-queue
// replay, which reads the tiles.
//
// k_step_post, when it has work: post-synaptic learning (reads the lists) and
// the replay when its sizes do not fit the tail's.
//
// The arguments travel by value (pointers read from a table in memory would
// be flat accesses), so a launch holds a fixed number of roles and a larger
// circuit takes several.  Per step: two small networks with plastic, train and
// Poisson inputs (800 AdEx and 200 LIF neurons) 74 us, 91 us with a kernel per
// role; a 2,501-granule cerebellum 134 and 152 us; 1,000 LIF neurons with
// Poisson inputs 64 us both ways (one launch less, a longer replay).
// ---------------------------------------------------------------------------
constexpr int kHeadRoles = 4, kHeadFolds = 2, kTailLists = 8, kTailFolds = 2, kPostRoles = 8;
struct FoldRole {
    FoldTarget target;
    RingEvents events;
    int blocks;
    int lanes;
};
struct StepHead {
    StepRef step;
    int n_tick, n_train, n_poisson, n_fold;
    TickArgs tick[kHeadRoles];
    TrainArgs train[kHeadRoles];
    int train_blocks[kHeadRoles];
    PoissonArgs poisson[kHeadRoles];
    FoldRole fold[kHeadFolds];
};
struct StepTail {
    int n_list, n_fold;
    CompactArgs list[kTailLists];
    int list_blocks[kTailLists];
    FoldRole fold[kTailFolds];
};
struct StepPost {
    int n_post, blocks;     // workgroups per role
    StdpPostArgs post[kPostRoles];
};

// kernel arguments are limited to 4 KB
static_assert(sizeof(StepHead) <= 3584 && sizeof(StepTail) + sizeof(EqArgs) <= 3584 && sizeof(StepPost) <= 3584, "");

__global__ __launch_bounds__(kBlock) void k_step_head(StepHead a) {
    int b = blockIdx.x;
    if (b < a.n_tick) {
        tick_body(a.tick[b], a.step.get());
        return;
    }
    b -= a.n_tick;
    for (int i = 0; i < a.n_train; i++) {
        if (b < a.train_blocks[i]) {
            train_body(a.train[i], b, a.train_blocks[i]);
            return;
        }
        b -= a.train_blocks[i];
    }
    for (int i = 0; i < a.n_poisson; i++) {
        if (b < a.poisson[i].n_tiles) {
            poisson_body(a.poisson[i], b);
            return;
        }
        b -= a.poisson[i].n_tiles;
    }
    for (int i = 0; i < a.n_fold; i++) {
        if (b < a.fold[i].blocks) {
            fold_ring_body<0, false>(a.fold[i].target, a.fold[i].events, b, a.fold[i].blocks, a.fold[i].lanes);
            return;
        }
        b -= a.fold[i].blocks;
    }
}

// ITEMS: heap entries of the replay in LDS; 0: no replay in this launch.
template <int ITEMS>
__global__ __launch_bounds__(kBlock) void k_step_tail(StepTail a, EqArgs q) {
    int b = blockIdx.x;
    if (ITEMS > 0) {
        if (b == 0) {
            eq_body<ITEMS == 0 ? 1 : ITEMS, kEqFusedDelays>(q);
            return;
        }
        b--;
    }
    for (int i = 0; i < a.n_list; i++) {
        if (b < a.list_blocks[i]) {
            clock_next_kernel(a.list[i]);
            compact_body(a.list[i], b, a.list_blocks[i]);
            return;
        }
        b -= a.list_blocks[i];
    }
    for (int i = 0; i < a.n_fold; i++) {
        if (b < a.fold[i].blocks) {
            if (a.fold[i].events.pulled)
                fold_ring_body<0, true>(a.fold[i].target, a.fold[i].events, b, a.fold[i].blocks, a.fold[i].lanes);
            else
                fold_ring_body<0, false>(a.fold[i].target, a.fold[i].events, b, a.fold[i].blocks, a.fold[i].lanes);
            return;
        }
        b -= a.fold[i].blocks;
    }
}

__global__ __launch_bounds__(kBlock) void k_step_post(StepPost a) {
    const int i = (int)blockIdx.x / a.blocks;
    if (i < a.n_post) stdp_post_body(a.post[i], (int)blockIdx.x % a.blocks, a.blocks);
}

// Adds every queued event of the population's keys to its conductances, in
// order (the groups delivered before a run's stop event), and clears the
// keys and fold flags.
__global__ __launch_bounds__(kBlock) void k_apply_fold(FoldTarget t, int32_t n, int par) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        for (int ty = 0; ty < 3; ty++) {
            const uint64_t key = (uint64_t)ty * (uint64_t)t.stride + (uint64_t)i;
            const uint32_t m = t.fill[key];
            if (m == 0u) continue;
            float *g = g_ptr(t, key);
            FoldEntry *e = t.b_ent + t.seg_off[key];
            *g = m == 1u ? *g + e->w : fold_sorted(e, t.rtab, par, m, *g);
            t.fill[key] = 0u;
        }
    }
}

}  // namespace edl
