// granule_bdf.hpp -- BDF step of the granule cell (EgidioGranuleCell_TimeDriven
// under BDFn, BDFn.h:288-423 and 682-786), one neuron on 16 lanes.
//
// The step is a Newton iteration on 15 equations with a 15 x 15 Jacobian that
// is inverted every time.  Lane z of a neuron's group holds row z: its state
// variable, predictor, history, Jacobian row and row of the inverse; lane 15
// evaluates the unperturbed membrane equation.  A group is one DPP row, so a
// pivot row reaches the other lanes as the DPP operand of the multiplication
// that uses it.  Every value takes exactly the reference's operations in its
// order:
//   * lane j evaluates the membrane equation with variable j perturbed (that
//     row of the Jacobian is the only dense one); a gate's column has besides
//     only the gate's own entry and, for xCa and yCa, calcium's (the other
//     rows difference to +0 exactly, as in the reference);
//   * the inverse is formed in place: at pivot s the dead column s of the
//     eliminated matrix becomes column s of the inverse, and the inverse's
//     still-unit columns are not stored (li[i][s] = 0 + li[s][s]*coef
//     included);
//   * a zero pivot (the reference then swaps rows) or a non-finite value
//     sends that Newton iteration through the reference arrangement
//     (granule_newton_reference) on a global working-storage slot.
#pragma once
#include "kernels.hpp"

namespace edl {

constexpr int kGrLanes = 16;   // lanes per neuron

// x of lane SRC of each group of 16 lanes (DPP row_newbcast).
template <int SRC>
__device__ __forceinline__ float group_bcast(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + SRC, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
// The largest of a group's values (none of them NaN), on all its lanes.
__device__ __forceinline__ float group_max(float x) {
    auto pick = [](float a, float b) { return b > a ? b : a; };
    x = pick(x, dpp_move<0xB1>(x));     // quad_perm 1,0,3,2
    x = pick(x, dpp_move<0x4E>(x));     // quad_perm 2,3,0,1
    x = pick(x, dpp_move<0x141>(x));    // row_half_mirror
    return pick(x, dpp_move<0x140>(x)); // row_mirror
}

// Loops over compile-time indices (the DPP control is an immediate).
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

struct GranuleGroup {
    using G = GranuleModel;
    static constexpr int ND = G::ND;
    int lane;                    // lane within the group, and its row (15: none)
    uint64_t bits;               // the group's lanes in a wave mask
    float S, P, D, ph;           // own row: state before the step, iterate, first difference, first previous state
    float syn[4];                // conductances and current of the step's equations (on every lane)
    float all[ND];               // the iterate on every lane
    float epsi;
    int st, k;

    // All 15 rows' values of a quantity, on every lane of the group.
    __device__ __forceinline__ static void gather(float own, float *v) {
        static_for<ND>([&](auto z) { v[z] = group_bcast<z>(own); });
    }
    // The row number for addresses, opaque to the compiler: the addresses of
    // a neuron's rows are then formed where they are used instead of being
    // kept in registers through the Newton iterations.  Lane 15 repeats row
    // 14's loads.
    __device__ __forceinline__ int row_here() const {
        int z = lane;
        asm volatile("" : "+v"(z));
        return min(z, ND - 1);
    }
    // true when `own` holds on every lane of the group
    __device__ __forceinline__ bool every(bool own) const { return (__ballot(own) & bits) == bits; }

    // One corrector iteration (granule_newton_reference's values).
    __device__ __forceinline__ void newton(const ModelParams &mp, const RhsCtx &c, float dt, const BdfState &b, int par,
                                           int64_t ld, uint32_t i) {
        const GranuleParams &p = mp.gran;
        const float *Cs = b.C + st * 7;
        const float c0 = Cs[0], c0dt = c0 * dt;
        const float eps = dt * 0.1f, inv_eps = 1.0f / eps;
        const float V = all[0], Vd = all[0] - eps, Ca = all[14], Cad = all[14] - eps;
        auto slope = [&](float f, float fn) { return c0dt * ((f - fn) * inv_eps); };
        // variable j, perturbed on lane j
        auto var = [&](int j) { return lane == j ? all[j] - eps : all[j]; };
        auto entry = [&](float v) {
            const int pos = trunc_i32_x86((v - kGrMinV) * kGrAux);
            return c.chan + (pos < 0 ? 0 : (pos > kGrTable - 1 ? kGrTable - 1 : pos)) * kGrVars;
        };
        const float *e0 = entry(V), *e1 = entry(Vd);
        // Nernst potentials at Ca and (lane 14) at Ca - eps
        const float nern = G::nernst_ca(p, lane == 14 ? Cad : Ca);
        const float vca = group_bcast<0>(nern);
        // the Ca-dependent K gate's steady state and rate at the iterate
        // (lane 0), with V perturbed (1) and with Ca perturbed (14)
        const float2 qk = *(const float2 *)((lane == 1 ? e1 : e0) + 18);
        const float ca_k = lane == 14 ? Cad : Ca;
        const float a_kca = p.a_xkca / (1.0f + qk.x / ca_k);
        const float b_kca = p.b_xkca / (1.0f + ca_k * qk.y);
        const float kinf = a_kca / (a_kca + b_kca), krate = a_kca + b_kca;
        // calcium equation (G::dca) at the iterate (lane 15), with V (0), xCa
        // (11), yCa (12) and Ca (14) perturbed; membrane equation (G::dv) at
        // the iterate (lane 15) and with variable j perturbed (lane j)
        constexpr float kFAd = ((2 * 96485.309f) * 1e-04f) * 0.2f;
        const float x0 = var(0), x11 = var(11), x12 = var(12);
        const float gCa = 0.00046f * x11 * x11 * x12;
        const float fca = (-gCa * (x0 - nern) / kFAd - (1.5f * (var(14) - 1e-04f)));
        float fv;
        {
            float cur = 0.0f;
            if (p.mask & 1u) cur += syn[0] * (p.e_exc - x0);
            if (p.mask & 2u) cur += syn[1] * (p.e_inh - x0);
            if (p.mask & 4u) {
                const float gi = nmda_inf(c.nmda_lut, p.nmda_aux, p.e_inh, x0);
                cur += syn[2] * gi * (p.e_exc - x0);
            }
            cur += syn[3];
            cur = (float)((double)cur * 3.34156941e-4);
            const float x1 = var(1), x6 = var(6), x7 = var(7);
            const float gNa_f = 0.013f * x1 * x1 * x1 * var(2);
            const float gNa_r = 0.0005f * var(3) * var(4);
            const float gNa_p = 0.0002f * var(5);
            const float gK_V = 0.003f * x6 * x6 * x6 * x6;
            const float gK_A = 0.004f * x7 * x7 * x7 * var(8);
            const float gK_IR = 0.0009f * var(9);
            const float gK_Ca = 0.004f * var(10);
            const float gK_sl = 0.00035f * var(13);
            const float dNa = 87.39f - x0, dK = -84.69f - x0;
            fv = (cur + gNa_f * dNa + gNa_r * dNa + gNa_p * dNa + gK_V * dK + gK_A * dK + gK_IR * dK + gK_Ca * dK +
                  gCa * (nern - x0) + gK_sl * dK + 5.68e-5f * (-58.0f - x0) + 2.17e-5f * (-65.0f - x0)) *
                 (1.0f / 1.0e-3f);
        }
        const float f0 = group_bcast<15>(fv);
        const float jv0 = slope(f0, fv);   // row 0 of the Jacobian, one entry per lane
        // own row at the iterate (f), with V (fV) and with the own variable
        // (fd) perturbed.  Voltage-gated variables (G::dgate) read their two
        // table columns (x_inf, 1/tau).
        const int zg = (lane < 1 || lane > 13) ? 1 : lane;
        const int col = zg < 10 ? 2 * (zg - 1) : 2 * zg - 2;
        const float2 q0 = *(const float2 *)(e0 + col), q1 = *(const float2 *)(e1 + col);
        float f = (q0.x - P) * q0.y, fV = (q1.x - P) * q1.y, fd = (q0.x - (P - eps)) * q0.y;
        float f14 = 0.0f, f11 = 0.0f, f12 = 0.0f;   // rows 10 and 14: with Ca, row 14: with xCa, yCa perturbed
        {
            const float ki = group_bcast<0>(kinf), kr = group_bcast<0>(krate);
            const float ki1 = group_bcast<1>(kinf), kr1 = group_bcast<1>(krate);
            const float ki14 = group_bcast<14>(kinf), kr14 = group_bcast<14>(krate);
            const float ca = group_bcast<15>(fca), ca0 = group_bcast<0>(fca), ca14 = group_bcast<14>(fca);
            f11 = group_bcast<11>(fca);
            f12 = group_bcast<12>(fca);
            if (lane == 10) {
                f = (ki - P) * kr;
                fV = (ki1 - P) * kr1;
                fd = (ki - (P - eps)) * kr;
                f14 = (ki14 - P) * kr14;
            }
            if (lane == 14) {
                f = ca;
                fV = ca0;
                fd = ca14;
            }
            if (lane == 0) f = f0;
            if (lane == 15) f = fV = fd = 0.0f;
        }
        const bool fin = every(__builtin_isfinite(f));
        // J = c0*dt*jac - I, jac[z][j] = (F[z] - Fn_j[z]) / eps (one-sided)
        float A[ND];
        {
            const float jV = slope(f, fV), jd = slope(f, fd) - 1;
            A[0] = lane == 15 ? 0.0f : jV;
#pragma unroll
            for (int j = 1; j < ND; j++) A[j] = lane == j ? jd : 0.0f;
            if (lane == 14) {
                A[11] = slope(f, f11);
                A[12] = slope(f, f12);
            }
            if (lane == 10) A[14] = slope(f, f14);
            static_for<ND>([&](auto j) {
                const float x = group_bcast<j>(jv0);
                A[j] = lane == 0 ? x : A[j];
            });
            if (lane == 0) A[0] -= 1;
        }
        float cc = c0 * dt * f + Cs[1] * S;
        if (st > 1) cc += Cs[2] * ph;
        if (st > 2) {
            const int z = row_here();
            for (int q = 2; q < st; q++) cc += Cs[q + 1] * ((const float *)b.prev)[((int64_t)(q - 1) * ND + z) * ld + i];
        }
        bool ok = true;
        // (opaque: the pivots' lane masks are compared where they are used
        // instead of being kept in registers)
        int zl = lane;
        asm volatile("" : "+v"(zl));
        static_for<ND>([&](auto sc) {
            constexpr int s = sc;
            const float element = group_bcast<s>(A[s]);
            ok = ok && element != 0.0f;
            const float inv = 1.0f / element;
            const bool pivot = zl == s;
            const float coef = -A[s];
            // the pivot row is scaled in place (x * 1 is x on the other rows)
            const float m = pivot ? inv : 1.0f;
            float t[ND];
#pragma unroll
            for (int j = 0; j < ND; j++)
                if (j != s) A[j] *= m;
#pragma unroll
            for (int j = 0; j < ND; j++)
                if (j != s) {
                    t[j] = group_bcast<s>(A[j]) * coef;
                    asm volatile("" : "+v"(t[j]));   // formed on all lanes: the DPP operand needs them
                }
            A[s] = inv;
            if (!pivot) {
#pragma unroll
                for (int j = 0; j < ND; j++)
                    if (j != s) A[j] += t[j];
                A[s] = 0.0f + inv * coef;
            }
        });
        // aux is finite only if the row of the inverse is (a non-finite entry
        // makes its product, and with it the sum, non-finite)
        float da[ND], aux = 0.0f;
        gather(P - cc, da);
#pragma unroll
        for (int q = 0; q < ND; q++) aux += A[q] * da[q];
        float P1 = aux + P;
        bool good = fin && ok;
        if (good && !every(__builtin_isfinite(aux))) {
            bool finA = true;
#pragma unroll
            for (int j = 0; j < ND; j++) finA = finA && __builtin_isfinite(A[j]);
            good = every(finA || lane == 15);
        }
        if (!good) {
            bool nan = false;
#pragma unroll
            for (int q = 0; q < ND; q++) nan = nan || all[q] != all[q];
            if (nan) {
                // An iterate with a NaN component corrects to all NaN
                // whatever the Jacobian: every P1[z] = sum_t iJ[z][t] * (P[t]
                // - Cc[t]) + P[z] takes the NaN term (and the max-norm change
                // below is then 0: no comparison with a NaN holds).  This is
                // the standing case of a neuron whose step once went NaN: the
                // NaN reset restores the state but not the BDF history
                // (TimeDrivenNeuronModel.cpp:75-88), so every later predictor
                // is NaN.  Only the NaN payload can differ from the full
                // correction's.
                P1 = __builtin_nanf("");
            } else {
                float ca[ND];
                gather(cc, ca);
                int32_t slot = -1;
                if (lane == 0) {
                    const uint32_t got = atomicAdd(&b.ws_count[par], 1u);
                    if (got < (uint32_t)b.ws_cap) {
                        slot = (int32_t)got;
                        float *w = b.ws + (size_t)slot * kGrWsFloats;
                        float *X = w + 450, *Cw = X + G::NV + 2 * ND;
#pragma unroll
                        for (int q = 0; q < ND; q++) X[q] = all[q];
#pragma unroll
                        for (int q = 0; q < 4; q++) X[ND + q] = syn[q];
#pragma unroll
                        for (int q = 0; q < ND; q++) Cw[q] = ca[q];
                        granule_newton_reference(mp, c, dt, c0, w);
                        const float *P1w = Cw + ND;
#pragma unroll
                        for (int q = 0; q < ND; q++) ca[q] = P1w[q];
                    } else {
                        atomicOr(b.err, 16u);   // reported to the host; the step is not the reference's
#pragma unroll
                        for (int q = 0; q < ND; q++) ca[q] = all[q];
                    }
                }
                static_for<ND>([&](auto z) {
                    const float x = group_bcast<0>(ca[z]);
                    P1 = lane == z ? x : P1;
                });
            }
        }
        const float change = fabsf(P1 - P);
        epsi = group_max((lane < ND && change > 0.0f) ? change : 0.0f);
        P = P1;
        gather(P, all);
        k++;
    }

    // Takes neuron i: its rows, the fold of its input events and the external
    // drive (on the group's first lane), and the predictor.
    template <bool EXT>
    __device__ __forceinline__ void take(const UpdateArgs &a, const RhsCtx &c, float dt, int32_t step,
                                         uint32_t step_key, uint32_t flag, uint32_t i) {
        const int64_t ld = a.stride;
        const float *Dh = (const float *)a.bdf.d;
        // every load at once: what the method's order makes of them is
        // decided afterwards
        st = a.bdf.st[i];
        const int64_t at = (int64_t)row_here() * ld + i;
        S = a.state[at];
        D = Dh[at];
        ph = ((const float *)a.bdf.prev)[at];
        const float D1 = a.bdf.order > 1 ? Dh[at + ND * ld] : 0.0f;
        float in[4];
#pragma unroll
        for (int q = 0; q < 4; q++) in[q] = 0.0f;
        if (lane == 0) {
#pragma unroll
            for (int q = 0; q < 4; q++) in[q] = a.state[(int64_t)(ND + q) * ld + i];
            if (flag) {
                const bool live[1] = {true};
                float g[3][1] = {{in[0]}, {in[1]}, {in[2]}};
                fold_keys<7u, 1>(a, step, i, live, g);
                for (int ty = 0; ty < 3; ty++) in[ty] = g[ty][0];
            }
            if (EXT) {
                const uint32_t u = drive_hash_keyed(step_key, i);
                int cnt = 0;
                while (cnt < a.ext.n_thr && u < a.ext.thr[cnt]) cnt++;
                for (int q = 0; q < cnt; q++) in[0] += a.ext.w;
            }
        }
#pragma unroll
        for (int q = 0; q < 4; q++) syn[q] = group_bcast<0>(in[q]);
        if (st == 0) {
            float X[G::NV], F[ND], f = 0.0f;
            gather(S, X);
#pragma unroll
            for (int q = 0; q < 4; q++) X[ND + q] = syn[q];
            G::rhs<15u>(a.mp, c, X, F);
#pragma unroll
            for (int q = 0; q < ND; q++) f = q == lane ? F[q] : f;
            P = S + dt * f;
        } else {
            P = S + D;
            if (st > 1) P += D1;
            for (int q = 2; q < st; q++) P += Dh[at + (int64_t)q * ND * ld];
        }
        const GranuleParams &p = a.mp.gran;
#pragma unroll
        for (int q = 0; q < 3; q++)
            if (p.mask & (1u << q)) syn[q] = decay_g(syn[q], p.cf[q]);
        gather(P, all);
        epsi = 1.0f;
        k = 0;
    }

    // Stores neuron i after its corrector: history, state (a NaN membrane
    // potential puts the whole state back to its initial values,
    // TimeDrivenNeuronModel.cpp:75-88) and spike bit.
    __device__ __forceinline__ void commit(const UpdateArgs &a, int32_t step, uint32_t i) {
        const int64_t ld = a.stride;
        float *Dh = (float *)a.bdf.d, *Ph = (float *)a.bdf.prev;
        if (st < a.bdf.order) st++;
        const bool nan = all[0] != all[0];
        if (lane < ND) {
            const int z = row_here();
            const int64_t at = (int64_t)z * ld + i, level = ND * ld;
            // differences: D[q] = -D[q-1] from the highest down, the step's
            // own in D[0], then each added to the next
            for (int q = st - 1; q > 1; q--) Dh[at + q * level] = -Dh[at + (q - 1) * level];
            const float d0 = P - S;
            Dh[at] = d0;
            if (st > 1) {
                float d = -D + d0;
                Dh[at + level] = d;
                for (int q = 2; q < st; q++) {
                    d = Dh[at + q * level] + d;
                    Dh[at + q * level] = d;
                }
                for (int q = st - 2; q > 0; q--) Ph[at + q * level] = Ph[at + (q - 1) * level];
                Ph[at] = S;
            }
            a.state[at] = nan ? G::init(a.mp, z) : P;
        }
        if (lane == 0) {
            a.bdf.st[i] = st;
            if (G::spike(a.mp, S, &P)) {
                if (a.last_spike) a.last_spike[i] = step;
                atomicOr(&a.bdf.spk_bits[i >> 5], 1u << (i & 31));
            }
#pragma unroll
            for (int q = 0; q < 3; q++) a.state[(int64_t)(ND + q) * ld + i] = nan ? G::init(a.mp, ND + q) : syn[q];
            if (nan) a.state[(int64_t)(ND + 3) * ld + i] = G::init(a.mp, ND + 3);
        }
    }
};

// Granule BDF update.  The corrector runs a data-dependent number of Newton
// iterations per neuron (about 3 on average, but 10 for the few percent
// whose iterate ends in a one-ulp cycle), so a wave that gave each group a
// fixed neuron would run each for its slowest group's count.  Here each wave
// owns a contiguous range of neurons and a group takes the range's next
// neuron when its own corrector has ended; a neuron's arithmetic is the same
// either way.  The grid is at most one workgroup per CU; the ranges are
// equal.
//   * The channel table (104 KB) is staged in LDS (every Newton iteration
//     gathers two of its rows), and so are the BDF coefficients.
//   * Spikes set bits of a.bdf.spk_bits; the last workgroup to finish turns
//     them into the per-tile spike lists (ascending, kFlagTile neurons per
//     tile) that the compaction reads, clears the bits and the tiles' fold
//     flags, and resets the workgroup count.
//   * A group reads its neuron's fold flag when it takes the neuron.
//
// Bound by VALU issue in large populations (a Newton iteration of a wave's
// four neurons is about 1,500 instructions, 64 of them per pivot) and by the
// latency of that chain in small ones.  BDF2 in the cerebellar circuit, per
// launch: 495 us with 200,000 cells, 59 us with 2,501.  With a whole neuron
// on one lane (14,000 instructions per iteration, the matrix in the register
// file of one wave per SIMD) 762 us and 585 us; on four lanes the matrix
// spills (1,554 us and 258 us).
constexpr int kGrBdfThreads = 1024;   // largest workgroup: four waves per SIMD (128 registers each)
template <bool EXT>
__global__ __launch_bounds__(kGrBdfThreads) void k_update_granule_bdf(UpdateArgs a) {
    constexpr int TILE = kBdfBlock, L = kGrLanes;   // spike lists by kBdfBlock neurons
    static_assert(TILE == kFlagTile, "one fold flag per spike list");
    const int32_t step = a.step.get();
    clock_begin(a, step);
    const int par = a.fold.par_by_step ? (step & 1) : a.fold.par;
    // the next step hands out working-storage slots from the other parity
    if (blockIdx.x == 0 && threadIdx.x == 0 && a.bdf.ws_count) a.bdf.ws_count[par ^ 1] = 0u;
    const uint32_t step_key = EXT ? drive_step_key(a.ext.seed, step) : 0u;
    __shared__ float s_bdfc[49];
    extern __shared__ float4 s_chan[];
    {
        const float4 *g4 = (const float4 *)a.chan;
        for (int q = threadIdx.x; q < kGrTable * kGrVars / 4; q += blockDim.x) s_chan[q] = g4[q];
        if (threadIdx.x < 49) s_bdfc[threadIdx.x] = a.bdf.C[threadIdx.x];
    }
    __syncthreads();
    BdfState bl = a.bdf;
    bl.C = s_bdfc;
    RhsCtx c;
    c.chan = (const float *)s_chan;
    c.exp_lut = a.exp_lut;
    c.nmda_lut = a.nmda_lut;
    c.refr = a.refr;
    c.refr_len = a.refr_len;
    c.since_spike = 1 << 30;
    const float dt = a.k.dt;
    const int wlane = threadIdx.x & (kWave - 1);
    GranuleGroup g;
    g.lane = wlane % L;
    g.bits = ((1ull << L) - 1ull) << (wlane - g.lane);
    g.epsi = 1.0f;
    g.st = g.k = 0;
    const uint64_t below = (1ull << (wlane - g.lane)) - 1ull;
    const int waves_per_block = (int)blockDim.x / kWave;
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * waves_per_block + threadIdx.x / kWave));
    const int64_t n_waves = (int64_t)gridDim.x * waves_per_block;
    int cursor = (int)((int64_t)a.n * wave / n_waves);
    const int end = (int)((int64_t)a.n * (wave + 1) / n_waves);
    int i = -1;          // neuron of this group (-1: none)
    for (;;) {
        bool busy = i >= 0 && g.epsi > 1e-6 && g.k < 10;   // the corrector's loop condition
        const uint64_t run = __ballot(busy);
        // groups whose corrector has ended commit and take new neurons
        if (run != ~0ull) {
            if (i >= 0 && !busy) {
                g.commit(a, step, (uint32_t)i);
                i = -1;
            }
            if (cursor < end) {
                const uint64_t idle = __ballot(i < 0);
                if (i < 0) {
                    const int j = cursor + __popcll(idle & below) / L;
                    if (j < end) {
                        i = j;
                        g.take<EXT>(a, c, dt, step, step_key, a.fold.tile_flag[j / TILE], (uint32_t)i);
                        busy = true;
                    }
                }
                cursor += __popcll(idle) / L;
            }
        }
        if (!__any(busy)) break;
        if (busy) g.newton(a.mp, c, dt, bl, par, a.stride, (uint32_t)i);
    }
    __shared__ uint32_t s_last;
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        s_last = atomicAdd(a.bdf.done, 1u) == gridDim.x - 1u;
    }
    __syncthreads();
    if (s_last) {
        __threadfence();
        for (int t = threadIdx.x; t < a.n_tiles; t += blockDim.x) {
            int32_t cnt = 0;
            for (int w = 0; w < TILE / 32; w++) {
                uint32_t bits = atomicExch(&a.bdf.spk_bits[t * (TILE / 32) + w], 0u);
                while (bits) {
                    const int b = __builtin_ctz(bits);
                    bits &= bits - 1u;
                    a.out.staging[(int64_t)t * TILE + cnt++] = t * TILE + w * 32 + b;
                }
            }
            a.out.tile_count[t] = cnt;
            clear_tile_flag<TILE>(a.fold.tile_flag, t);
        }
        if (threadIdx.x == 0) *a.bdf.done = 0u;
    }
    clock_finish(a, step);
}

}  // namespace edl
