// adjoint.hpp -- differentiable trace fitting: forward simulation of
// independent LIF (Euler) or AdEx (RK4) neurons driven by fixed input spike
// trains, and the discrete adjoint of that simulation with checkpointed
// recomputation.
//
// Forward map of one step (the plain path's update, made differentiable):
// events of the step add their weights to g_exc / g_inh; LIF takes an Euler
// step scaled by the refractory fraction, AdEx an RK4 step with conductances
// decayed at the half steps; conductances below 1e-9 snap to zero; a spike
// resets V (LIF to e_leak; AdEx to e_reset, w += b).  The AdEx exponential
// term uses expf (the reference's CUDA kernels do the same,
// AdExTimeDrivenModel_GPU2.cuh:307,313; the CPU table's derivative is zero
// almost everywhere) and decay factors are exp(-h/tau) of each neuron's tau.
//
// The forward recurrence is sequential: one lane per neuron, one wave per
// workgroup advancing it and a second wave bringing the inputs of the next
// steps into LDS.  The adjoint recurrence is linear in the adjoint state, so
// the backward pass runs every checkpoint segment at once:
//
//   k_fit_forward  V trace [steps][n]; state + event cursor every `keep`
//                  segments of `seg` steps
//   k_fit_expand   (keep > 1) per (kept checkpoint, neuron): the forward pass
//                  again from there, giving every segment's state and cursor
//   k_fit_maps     per (segment, neuron): the affine map from the adjoint
//                  state at the segment's end to the one at its start
//   k_fit_scan     per neuron: those maps applied from the last segment to
//                  the first, giving the adjoint state at every segment's end
//   k_fit_sweep    per (segment, neuron): the reverse sweep from that state
//                  (reverse-mode differentiation of each step with the
//                  forward run's spike pattern held fixed: a reset stops the
//                  V adjoint and, for LIF, routes it to e_leak)
//   k_fit_grads    per neuron: the segments' parameter gradients and the
//                  synapses' weight gradients summed, last step first
//
// 256 neurons, 50 inputs at 20 Hz, 10,000 steps, on one MI355X: the backward
// pass takes 0.33 ms (LIF) and 0.48 ms (AdEx).  With one lane walking a
// neuron's whole sweep it took 15.2 ms and 25.1 ms on 4 of 256 CUs; the
// segments give it 80,000 lanes.
#pragma once
#include "device_common.hpp"

namespace edl {

constexpr int kFitBlock = 64;   // neurons (forward) or (segment, neuron) pairs per workgroup
// Longest segment: the forward pass stages a segment's inputs (four values
// per step and lane, twice, one step of padding each: 66 KB, 68 KB with its
// small tables) and the backward pass its states (four values, 32 KB) in LDS, so
// two forward workgroups or five backward waves share a CU's 160 KB.
constexpr int kFitSeg = 32;
constexpr int kFitRefr = 256;   // refractory fractions staged in LDS (longer tables: read from memory)
constexpr int kFitGradBlock = 128;

struct FitArgs {
    int n, steps, n_syn, seg, segs;
    float dt, h, s6;
    // fixed parameters
    float e_exc, e_inh, v_thr, inv_c_m;          // both
    float a, b, thr, inv_thr, inv_tau_w, e_reset, v_cap;   // AdEx
    const float *refr;                           // LIF refractory fractions
    int refr_len;
    // trainable
    const float *gl, *el, *te, *ti;              // [n]
    const float *w;                              // [n][n_syn]
    const uint8_t *syn_type;                     // [n][n_syn] 0 exc, 1 inh
    // inputs: per neuron, events sorted by step
    const int32_t *ev_ptr, *ev_step, *ev_syn;
    // forward outputs
    float *v_trace;                              // [steps][n]
    uint8_t *spikes;                             // [steps][n] (optional)
    float *traj;                                 // [steps][4][n] state before integration (optional)
    int32_t *traj_since;                         // [steps][n] refractory count (optional)
    int keep;                                    // segments per checkpoint
    float *kept_state;                           // [checkpoints+1][4][n]
    int32_t *kept_int;                           // [checkpoints+1][2][n]: event cursor, last spike
    // backward: segments [c_lo, c_hi) of this launch
    int c_lo, c_hi;
    int ck_lo;                                   // segment of the first row below
    float *ck_state;                             // [segments][4][n]
    int32_t *ck_int;                             // [segments+1][2][n]: event cursor, last spike
    const float *grad_v;                         // [steps][n]
    float *grad_par;                             // [4][n]: g_leak e_leak tau_exc tau_inh
    float *grad_w;                               // [n][n_syn]
    double *maps;                                // [segments of a launch][kFitMap][n]
    double *part;                                // [segments of a launch][4][n] parameter gradients
    float *lg;                                   // [steps of a launch][2][n] conductance adjoints
    double *carry;                               // [8][n]: adjoint state entering the launch, gradient sums
};

__device__ __forceinline__ float fit_decay(float g, float cf) { return (g < 1e-9f) ? 0.0f : g * cf; }

__device__ __forceinline__ float lif_frac(const FitArgs &a, int since) {
    if (since >= a.refr_len) return 1.0f;
    const float f = a.refr[since];
    return f < 0.0f ? 0.0f : f;
}

// AdEx right-hand side; E returns the exponential term's exp() (0 above 0 mV)
__device__ __forceinline__ void fit_adex_f(const FitArgs &a, float gl, float el, float V, float W, float ge,
                                           float gi, float &dV, float &dW, float &E) {
    // up to v_cap as it stands, then V held at v_cap up to 0 mV, nothing above
    const bool low = V <= a.v_cap, live = low || V <= 0.0f;
    const float Vm = low ? V : a.v_cap;
    const float e = expf((Vm - a.v_thr) * a.inv_thr);
    const float cur = ge * (a.e_exc - Vm) + gi * (a.e_inh - Vm);
    const float v = (gl * (el - Vm) + gl * a.thr * e - W + cur) * a.inv_c_m;
    const float w = (a.a * (V - el) - W) * a.inv_tau_w;
    E = live ? e : 0.0f;
    dV = live ? v : 0.0f;
    dW = live ? w : 0.0f;
}

// (ldV, ldW) . d(dV, dW)/d(V, W, ge, gi, gl, el) given the stage point and E;
// lp (g_leak and e_leak gradients) may be null
__device__ __forceinline__ void fit_adex_vjp(const FitArgs &a, float gl, float el, float V, float ge,
                                             float gi, float E, float ldV, float ldW, float *lx,
                                             double *lp) {
    if (V <= a.v_cap) {
        lx[0] += ldV * (-gl - ge - gi + gl * a.thr * E * a.inv_thr) * a.inv_c_m + ldW * a.a * a.inv_tau_w;
        lx[1] += -ldV * a.inv_c_m - ldW * a.inv_tau_w;
        lx[2] += ldV * (a.e_exc - V) * a.inv_c_m;
        lx[3] += ldV * (a.e_inh - V) * a.inv_c_m;
        if (lp) {
            lp[0] += (double)(ldV * ((el - V) + a.thr * E) * a.inv_c_m);
            lp[1] += (double)(ldV * gl * a.inv_c_m - ldW * a.a * a.inv_tau_w);
        }
    } else if (V <= 0.0f) {
        const float Vm = a.v_cap;
        lx[0] += ldW * a.a * a.inv_tau_w;
        lx[1] += -ldV * a.inv_c_m - ldW * a.inv_tau_w;
        lx[2] += ldV * (a.e_exc - Vm) * a.inv_c_m;
        lx[3] += ldV * (a.e_inh - Vm) * a.inv_c_m;
        if (lp) {
            lp[0] += (double)(ldV * ((el - Vm) + a.thr * E) * a.inv_c_m);
            lp[1] += (double)(ldV * gl * a.inv_c_m - ldW * a.a * a.inv_tau_w);
        }
    }
}

// The stage points the adjoint of an AdEx step needs, recomputed from the
// state before it.
struct AdexStages {
    float aV[3], E[4];   // V of stages 2-4, exp() of stages 1-4
    bool fired;
};

// One forward step from state (V, W, ge, gi) after the step's inputs.  MODEL
// 0: LIF, `frac` its refractory fraction; 1: AdEx, `st` (if non-null)
// receives its stages.
template <int MODEL>
__device__ __forceinline__ bool fit_step(const FitArgs &a, float gl, float el, float cfe, float cfi,
                                         float frac, float &V, float &W, float &ge, float &gi,
                                         AdexStages *st = nullptr) {
    if (MODEL == 0) {
        const float cur = ge * (a.e_exc - V) + gi * (a.e_inh - V);
        const float f = frac * ((cur + gl * (el - V)) * a.inv_c_m);
        V = V + a.dt * f;
        ge = fit_decay(ge, cfe);
        gi = fit_decay(gi, cfi);
        const bool fired = V > a.v_thr;
        V = fired ? el : V;
        return fired;
    }
    float d1V, d1W, d2V, d2W, d3V, d3W, d4V, d4W, E1, E2, E3, E4;
    fit_adex_f(a, gl, el, V, W, ge, gi, d1V, d1W, E1);
    const float gem = fit_decay(ge, cfe), gim = fit_decay(gi, cfi);
    const float a1V = V + d1V * a.h, a1W = W + d1W * a.h;
    fit_adex_f(a, gl, el, a1V, a1W, gem, gim, d2V, d2W, E2);
    const float a2V = V + d2V * a.h, a2W = W + d2W * a.h;
    fit_adex_f(a, gl, el, a2V, a2W, gem, gim, d3V, d3W, E3);
    const float ge2 = fit_decay(gem, cfe), gi2 = fit_decay(gim, cfi);
    const float a3V = V + d3V * a.dt, a3W = W + d3W * a.dt;
    fit_adex_f(a, gl, el, a3V, a3W, ge2, gi2, d4V, d4W, E4);
    V = V + (d1V + 2.0f * (d2V + d3V) + d4V) * a.s6;
    W = W + (d1W + 2.0f * (d2W + d3W) + d4W) * a.s6;
    ge = ge2;
    gi = gi2;
    const bool fired = V > 0.0f;
    V = fired ? a.e_reset : V;
    W = fired ? W + a.b : W;
    if (st) {
        st->aV[0] = a1V; st->aV[1] = a2V; st->aV[2] = a3V;
        st->E[0] = E1; st->E[1] = E2; st->E[2] = E3; st->E[3] = E4;
        st->fired = fired;
    }
    return fired;
}

// A neuron's events from a cursor on, applied step by step in list order.
struct FitEvents {
    const float *w;
    const uint8_t *ty;
    const int32_t *step, *syn;
    int e, end, next;
    __device__ __forceinline__ void seek(const FitArgs &a, int i, int cursor) {
        w = a.w + (int64_t)i * a.n_syn;
        ty = a.syn_type + (int64_t)i * a.n_syn;
        step = a.ev_step;
        syn = a.ev_syn;
        e = cursor;
        end = a.ev_ptr[i + 1];
        next = e < end ? step[e] : 0x7fffffff;
    }
    __device__ __forceinline__ void apply(int k, float &ge, float &gi) {
        while (next == k) {
            const int s = syn[e];
            if (ty[s] == 0) ge += w[s];
            else gi += w[s];
            e++;
            next = e < end ? step[e] : 0x7fffffff;
        }
    }
};

// Forward pass, one segment of steps at a time.  The step recurrence is a
// chain of dependent instructions (about 45 for LIF, 240 for AdEx), so wave 0
// does little but that chain: it reads its inputs from LDS one step ahead
// and never waits on memory.  Wave 1 meanwhile fills the next segment's
// inputs: per step and neuron the first two events of each type (absent ones
// are 0: adding it changes nothing), and a bit for the steps that have more,
// whose events wave 0 then walks itself.  Lanes past the last neuron repeat
// it (the same values to the same places).  EXTRA: with the optional outputs,
// with a refractory table too long for LDS, or with checkpoints further apart
// than segments (the counters of their rows in the other variants take the LIF
// forward of 256 neurons from 1.64 to 1.75 ms).
//
// 256 neurons, 10,000 steps: 1.63 ms (LIF) and 4.7 ms (AdEx).  With the events
// walked inside the recurrence (three dependent loads in nearly every step of
// a wave) it took 5.6 ms and 9.2 ms.
template <int MODEL, bool EXTRA>
__global__ __launch_bounds__(2 * kFitBlock) void k_fit_forward(FitArgs a) {
    __shared__ __align__(16) float s_in[2][kFitSeg + 1][4][kFitBlock];   // one step of padding: read ahead
    __shared__ uint32_t s_more[2][kFitBlock];
    __shared__ uint32_t s_any[2];
    __shared__ int32_t s_cur[2][kFitBlock];
    __shared__ float s_refr[kFitRefr + 1];
    const int lane = (int)(threadIdx.x & (kFitBlock - 1));
    const bool producer = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kFitBlock)) != 0;
    const int i = min((int)blockIdx.x * kFitBlock + lane, a.n - 1);
    const float *w = a.w + (int64_t)i * a.n_syn;
    const uint8_t *ty = a.syn_type + (int64_t)i * a.n_syn;
    const bool refr_lds = MODEL == 0 && (!EXTRA || a.refr_len <= kFitRefr);
    if (refr_lds)
        for (int q = threadIdx.x; q <= a.refr_len; q += 2 * kFitBlock) s_refr[q] = lif_frac(a, q);
    // wave 1: the next event to place and the step of the last one placed (an
    // event out of order ends the list, as it does for a step-by-step walk)
    const int e_end = a.ev_ptr[i + 1];
    const bool any_event = a.ev_ptr[a.n] > 0;
    int e = a.ev_ptr[i], pos = 1;
    auto fill = [&](int c, int buf) {
        const int k0 = c * a.seg + 1, k1 = min(a.steps, (c + 1) * a.seg);
        float *in = &s_in[buf][0][0][0];
        for (int q = 0; q <= k1 - k0; q++) ((float4 *)in)[q * kFitBlock + lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        s_cur[buf][lane] = e;
        uint32_t more = 0;
        int n_e = 0, n_i = 0;
        bool run = any_event && e < e_end;
        while (__any(run)) {
            // eight events' loads in flight at once (past the neuron's last
            // one the index stays on it; it is then not placed)
            constexpr int B = 8;
            int st[B], sy[B];
            float wt[B];
            uint8_t tp[B];
            const int hi = max(e_end - 1, 0);
#pragma unroll
            for (int u = 0; u < B; u++) {
                st[u] = a.ev_step[min(e + u, hi)];
                sy[u] = a.ev_syn[min(e + u, hi)];
            }
#pragma unroll
            for (int u = 0; u < B; u++) {
                // a lane without events sees another neuron's synapse number:
                // as much in range as its own
                wt[u] = w[sy[u]];
                tp[u] = ty[sy[u]];
            }
#pragma unroll
            for (int u = 0; u < B; u++) {
                run = run && e < e_end && st[u] >= pos && st[u] <= k1;
                if (run) {
                    if (st[u] != pos) n_e = n_i = 0;
                    pos = st[u];
                    const int j = pos - k0;
                    const int m = tp[u] == 0 ? n_e++ : n_i++;
                    if (m < 2) in[(j * 4 + (tp[u] == 0 ? m : 2 + m)) * kFitBlock + lane] = wt[u];
                    else more |= 1u << j;
                    e++;
                }
            }
            run = run && e < e_end;
        }
        pos = max(pos, k1 + 1);
        s_more[buf][lane] = more;
        for (int off = 32; off > 0; off >>= 1) more |= (uint32_t)__shfl_xor((int)more, off);
        if (lane == 0) s_any[buf] = more;
    };
    if (producer) fill(0, 0);
    __syncthreads();
    const float gl = a.gl[i], el = a.el[i];
    const float cfe = expf(-a.h / a.te[i]), cfi = expf(-a.h / a.ti[i]);
    float V = el, W = 0.0f, ge = 0.0f, gi = 0.0f;
    int last = -(1 << 30);
    // refractory fraction of the coming step, and its entry in the table (LIF)
    float frac = 1.0f;
    int since = a.refr_len;
    const float frac0 = refr_lds ? s_refr[0] : 1.0f;
    float *vt = a.v_trace + i;
    int row = 0, to_keep = 1;   // checkpoint row, segments it still takes
    for (int c = 0; c < a.segs; c++) {
        const int buf = c & 1;
        if (producer) {
            if (c + 1 < a.segs) fill(c + 1, buf ^ 1);
            else a.kept_int[(int64_t)(EXTRA ? (a.segs + a.keep - 1) / a.keep : a.segs) * 2 * a.n + i] = e;   // past the last event
        } else {
            const int k0 = c * a.seg + 1, k1 = min(a.steps, (c + 1) * a.seg);
            // a row is written over until its last segment, the kept one
            float *cs = a.kept_state + (int64_t)(EXTRA ? row : c) * 4 * a.n;
            cs[i] = V;
            cs[a.n + i] = W;
            cs[2 * a.n + i] = ge;
            cs[3 * a.n + i] = gi;
            int32_t *ci = a.kept_int + (int64_t)(EXTRA ? row : c) * 2 * a.n;
            ci[i] = s_cur[buf][lane];
            ci[a.n + i] = last;
            if (EXTRA && --to_keep == 0) {
                to_keep = a.keep;
                row++;
            }
            int cur = s_cur[buf][lane];   // events up to it belong to earlier steps
            uint32_t any = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_any[buf]);
            const float *in = &s_in[buf][0][0][lane];
            float x[4];
#pragma unroll
            for (int q = 0; q < 4; q++) x[q] = in[q * kFitBlock];
            for (int k = k0; k <= k1; k++) {
                in += 4 * kFitBlock;
                float y[4];
#pragma unroll
                for (int q = 0; q < 4; q++) y[q] = in[q * kFitBlock];
                float fnext = 1.0f;
                if (refr_lds) {
                    since = min(since + 1, a.refr_len);
                    fnext = s_refr[since];   // the next step's, without a spike
                }
                const bool more = (any & 1u) && ((s_more[buf][lane] >> (k - k0)) & 1u);
                any >>= 1;
                if (more) {
                    // more than two events of a type in this step
                    while (a.ev_step[cur] < k) cur++;
                    for (; cur < e_end && a.ev_step[cur] == k; cur++) {
                        const int s = a.ev_syn[cur];
                        if (ty[s] == 0) ge += w[s];
                        else gi += w[s];
                    }
                } else {
                    ge += x[0];
                    ge += x[1];
                    gi += x[2];
                    gi += x[3];
                }
                if (EXTRA && a.traj) {
                    float *yt = a.traj + (int64_t)(k - 1) * 4 * a.n + i;
                    yt[0] = V;
                    yt[a.n] = W;
                    yt[2 * (int64_t)a.n] = ge;
                    yt[3 * (int64_t)a.n] = gi;
                    a.traj_since[(int64_t)(k - 1) * a.n + i] = k - 1 - last;
                }
                if (MODEL == 0 && !refr_lds) frac = lif_frac(a, k - 1 - last);
                const bool fired = fit_step<MODEL>(a, gl, el, cfe, cfi, frac, V, W, ge, gi);
                if (refr_lds) {
                    frac = fired ? frac0 : fnext;
                    since = fired ? 0 : since;
                }
                last = fired ? k : last;
                *vt = V;
                vt += a.n;
                if (EXTRA && a.spikes) a.spikes[(int64_t)(k - 1) * a.n + i] = fired ? 1 : 0;
#pragma unroll
                for (int q = 0; q < 4; q++) x[q] = y[q];
            }
        }
        __syncthreads();
    }
}

// ---- backward -------------------------------------------------------------
// Entries of a segment's map: the adjoint state (V, W, g_exc, g_inh) at its
// start as a function of the one at its end: the columns of V and W, the
// factors of g_exc and g_inh (they reach nothing but themselves), and the
// part that comes from the segment's own dL/dV.
constexpr int kFitMap = 14;

// Replays a segment from its checkpoint: s[0..3][step][lane] = V, W (AdEx) or
// the refractory fraction with the sign bit set on a spike (LIF), g_exc,
// g_inh before each step's integration.
template <int MODEL>
__device__ __forceinline__ void fit_replay(const FitArgs &a, int c, int i, float gl, float el, float cfe,
                                           float cfi, float (*s)[kFitSeg][kFitBlock]) {
    const int lane = (int)threadIdx.x;
    const float *cs = a.ck_state + (int64_t)(c - a.ck_lo) * 4 * a.n;
    float V = cs[i], W = cs[a.n + i], ge = cs[2 * a.n + i], gi = cs[3 * a.n + i];
    const int32_t *ci = a.ck_int + (int64_t)(c - a.ck_lo) * 2 * a.n;
    int last = ci[a.n + i];
    FitEvents ev;
    ev.seek(a, i, ci[i]);
    const int k0 = c * a.seg + 1, k1 = min(a.steps, (c + 1) * a.seg);
    for (int k = k0; k <= k1; k++) {
        ev.apply(k, ge, gi);
        const int j = k - k0;
        s[0][j][lane] = V;
        s[2][j][lane] = ge;
        s[3][j][lane] = gi;
        if (MODEL == 0) {
            const float frac = lif_frac(a, k - 1 - last);
            const bool fired = fit_step<MODEL>(a, gl, el, cfe, cfi, frac, V, W, ge, gi);
            if (fired) last = k;
            s[1][j][lane] = fired ? -frac : frac;
        } else {
            s[1][j][lane] = W;
            fit_step<MODEL>(a, gl, el, cfe, cfi, 1.0f, V, W, ge, gi);
        }
    }
}

// Segments c_lo to c_hi from their kept checkpoints (c_lo is one), one lane
// per (checkpoint, neuron): the forward pass again, its state and event cursor
// written at every segment's start, the cursor also past the last one.
template <int MODEL>
__global__ __launch_bounds__(kFitBlock) void k_fit_expand(FitArgs a) {
    const int64_t q = (int64_t)blockIdx.x * kFitBlock + threadIdx.x;
    const int i = (int)(q % a.n);
    const int64_t c0 = a.c_lo + q / a.n * a.keep;
    if (c0 >= a.c_hi) return;
    const int c1 = (int)min(c0 + a.keep, (int64_t)a.c_hi);
    const float gl = a.gl[i], el = a.el[i];
    const float cfe = expf(-a.h / a.te[i]), cfi = expf(-a.h / a.ti[i]);
    const float *ks = a.kept_state + c0 / a.keep * 4 * a.n;
    float V = ks[i], W = ks[a.n + i], ge = ks[2 * a.n + i], gi = ks[3 * a.n + i];
    const int32_t *ki = a.kept_int + c0 / a.keep * 2 * a.n;
    int last = ki[a.n + i];
    FitEvents ev;
    ev.seek(a, i, ki[i]);
    for (int c = (int)c0; c < c1; c++) {
        float *cs = a.ck_state + (int64_t)(c - a.ck_lo) * 4 * a.n;
        cs[i] = V;
        cs[a.n + i] = W;
        cs[2 * a.n + i] = ge;
        cs[3 * a.n + i] = gi;
        int32_t *ci = a.ck_int + (int64_t)(c - a.ck_lo) * 2 * a.n;
        ci[i] = ev.e;
        ci[a.n + i] = last;
        const int k1 = min(a.steps, (c + 1) * a.seg);
        for (int k = c * a.seg + 1; k <= k1; k++) {
            ev.apply(k, ge, gi);
            const float frac = MODEL == 0 ? lif_frac(a, k - 1 - last) : 1.0f;
            if (fit_step<MODEL>(a, gl, el, cfe, cfi, frac, V, W, ge, gi)) last = k;
        }
    }
    if (c1 == a.c_hi) a.ck_int[(int64_t)(c1 - a.ck_lo) * 2 * a.n + i] = ev.e;
}

// The vector-Jacobian product of one AdEx step (without its reset): (lV, lW,
// lge, lgi) after the step to the same before it.  lp and lc (gradients of
// g_leak, e_leak and of the two decay factors) may be null.
__device__ __forceinline__ void fit_adex_step_vjp(const FitArgs &a, float gl, float el, float cfe, float cfi,
                                                  float Vy, float gey, float giy, const AdexStages &st,
                                                  float &lV, float &lW, float &lge, float &lgi, double *lp,
                                                  double *lc) {
    const float gem = fit_decay(gey, cfe), gim = fit_decay(giy, cfi);
    const float ge2 = fit_decay(gem, cfe), gi2 = fit_decay(gim, cfi);
    const float l4V = lV * a.s6, l4W = lW * a.s6;
    float l3V = 2.0f * lV * a.s6, l3W = 2.0f * lW * a.s6;
    float l2V = l3V, l2W = l3W;
    float l1V = l4V, l1W = l4W;
    float nV = lV, nW = lW;
    float lg2e = lge, lg2i = lgi, lgme = 0.0f, lgmi = 0.0f;
    float lx[4];
    lx[0] = lx[1] = lx[2] = lx[3] = 0.0f;
    fit_adex_vjp(a, gl, el, st.aV[2], ge2, gi2, st.E[3], l4V, l4W, lx, lp);
    nV += lx[0]; nW += lx[1]; l3V += a.dt * lx[0]; l3W += a.dt * lx[1];
    lg2e += lx[2]; lg2i += lx[3];
    lx[0] = lx[1] = lx[2] = lx[3] = 0.0f;
    fit_adex_vjp(a, gl, el, st.aV[1], gem, gim, st.E[2], l3V, l3W, lx, lp);
    nV += lx[0]; nW += lx[1]; l2V += a.h * lx[0]; l2W += a.h * lx[1];
    lgme += lx[2]; lgmi += lx[3];
    lx[0] = lx[1] = lx[2] = lx[3] = 0.0f;
    fit_adex_vjp(a, gl, el, st.aV[0], gem, gim, st.E[1], l2V, l2W, lx, lp);
    nV += lx[0]; nW += lx[1]; l1V += a.h * lx[0]; l1W += a.h * lx[1];
    lgme += lx[2]; lgmi += lx[3];
    lx[0] = lx[1] = lx[2] = lx[3] = 0.0f;
    fit_adex_vjp(a, gl, el, Vy, gey, giy, st.E[0], l1V, l1W, lx, lp);
    nV += lx[0]; nW += lx[1];
    float nge = lx[2], ngi = lx[3];
    if (!(gem < 1e-9f)) { lgme += lg2e * cfe; if (lc) lc[0] += (double)(lg2e * gem); }
    if (!(gim < 1e-9f)) { lgmi += lg2i * cfi; if (lc) lc[1] += (double)(lg2i * gim); }
    if (!(gey < 1e-9f)) { nge += lgme * cfe; if (lc) lc[0] += (double)(lgme * gey); }
    if (!(giy < 1e-9f)) { ngi += lgmi * cfi; if (lc) lc[1] += (double)(lgmi * giy); }
    lV = nV;
    lW = nW;
    lge = nge;
    lgi = ngi;
}

// The affine map of every segment of the launch, one lane per (segment,
// neuron).  The step's coefficients are the float ones of the reverse sweep;
// they are composed in double, so that the adjoint state a segment starts
// from is no further from the exact one than a sweep that walks there.
template <int MODEL>
__global__ __launch_bounds__(kFitBlock) void k_fit_maps(FitArgs a) {
    __shared__ float s[4][kFitSeg][kFitBlock];
    const int lane = (int)threadIdx.x;
    const int64_t q = (int64_t)blockIdx.x * kFitBlock + lane;
    const int c = a.c_lo + (int)(q / a.n), i = (int)(q % a.n);
    if (c >= a.c_hi) return;
    const float gl = a.gl[i], el = a.el[i];
    const float cfe = expf(-a.h / a.te[i]), cfi = expf(-a.h / a.ti[i]);
    fit_replay<MODEL>(a, c, i, gl, el, cfe, cfi, s);
    const int k0 = c * a.seg + 1, k1 = min(a.steps, (c + 1) * a.seg);
    // m[0]: the column of V, m[1]: of W, m[2]: the segment's own part
    double m[3][4] = {{1, 0, 0, 0}, {0, 1, 0, 0}, {0, 0, 0, 0}};
    double de = 1.0, di = 1.0;
    float gv_n = a.grad_v[(int64_t)(k1 - 1) * a.n + i];
    for (int k = k1; k >= k0; k--) {
        const int j = k - k0;
        const float gv = gv_n;
        if (k > k0) gv_n = a.grad_v[(int64_t)(k - 2) * a.n + i];
        float V = s[0][j][lane], x1 = s[1][j][lane], ge = s[2][j][lane], gi = s[3][j][lane];
        m[2][0] += (double)gv;
        if (MODEL == 0) {
            const bool fired = __float_as_uint(x1) >> 31;
            const float frac = fabsf(x1);
            const double c1 = (double)(a.dt * frac * a.inv_c_m);
            const double fV = 1.0 + c1 * (double)(-ge - gi - gl);
            const double fe = c1 * (double)(a.e_exc - V), fi = c1 * (double)(a.e_inh - V);
            const double ce = ge < 1e-9f ? 0.0 : (double)cfe, cg = gi < 1e-9f ? 0.0 : (double)cfi;
#pragma unroll
            for (int r = 0; r < 3; r += 2) {
                const double lV = fired ? 0.0 : m[r][0];
                m[r][0] = lV * fV;
                m[r][2] = lV * fe + m[r][2] * ce;
                m[r][3] = lV * fi + m[r][3] * cg;
            }
            de *= ce;
            di *= cg;
        } else {
            AdexStages st;
            float Vn = V, Wn = x1, gen = ge, gin = gi;
            fit_step<MODEL>(a, gl, el, cfe, cfi, 1.0f, Vn, Wn, gen, gin, &st);
            // rows of the step's Jacobian: unit adjoints of V and of W
            float rV[4] = {1.0f, 0.0f, 0.0f, 0.0f}, rW[4] = {0.0f, 1.0f, 0.0f, 0.0f};
            fit_adex_step_vjp(a, gl, el, cfe, cfi, V, ge, gi, st, rV[0], rV[1], rV[2], rV[3], nullptr, nullptr);
            fit_adex_step_vjp(a, gl, el, cfe, cfi, V, ge, gi, st, rW[0], rW[1], rW[2], rW[3], nullptr, nullptr);
            const float gem = fit_decay(ge, cfe), gim = fit_decay(gi, cfi);
            const double ce = (gem < 1e-9f || ge < 1e-9f) ? 0.0 : (double)cfe * (double)cfe;
            const double cg = (gim < 1e-9f || gi < 1e-9f) ? 0.0 : (double)cfi * (double)cfi;
#pragma unroll
            for (int r = 0; r < 3; r++) {
                const double lV = st.fired ? 0.0 : m[r][0], lW = m[r][1];
                m[r][0] = lV * (double)rV[0] + lW * (double)rW[0];
                m[r][1] = lV * (double)rV[1] + lW * (double)rW[1];
                m[r][2] = lV * (double)rV[2] + lW * (double)rW[2] + m[r][2] * ce;
                m[r][3] = lV * (double)rV[3] + lW * (double)rW[3] + m[r][3] * cg;
            }
            de *= ce;
            di *= cg;
        }
    }
    double *o = a.maps + (int64_t)(c - a.c_lo) * kFitMap * a.n + i;
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int v = 0; v < 4; v++) o[(int64_t)(4 * r + v) * a.n] = m[r][v];
    o[(int64_t)12 * a.n] = de;
    o[(int64_t)13 * a.n] = di;
}

// Per neuron: the adjoint state at the end of every segment of the launch,
// last first, over the first four entries of the segment's map; carry holds
// the state that enters the launch and then the one that leaves it.
__global__ __launch_bounds__(kFitBlock) void k_fit_scan(FitArgs a) {
    const int i = (int)blockIdx.x * kFitBlock + (int)threadIdx.x;
    if (i >= a.n) return;
    double l[4];
#pragma unroll
    for (int v = 0; v < 4; v++) l[v] = a.carry[(int64_t)v * a.n + i];
    // the maps are read four segments ahead: the chain below is short
    constexpr int U = 4;
    const int m = a.c_hi - a.c_lo;
    double nx[U][kFitMap];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int v = 0; v < kFitMap; v++) nx[u][v] = a.maps[((int64_t)max(m - 1 - u, 0) * kFitMap + v) * a.n + i];
    for (int c0 = m - 1; c0 >= 0; c0 -= U) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int c = c0 - u;
            if (c < 0) break;
            double *o = a.maps + (int64_t)c * kFitMap * a.n + i;
            double x[kFitMap];
#pragma unroll
            for (int v = 0; v < kFitMap; v++) x[v] = nx[u][v];
#pragma unroll
            for (int v = 0; v < kFitMap; v++)
                nx[u][v] = a.maps[((int64_t)max(c - U, 0) * kFitMap + v) * a.n + i];
#pragma unroll
            for (int v = 0; v < 4; v++) o[(int64_t)v * a.n] = l[v];
            const double lV = l[0], lW = l[1];
            l[0] = x[0] * lV + x[4] * lW + x[8];
            l[1] = x[1] * lV + x[5] * lW + x[9];
            l[2] = x[2] * lV + x[6] * lW + x[10] + x[12] * l[2];
            l[3] = x[3] * lV + x[7] * lW + x[11] + x[13] * l[3];
        }
    }
#pragma unroll
    for (int v = 0; v < 4; v++) a.carry[(int64_t)v * a.n + i] = l[v];
}

// Reverse sweep of every segment of the launch from the adjoint state at its
// end, one lane per (segment, neuron): parameter gradients of the segment,
// and the conductances' adjoints after each step's inputs (the gradient of a
// weight is their sum over its events).
template <int MODEL>
__global__ __launch_bounds__(kFitBlock) void k_fit_sweep(FitArgs a) {
    __shared__ float s[4][kFitSeg][kFitBlock];
    const int lane = (int)threadIdx.x;
    const int64_t q = (int64_t)blockIdx.x * kFitBlock + lane;
    const int c = a.c_lo + (int)(q / a.n), i = (int)(q % a.n);
    if (c >= a.c_hi) return;
    const float gl = a.gl[i], el = a.el[i];
    const float cfe = expf(-a.h / a.te[i]), cfi = expf(-a.h / a.ti[i]);
    fit_replay<MODEL>(a, c, i, gl, el, cfe, cfi, s);
    const int k0 = c * a.seg + 1, k1 = min(a.steps, (c + 1) * a.seg);
    const double *l0 = a.maps + (int64_t)(c - a.c_lo) * kFitMap * a.n + i;
    float lV = (float)l0[0], lW = (float)l0[(int64_t)a.n], lge = (float)l0[2 * (int64_t)a.n],
          lgi = (float)l0[3 * (int64_t)a.n];
    double lp[2] = {0.0, 0.0}, lc[2] = {0.0, 0.0};
    float gv_n = a.grad_v[(int64_t)(k1 - 1) * a.n + i];
    float *lg = a.lg + (int64_t)(k1 - 1 - c * a.seg + (int64_t)(c - a.c_lo) * a.seg) * 2 * a.n + i;
    for (int k = k1; k >= k0; k--) {
        const int j = k - k0;
        const float gv = gv_n;
        if (k > k0) gv_n = a.grad_v[(int64_t)(k - 2) * a.n + i];
        const float V = s[0][j][lane], x1 = s[1][j][lane], ge = s[2][j][lane], gi = s[3][j][lane];
        lV += gv;
        if (MODEL == 0) {
            const float frac = fabsf(x1);
            if (__float_as_uint(x1) >> 31) {
                lp[1] += (double)lV;
                lV = 0.0f;
            }
            const float ld = a.dt * lV;
            const float nV = lV + ld * frac * (-ge - gi - gl) * a.inv_c_m;
            float nge = ld * frac * (a.e_exc - V) * a.inv_c_m;
            float ngi = ld * frac * (a.e_inh - V) * a.inv_c_m;
            lp[0] += (double)(ld * frac * (el - V) * a.inv_c_m);
            lp[1] += (double)(ld * frac * gl * a.inv_c_m);
            if (!(ge < 1e-9f)) {
                nge += lge * cfe;
                lc[0] += (double)(lge * ge);
            }
            if (!(gi < 1e-9f)) {
                ngi += lgi * cfi;
                lc[1] += (double)(lgi * gi);
            }
            lV = nV;
            lge = nge;
            lgi = ngi;
        } else {
            AdexStages st;
            float Vn = V, Wn = x1, gen = ge, gin = gi;
            fit_step<MODEL>(a, gl, el, cfe, cfi, 1.0f, Vn, Wn, gen, gin, &st);
            if (st.fired) lV = 0.0f;
            fit_adex_step_vjp(a, gl, el, cfe, cfi, V, ge, gi, st, lV, lW, lge, lgi, lp, lc);
        }
        lg[0] = lge;
        lg[a.n] = lgi;
        lg -= 2 * (int64_t)a.n;
    }
    double *o = a.part + (int64_t)(c - a.c_lo) * 4 * a.n + i;
    o[0] = lp[0];
    o[(int64_t)a.n] = lp[1];
    o[2 * (int64_t)a.n] = lc[0];
    o[3 * (int64_t)a.n] = lc[1];
}

// One workgroup per neuron: the segments' parameter gradients added to the
// sums in carry[4..7], and each synapse's weight gradient over its events,
// both from the last step to the first.  After the launch that holds the
// first segment the parameter gradients are complete.
__global__ __launch_bounds__(kFitGradBlock) void k_fit_grads(FitArgs a) {
    constexpr int T = kFitGradBlock;
    __shared__ int32_t s_syn[T];
    __shared__ float s_val[T];
    __shared__ double s_red[4][T / 4];
    const int i = (int)blockIdx.x, tid = (int)threadIdx.x;
    const bool first = a.c_hi == a.segs, final = a.c_lo == 0;
    // parameter gradients: T/4 lanes per parameter, each a contiguous range
    // of segments, then the ranges in order
    {
        const int v = tid / (T / 4), t = tid % (T / 4), m = a.c_hi - a.c_lo;
        const int hi = m - (int)((int64_t)m * t / (T / 4)), lo = m - (int)((int64_t)m * (t + 1) / (T / 4));
        double x = 0.0;
        for (int c = hi - 1; c >= lo; c--) x += a.part[((int64_t)c * 4 + v) * a.n + i];
        s_red[v][t] = x;
    }
    __syncthreads();
    if (tid < 4) {
        double x = first ? 0.0 : a.carry[(int64_t)(4 + tid) * a.n + i];
        for (int t = 0; t < T / 4; t++) x += s_red[tid][t];
        // the initial state is V = e_leak; decay factors are exp(-h/tau), so
        // d/dtau = cf * h / tau^2
        if (final) {
            if (tid == 1) x += a.carry[i];
            if (tid >= 2) {
                const float tau = tid == 2 ? a.te[i] : a.ti[i];
                const float cf = expf(-a.h / tau);
                x = x * (double)cf * (double)a.h / ((double)tau * (double)tau);
            }
            a.grad_par[(int64_t)tid * a.n + i] = (float)x;
        } else {
            a.carry[(int64_t)(4 + tid) * a.n + i] = x;
        }
    }
    const int e_lo = a.ck_int[(int64_t)(a.c_lo - a.ck_lo) * 2 * a.n + i];
    const int e_hi = a.ck_int[(int64_t)(a.c_hi - a.ck_lo) * 2 * a.n + i];
    const uint8_t *ty = a.syn_type + (int64_t)i * a.n_syn;
    float *gw = a.grad_w + (int64_t)i * a.n_syn;
    for (int s0 = 0; s0 < a.n_syn; s0 += T) {
        const int s = s0 + tid;
        float g = (first || s >= a.n_syn) ? 0.0f : gw[s];
        for (int e1 = e_hi; e1 > e_lo; e1 -= T) {
            const int e = e1 - 1 - tid;
            __syncthreads();
            s_syn[tid] = -1;
            if (e >= e_lo) {
                const int sy = a.ev_syn[e];
                s_syn[tid] = sy;
                s_val[tid] = a.lg[((int64_t)(a.ev_step[e] - 1 - a.c_lo * a.seg) * 2 + (ty[sy] == 0 ? 0 : 1)) * a.n + i];
            }
            __syncthreads();
            const int m = min(T, e1 - e_lo);
            for (int u = 0; u < m; u++)
                if (s_syn[u] == s) g += s_val[u];
        }
        if (s < a.n_syn) gw[s] = g;
    }
}

}  // namespace edl
