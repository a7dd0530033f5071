// Per-element update rules shared by the neuron / filter kernels and by GEMV epilogues.
#pragma once

#include "nhip_common.h"
#include "small_arg_math.h"

// One population of LIF neurons driven by one output item of a GEMV: element
// offsets of its state, and its parameters as float bits or (pflags bit set) as the
// element offset of a per-neuron vector.
struct LifPop {
    int v_start, w_start, s_start;
    int decay;                  // float bits of -expm1(-dtu / tau), valid with LIF_POP_DECAY
    int tau, ref, amp, pflags;  // bit 0/1/2 of pflags: tau/ref/amp is a per-neuron vector
};
constexpr int LIF_POP_ENABLED = 1 << 8;  // pflags: the item has a population at all
constexpr int LIF_POP_DECAY = 1 << 9;    // pflags: `decay` is set (one tau, upsample == 1)
// pflags: nothing but this epilogue reads the population's input current (the host's word),
// so the launch does not store it; the host recomputes it when somebody asks
constexpr int LIF_POP_NO_J = 1 << 10;
// pflags: nothing but launches that visit active columns reads the population's spikes (the
// host's word), so the large-item launch stores them as one bit per neuron -- a 64-bit word
// per 64 neurons, in the first words of the signal's own memory (s_start even, the rows of
// every task starting at a multiple of 64) -- instead of a float each: a sixteenth of a
// percent of the bytes, and writes next to a read stream cost about three times theirs
constexpr int LIF_POP_BITS = 1 << 11;
// pflags: the small-item launch also leaves the population's spikes as one bit per neuron, in
// LifArgs::mask, for a sparse product (EPI_LIF_BITS); the floats are stored as always.  A launch of its
// own for the bits of 100,000 neurons takes 4.6 us of a step of 28.
constexpr int LIF_POP_MASK = 1 << 12;

// State arrays and constants of a fused LIF update (all populations of a launch).
struct LifArgs {
    const LifPop* pops;  // one per GEMV item
    float dtu, dt_inv;   // dt / upsample, 1 / dt
    int upsample;
    float* V;
    float* W;
    float* S;
    const float* TAU;
    const float* REF;
    const float* AMP;
    // input sums formed by the launch itself (large-item kernel with compile-time shapes):
    // the vector operand of an item's first dot product is the sum of `n` vectors times
    // scalars, parts[begin .. begin + n) = {vector start, scalar start} in the X buffer;
    // begin / n ride in the spare words of the task record.  Null: no item has one.
    const int2* parts;
    // the same for the small-item kernel, whose task records have no spare words: per GEMV
    // item {first part, number of parts} (0 parts: the operand is read as usual).  Null: none.
    const int2* sum_ranges;
    // first-order filters of the populations' OLD spikes, stepped by the task that is about
    // to overwrite those spikes (large-item kernel with compile-time shapes, the instance for
    // it): per GEMV item {f_start, a0 bits, b0 bits, flags} -- flags bit 0: the item's
    // population has such a filter, bit 1: it has a denominator coefficient; element i of the
    // filter output is Fdef[f_start + i] = b0 * S_old[i] - a0 * Fdef[f_start + i].  This is the
    // filter step that follows the neuron update of the PREVIOUS step, moved to where its
    // input is about to be replaced (see nhip_gemv_tile_lif_deferred).  Null: none.
    const int4* deferred;
    float* Fdef;
    // neuron types other than the plain LIF (EPI_NEURON): `pops` then points at NeuronPop records
    float* N;            // adaptation states
    float dt;
    unsigned* mask;      // EPI_LIF_BITS: a bit per neuron of the population with LIF_POP_MASK
};

// One population of neurons of another type than the plain LIF, driven by one output item of a
// GEMV: element offsets of its state and float bits of its parameters (one value per population).
struct NeuronPop {
    int v_start, w_start, out_start, n_start;  // voltage, refractory time, output (S or R), adaptation
    int tau, ref, amp, tau_n;
    int inc_n, kind, flags, pad;               // flags: LIF_POP_ENABLED, LIF_POP_NO_J
};
enum { NEURON_LIF_RATE = 1, NEURON_ALIF = 2, NEURON_ALIF_RATE = 3, NEURON_RELU = 4,
       NEURON_SPIKING_RELU = 5, NEURON_SIGMOID = 6 };
__device__ __forceinline__ bool neuron_has_v(int kind) { return kind == NEURON_ALIF || kind == NEURON_SPIKING_RELU; }
__device__ __forceinline__ bool neuron_has_w(int kind) { return kind == NEURON_ALIF; }
__device__ __forceinline__ bool neuron_has_n(int kind) { return kind == NEURON_ALIF || kind == NEURON_ALIF_RATE; }

__device__ __forceinline__ float lif_param(int word, bool is_vector, const float* data, int i) {
    return is_vector ? data[(size_t)word + i] : nhip_bits(word);
}

// The update follows the reference kernel text (clra_nonlinearities.py:1086-1133)
// operation by operation: refractory countdown, partial-step integration time,
// exponential-Euler voltage step, threshold test with spike-time interpolation.
// Sums that follow a product are written with explicit rounded operations so
// that the compiler cannot fuse them differently from one build to the next.
// expm1 and log1p are evaluated in double and rounded once to float: that is the
// correctly rounded float32 value (the best any float implementation can return),
// so every conforming host or device math library gives the same bits and spike
// decisions do not depend on the library.  Their arguments are small here (at most
// dt / tau in magnitude), which `nhip_expm1` / `nhip_log1p` use: a short series for
// |x| <= 1/16, the library routine otherwise.  Returns whether the neuron spiked.
__device__ __forceinline__ bool lif_step(float j, float& v, float& w, float tau, float ref,
                                         float dtu, int upsample) {
    bool spiked = false;
    for (int u = 0; u < upsample; ++u) {
        w -= dtu;
        const float delta_t = (w > dtu) ? 0.0f : (w < 0.0f) ? dtu : dtu - w;
        const float dv = __fmul_rn(-(float)nhip_expm1((double)__fdiv_rn(-delta_t, tau)), j - v);
        v = __fadd_rn(v, dv);
        if (v > 1.0f) {
            const float t_spike =
                __fadd_rn(dtu, __fmul_rn(tau, (float)nhip_log1p((double)__fdiv_rn(-(v - 1.0f), j - 1.0f))));
            w = ref + t_spike;
            v = 0.0f;
            spiked = true;
        } else if (v < 0.0f) {
            v = 0.0f;
        }
    }
    return spiked;
}

// The same for one time constant and no sub-steps: the factor of a whole step comes with the population
// (LIF_POP_DECAY), that of no time is +0, and a wave in which no neuron leaves its refractory period or spikes
// skips the evaluations in double.
__device__ __forceinline__ bool lif_step_decay(float j, float& v, float& w, float decay, float tau, float ref,
                                               float dtu) {
    w -= dtu;
    const float delta_t = (w > dtu) ? 0.0f : (w < 0.0f) ? dtu : dtu - w;
    float factor = delta_t == dtu ? decay : 0.0f;
    if (delta_t != dtu && delta_t != 0.0f) factor = -(float)nhip_expm1((double)__fdiv_rn(-delta_t, tau));
    v = __fadd_rn(v, __fmul_rn(factor, j - v));
    const bool spiked = v > 1.0f;
    if (spiked) {
        const float t_spike =
            __fadd_rn(dtu, __fmul_rn(tau, (float)nhip_log1p((double)__fdiv_rn(-(v - 1.0f), j - 1.0f))));
        w = ref + t_spike;
        v = 0.0f;
    } else if (v < 0.0f) {
        v = 0.0f;
    }
    return spiked;
}

// Adaptive LIF (clra_nonlinearities.py:1086-1133 with `adaptive`): the LIF update with
// j - n in place of j in the voltage step, then n += (dt / tau_n) (inc_n s - n).  Returns s.
__device__ __forceinline__ float alif_step(float j, float& v, float& w, float& n, float tau, float ref,
                                           float amp, float tau_n, float inc_n, float dt, float dtu,
                                           float dt_inv, int upsample) {
    bool spiked = false;
    for (int u = 0; u < upsample; ++u) {
        w -= dtu;
        const float delta_t = (w > dtu) ? 0.0f : (w < 0.0f) ? dtu : dtu - w;
        const float dv = __fmul_rn(-(float)nhip_expm1((double)__fdiv_rn(-delta_t, tau)), (j - n) - v);
        v = __fadd_rn(v, dv);
        if (v > 1.0f) {
            // the spike time interpolates with the unadapted current, as the reference does
            const float t_spike = __fadd_rn(
                dtu, __fmul_rn(tau, (float)nhip_log1p((double)__fdiv_rn(-(v - 1.0f), j - 1.0f))));
            w = ref + t_spike;
            v = 0.0f;
            spiked = true;
        } else if (v < 0.0f) {
            v = 0.0f;
        }
    }
    const float s = spiked ? __fmul_rn(amp, dt_inv) : 0.0f;
    n = __fadd_rn(n, __fmul_rn(__fdiv_rn(dt, tau_n), __fsub_rn(__fmul_rn(inc_n, s), n)));
    return s;
}

// LIF rate (clra_nonlinearities.py:1174-1184): j <= 1 gives 1/0 = inf, log1p(inf) = inf, amp/inf = 0.
__device__ __forceinline__ float lif_rate(float current, float tau, float ref, float amp) {
    const float j = fmaxf(current - 1.0f, 0.0f);
    const float denom = __fadd_rn(ref, __fmul_rn(tau, (float)nhip_log1p((double)__fdiv_rn(1.0f, j))));
    return __fdiv_rn(amp, denom);
}

// Adaptive LIF rate (clra_nonlinearities.py:1174-1188 with `adaptive`).
__device__ __forceinline__ float alif_rate_step(float current, float& n, float tau, float ref, float amp,
                                                float tau_n, float inc_n, float dt) {
    const float r = lif_rate(current - n, tau, ref, amp);
    n = __fadd_rn(n, __fmul_rn(__fdiv_rn(dt, tau_n), __fsub_rn(__fmul_rn(inc_n, r), n)));
    return r;
}

// Rectified linear R = amp max(J, 0) (clra_nonlinearities.py:1238-1258).
__device__ __forceinline__ float relu(float j, float amp) { return __fmul_rn(amp, fmaxf(j, 0.0f)); }

// Spiking rectified linear (:1200-1235): V += dt max(J, 0), spikes = floor(V), V -= spikes,
// S = amp spikes / dt.
__device__ __forceinline__ float spiking_relu_step(float j, float& v, float amp, float dt, float dt_inv) {
    v = __fadd_rn(v, (j > 0.0f) ? __fmul_rn(dt, j) : 0.0f);
    const float n_spikes = floorf(v);
    v = v - n_spikes;
    return __fmul_rn(__fmul_rn(amp, n_spikes), dt_inv);
}

// Sigmoid R = 1 / (ref (1 + exp(-J))) with the reference's cut-offs at -88 and 15 (:1261-1283; exp
// in double, rounded once, so that the value does not depend on the math library).
__device__ __forceinline__ float sigmoid(float j, float ref) {
    return (j < -88.0f) ? 0.0f
           : (j > 15.0f) ? __fdiv_rn(1.0f, ref)
                         : __fdiv_rn(1.0f, __fmul_rn(ref, __fadd_rn(1.0f, (float)exp((double)-j))));
}

// Work-list rows of the neuron kernels: a block of <= 512 neurons of one population.
struct LifDesc {
    int j_start, v_start, w_start, s_start;
    int count, tau, ref, amp;  // tau/ref/amp: float bits, or element offsets (see pflags)
    int pflags, p0, p1, p2;    // bit 0/1/2: tau/ref/amp is a per-neuron vector
};
struct RateDesc { int j_start, r_start, count, tau, ref, amp, pflags, pad; };

// One thread per neuron; the update itself is `lif_step`.  dtu = dt / upsample.
__device__ __forceinline__ void lif_block(const LifDesc d, float dtu, float dt_inv, int upsample,
                                          const float* J, float* V, float* W, float* S,
                                          const float* __restrict__ TAU,
                                          const float* __restrict__ REF,
                                          const float* __restrict__ AMP, int tid) {
    for (int i = tid; i < d.count; i += NHIP_WG) {
        const float j = J[(size_t)d.j_start + i];
        float v = V[(size_t)d.v_start + i];
        float w = W[(size_t)d.w_start + i];
        const float tau = lif_param(d.tau, d.pflags & 1, TAU, i);
        const float ref = lif_param(d.ref, d.pflags & 2, REF, i);
        const float amp = lif_param(d.amp, d.pflags & 4, AMP, i);
        const bool spiked = lif_step(j, v, w, tau, ref, dtu, upsample);
        V[(size_t)d.v_start + i] = v;
        W[(size_t)d.w_start + i] = w;
        S[(size_t)d.s_start + i] = spiked ? __fmul_rn(amp, dt_inv) : 0.0f;
    }
}

__device__ __forceinline__ void lif_rate_block(const RateDesc d, const float* J, float* R,
                                               const float* __restrict__ TAU,
                                               const float* __restrict__ REF,
                                               const float* __restrict__ AMP, int tid) {
    for (int i = tid; i < d.count; i += NHIP_WG) {
        const float tau = lif_param(d.tau, d.pflags & 1, TAU, i);
        const float ref = lif_param(d.ref, d.pflags & 2, REF, i);
        const float amp = lif_param(d.amp, d.pflags & 4, AMP, i);
        R[(size_t)d.r_start + i] = lif_rate(J[(size_t)d.j_start + i], tau, ref, amp);
    }
}

// LIF update of neuron i of population p with input current j (GEMV epilogue);
// v and w are the neuron's voltage and refractory time, read earlier
__device__ __forceinline__ bool lif_epilogue(const LifArgs& a, const LifPop& p, int i, float j,
                                             float v, float w) {
    const float tau = lif_param(p.tau, p.pflags & 1, a.TAU, i);
    const float ref = lif_param(p.ref, p.pflags & 2, a.REF, i);
    const float amp = lif_param(p.amp, p.pflags & 4, a.AMP, i);
    const bool spiked = lif_step(j, v, w, tau, ref, a.dtu, a.upsample);
    a.V[(size_t)p.v_start + i] = v;
    a.W[(size_t)p.w_start + i] = w;
    a.S[(size_t)p.s_start + i] = spiked ? __fmul_rn(amp, a.dt_inv) : 0.0f;
    return spiked;
}

// Update of neuron i of a population of another type with input current j (GEMV epilogue); v, w and n
// are its states, read earlier (0 where the type has none).  The same functions as the neuron kernels.
__device__ __forceinline__ void neuron_epilogue(const LifArgs& a, const NeuronPop& p, int i, float j,
                                                float v, float w, float n) {
    const float tau = nhip_bits(p.tau), ref = nhip_bits(p.ref), amp = nhip_bits(p.amp);
    float out;
    switch (p.kind) {
        case NEURON_LIF_RATE: out = lif_rate(j, tau, ref, amp); break;
        case NEURON_ALIF:
            out = alif_step(j, v, w, n, tau, ref, amp, nhip_bits(p.tau_n), nhip_bits(p.inc_n), a.dt,
                            a.dtu, a.dt_inv, a.upsample);
            break;
        case NEURON_ALIF_RATE:
            out = alif_rate_step(j, n, tau, ref, amp, nhip_bits(p.tau_n), nhip_bits(p.inc_n), a.dt);
            break;
        case NEURON_RELU: out = relu(j, amp); break;
        case NEURON_SPIKING_RELU: out = spiking_relu_step(j, v, amp, a.dt, a.dt_inv); break;
        default: out = sigmoid(j, ref); break;
    }
    a.S[(size_t)p.out_start + i] = out;
    if (neuron_has_v(p.kind)) a.V[(size_t)p.v_start + i] = v;
    if (neuron_has_w(p.kind)) a.W[(size_t)p.w_start + i] = w;
    if (neuron_has_n(p.kind)) a.N[(size_t)p.n_start + i] = n;
}

// Filters fed by one output item of a GEMV (a decoded value and the synapses of the
// connections that carry it): y = b0 x - a0 y, or y = b0 x; or, with FILTER_SECOND_ORDER bits in
// `na`, one with two coefficients on either side, whose further coefficients and state are the
// FilterSecond record in the rows (na >> FILTER_SECOND_SHIFT) of the table of targets.
struct FilterTarget { int y_start, a_bits, b_bits, na; };
constexpr int FILTER_NA = 3, FILTER_NB2 = 4, FILTER_SECOND_SHIFT = 3;
struct FilterSecond {          // two rows of the table of targets
    int a1_bits, b1_bits, n, pad;
    float* state;              // x[t-1], y[t-1], y[t-2]: n elements each
    int pad2, pad3;
};

struct FilterArgs {
    const int2* item_targets;     // per GEMV item: {first target, number of targets}
    const FilterTarget* targets;
    float* F;                     // buffer that holds the filter outputs
    // matrices a learning rule updates in place while the launch streams them (large-item
    // kernel with compile-time shapes, the instance for it): per TASK {e_start, f_start,
    // alpha bits, flags}; with flags bit 0 set, element (i, j) of the task's matrix becomes
    // A + (alpha * X[e_start + i]) * X[f_start + j] after its old value has gone into the
    // sums (see nhip_gemv_tile_filter_learn).  Null: none.
    const int4* learn;
};

// The step of one filter for its element i: x is the fresh input, f_old the output's old value;
// returns the new one.  Rounded products and sums in the order of the filter kernel
// (clra_nonlinearities.py:630-711: b0 x [+ b1 x'] [- a0 y] [- a1 y'']).  A second-order filter keeps
// its two older outputs itself (the ring buffers of the launch it replaces do the same: y[t-2] is
// what the filter computed, also where somebody has written its output since) and shifts them
// instead of moving positions: the rows of an item are stepped by many groups, none of which could
// move a position that the others still read.
// As a launch of their own, second-order synapses of 48 decoded vectors of 32 took 5.2 us of a step.
// SECOND: false for launches whose targets are all of first order.
template <bool SECOND>
__device__ __forceinline__ float filter_step(const FilterTarget* __restrict__ targets, const FilterTarget& t,
                                             int i, float x, float f_old) {
    const float bx = __fmul_rn(nhip_bits(t.b_bits), x);
    if (!SECOND || (t.na >> FILTER_SECOND_SHIFT) == 0)
        return t.na ? __fsub_rn(bx, __fmul_rn(nhip_bits(t.a_bits), f_old)) : bx;
    const FilterSecond e = *reinterpret_cast<const FilterSecond*>(targets + (t.na >> FILTER_SECOND_SHIFT));
    float* x1 = e.state + i;
    float* y1 = x1 + e.n;
    float* y2 = y1 + e.n;
    const float x_1 = *x1, y_1 = *y1, y_2 = *y2;
    float y = bx;
    if (t.na & FILTER_NB2) y = __fadd_rn(y, __fmul_rn(nhip_bits(e.b1_bits), x_1));
    if (t.na & FILTER_NA) y = __fsub_rn(y, __fmul_rn(nhip_bits(t.a_bits), f_old));
    if ((t.na & FILTER_NA) > 1) y = __fsub_rn(y, __fmul_rn(nhip_bits(e.a1_bits), y_2));
    *x1 = x;
    *y1 = y;
    *y2 = y_1;
    return y;
}

// Filter step of element i of every target of a GEMV item whose fresh output is x.
template <bool SECOND>
__device__ __forceinline__ void filter_epilogue(const FilterArgs& a, int2 range, int i, float x) {
    for (int q = 0; q < range.y; ++q) {
        const FilterTarget t = a.targets[range.x + q];
        float* f = a.F + (size_t)t.y_start + i;
        *f = filter_step<SECOND>(a.targets, t, i, x, *f);
    }
}

// What a GEMV launch does with a finished output row besides storing it.
// EPI_NEURON: the update of a neuron of another type than the plain LIF (an instance of its own: the
// LIF instances keep their registers, and their compacted update of the rare cases).
// EPI_FILTER2: EPI_FILTER where a target is of second order (in the instances of EPI_FILTER the code
// for it cost launches without one 1-3 % of a step).
// EPI_LIF_BITS: EPI_LIF where a population's spikes are wanted as bits too.
enum { EPI_NONE = 0, EPI_LIF = 1, EPI_FILTER = 2, EPI_NEURON = 3, EPI_FILTER2 = 4, EPI_LIF_BITS = 5 };
constexpr bool epi_lif(int epi) { return epi == EPI_LIF || epi == EPI_LIF_BITS; }
constexpr bool epi_filters(int epi) { return epi == EPI_FILTER || epi == EPI_FILTER2; }
struct EpilogueArgs {
    LifArgs lif;
    FilterArgs filter;
};
