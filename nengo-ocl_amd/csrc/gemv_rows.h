// The reference-order GEMV for small items as a block function (what one 256-thread
// group does for group index `block`): used by its own kernel and by the sequence
// kernel that runs several short operations of a step in one launch.
#pragma once

#include "nhip_common.h"
#include "gemv_types.h"
#include "neuron_math.h"

// Element q of lane p of a quad of lanes and element p of lane q change places (all four lanes are active).
__device__ __forceinline__ void transpose_quad(float4& v, int lane) {
    constexpr int XOR1 = 0xB1, XOR2 = 0x4E;  // quad_perm [1,0,3,2] and [2,3,0,1]
#define NHIP_QUAD(x, ctrl) __int_as_float(__builtin_amdgcn_update_dpp( \
    0, __float_as_int(x), ctrl, 0xF, 0xF, true))
    const bool b0 = lane & 1, b1 = lane & 2;
    // (every exchange before its choice: a lane that is switched off gives nothing)
    const float x1 = NHIP_QUAD(v.x, XOR1), y1 = NHIP_QUAD(v.y, XOR1), z1 = NHIP_QUAD(v.z, XOR1), w1 = NHIP_QUAD(v.w, XOR1);
    const float a0 = b0 ? y1 : v.x, a1 = b0 ? v.y : x1, a2 = b0 ? w1 : v.z, a3 = b0 ? v.w : z1;
    const float x2 = NHIP_QUAD(a0, XOR2), y2 = NHIP_QUAD(a1, XOR2), z2 = NHIP_QUAD(a2, XOR2), w2 = NHIP_QUAD(a3, XOR2);
    v.x = b1 ? z2 : a0;
    v.y = b1 ? w2 : a1;
    v.z = b1 ? a2 : x2;
    v.w = b1 ? a3 : y2;
#undef NHIP_QUAD
}

// ---------------------------------------------------------------- reference order, small items
// One output row per task (task = {item, row, 1, 0}); a wave takes 64 / LPR
// consecutive tasks, LPR lanes each, whatever items they belong to -- thousands of
// one-row items (decoders of small populations) fill waves as well as a few tall ones.
// Sums are formed in the order of the reference's block kernel (clra_gemv.py:1043-1058,
// :1148-1153): per 128-column tile four strided partial sums, one fused multiply-add
// per element, (s0+s2)+(s1+s3), tiles in order onto beta*y_in, gamma last.
//   LPR = 4: lane j of a row carries partial sum j; any number of columns.
//   LPR = 64, 256: a wave, or the whole group, on one row: four lanes per 128-column tile, so
//            sixteen tiles (64) side by side; the tile sums are then added in order.  For
//            launches of few rows of many columns, where four lanes (or a wave of the
//            large-item kernel that walks whole rows) would leave most of the device idle.
//   LPR = 1: one lane per row, for items whose dot products all have <= 4 columns
//            (vector sums, "scalar times vector" increments): the four partial sums are
//            the (up to) four products themselves.
// These launches are latency bound (a wave or two per SIMD, each a chain of dependent
// reads): the records of four dot products and, when those have at most four columns,
// all their operands are fetched together before the sums are formed in order; wider
// dot products fetch the operands of 8 steps of a partial sum at a time; and what the
// epilogue needs (population record, old neuron state, first filter target and its old
// value) is requested as soon as the task is known, not after the sums.  Task, item and
// dot records are per-lane values on purpose (different rows of a wave may belong to
// different items).
// EPI: what happens to a finished row besides being stored -- nothing, the update
// of the neuron whose input current the row is (LIF, or another type), or the step of the first-order filters
// fed by the row (the same epilogues as the kernel for large items has; small
// populations and low-dimensional decoded values save a launch the same way).
// WIDE: the task table holds GemvRowTask records.
// WAVE_TASK (with LPR = 1 and WIDE): a task is up to 64 consecutive rows of one item (n_rows) and
// takes a whole wave, lane l the row row0 + l.  Launches of very many thin rows (hundreds of
// thousands of neurons of one- to four-dimensional populations) otherwise read a record per
// row; here the record is the wave's: every lane reads the same addresses for the task, the
// item's dot products, its population and its input sum, and the parts of an input sum are
// fetched by the lanes side by side instead of in rounds.
template <int LPR, int EPI = EPI_NONE, bool WIDE = false, bool WAVE_TASK = false>
__device__ __forceinline__ void gemv_rows_ref_block(
    const GemvItem* __restrict__ items, const float4* __restrict__ coefs,
    const GemvDot* __restrict__ dots, const GemvTask* __restrict__ tasks, int n_tasks,
    const float* A, const float* X, const float* Yin, float* Y, int block, int tid,
    const EpilogueArgs* epi = nullptr)
{
    constexpr int TILE = 128;
    constexpr int QUAD_MIN_TASKS = 4 * 256;  // rows that give every compute unit of the card four waves
    constexpr bool NEURONS = epi_lif(EPI) || EPI == EPI_NEURON;
    constexpr int BATCH = 4;             // dot products whose operands are fetched together
    constexpr int CHUNK = 8;             // steps of a partial sum whose operands are fetched together
    constexpr int ROWS = LPR > NHIP_WAVE ? 1 : NHIP_WAVE / LPR;  // rows (tasks) per wave
    constexpr int PER_LANE = LPR > 4 ? 1 : 4 / LPR;  // elements of a <= 4 column dot product per lane
    static_assert(!WAVE_TASK || (LPR == 1 && WIDE), "tasks of several rows: one lane per row, wide records");
    const int lane = tid & (NHIP_WAVE - 1);
    const int lir = LPR > NHIP_WAVE ? tid : lane % LPR;
    const int wave_slot = block * (NHIP_WG / NHIP_WAVE) + __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slot = LPR > NHIP_WAVE ? block : WAVE_TASK ? wave_slot : wave_slot * ROWS + lane / LPR;
    bool valid = slot < n_tasks;
    GemvTask task;
    GemvItem it;
    float4 cf;
    int wide_pad = 0;
    if (WIDE) {
        const GemvRowTask rt = reinterpret_cast<const GemvRowTask*>(tasks)[valid ? slot : n_tasks - 1];
        task = rt.task;
        it = rt.item;
        cf = make_float4(rt.alpha, rt.beta, rt.gamma, 0.0f);
        wide_pad = rt.pad;
    } else {
        task = tasks[valid ? slot : n_tasks - 1];
        it = items[task.item];
        cf = coefs[task.item];
    }
    int r = task.row0;
    if (WAVE_TASK) {  // a lane past the task's rows keeps the last row's addresses and stores nothing
        valid = valid && lane < task.n_rows;
        r = task.row0 + min(lane, task.n_rows - 1);
    }
    const int n_dots = valid ? it.n_dots : 0;
    // epilogue operands, fetched ahead (no branch around the loads: a row without a
    // population or a target reads the first element of the buffer instead)
    LifPop pop = {};
    NeuronPop npop = {};
    float v_old = 0.0f, w_old = 0.0f, n_old = 0.0f;
    int2 f_range = make_int2(0, 0);
    FilterTarget f_first = {};
    float f_old = 0.0f;
    if (epi_lif(EPI)) {
        pop = epi->lif.pops[task.item];
        // where the neuron's state is: from the task record if it says so (the state is
        // then requested together with the population record, not after it)
        const bool enabled = (WIDE ? wide_pad : pop.pflags) & LIF_POP_ENABLED;
        v_old = epi->lif.V[enabled ? (size_t)(WIDE ? task.pad : pop.v_start) + r : 0];
        w_old = epi->lif.W[enabled ? (size_t)(WIDE ? it.pad : pop.w_start) + r : 0];
    }
    if (EPI == EPI_NEURON) {
        npop = reinterpret_cast<const NeuronPop*>(epi->lif.pops)[task.item];
        v_old = epi->lif.V[neuron_has_v(npop.kind) ? (size_t)npop.v_start + r : 0];
        w_old = epi->lif.W[neuron_has_w(npop.kind) ? (size_t)npop.w_start + r : 0];
        n_old = epi->lif.N[neuron_has_n(npop.kind) ? (size_t)npop.n_start + r : 0];
    }
    if (epi_filters(EPI)) {
        f_range = WIDE ? make_int2(task.pad, it.pad) : epi->filter.item_targets[task.item];
        f_first = epi->filter.targets[f_range.y > 0 ? f_range.x : 0];
        f_old = epi->filter.F[f_range.y > 0 ? (size_t)f_first.y_start + r : 0];
    }
    float sum = cf.y * Yin[it.yin_start + (size_t)r * it.yin_stride0];
    // Launches with neurons that form input sums themselves: the vector operand of the item's first
    // dot product (at most 4 columns), or the whole row of an item without dot products, is
    // (...(0 + v_0[c] s_0) + v_1[c] s_1) + ..., what this kernel computes for
    // Y = 0 * Y + sum_k v_k s_k as a launch of its own
    int2 sum_range = make_int2(0, 0);
    if (NEURONS && epi->lif.sum_ranges != nullptr && (WAVE_TASK ? slot < n_tasks : valid))
        sum_range = epi->lif.sum_ranges[task.item];
    if (WAVE_TASK)  // the same for all lanes of the wave (the lanes past the task's rows take part)
        sum_range = make_int2(__builtin_amdgcn_readfirstlane(sum_range.x),
                              __builtin_amdgcn_readfirstlane(sum_range.y));
    // WAVE_TASK: element c of the sum with c the same for all lanes (the vector operand of a dot
    // product): lane k fetches the record, the scalar and element c of part k and forms
    // their product -- two dependent reads however many parts there are -- and the products
    // are added in order
    auto summed_uniform = [&](int c) {
        float s = 0.0f;
        for (int q0 = 0; q0 < sum_range.y; q0 += NHIP_WAVE) {
            const int m = min(sum_range.y - q0, NHIP_WAVE);
            const int2 mine = epi->lif.parts[sum_range.x + q0 + min(lane, m - 1)];
            const float p = fmaf(X[(size_t)mine.x + c], X[mine.y], 0.0f);
            for (int k = 0; k < m; ++k)
                s = s + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), k));
        }
        return s;
    };
    auto summed = [&](int c) {
        float s = 0.0f;
        if (WAVE_TASK) {
            // element c of the sum with c the lane's own (rows of an item that is a sum):
            // lane k fetches the record and the scalar of part k, the vector elements of
            // four parts are requested together
            for (int q0 = 0; q0 < sum_range.y; q0 += NHIP_WAVE) {
                const int m = min(sum_range.y - q0, NHIP_WAVE);
                const int2 mine = epi->lif.parts[sum_range.x + q0 + min(lane, m - 1)];
                const float my_w = X[mine.y];
                for (int k0 = 0; k0 < m; k0 += 4) {
                    float v[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        v[u] = X[(size_t)__builtin_amdgcn_readlane(mine.x, min(k0 + u, m - 1)) + c];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const float w = __int_as_float(__builtin_amdgcn_readlane(
                            __float_as_int(my_w), min(k0 + u, m - 1)));
                        if (k0 + u < m) s = s + fmaf(v[u], w, 0.0f);
                    }
                }
            }
            return s;
        }
        // (the records of four parts, then their operands, are requested together: the
        // launch is a chain of dependent reads, and this keeps it two links per four parts)
        for (int q0 = 0; q0 < sum_range.y; q0 += 4) {
            int2 part[4];
            float v[4], w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                part[u] = epi->lif.parts[sum_range.x + min(q0 + u, sum_range.y - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                v[u] = X[(size_t)part[u].x + c];
                w[u] = X[part[u].y];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (q0 + u < sum_range.y) s = s + fmaf(v[u], w[u], 0.0f);
        }
        return s;
    };
    // (WAVE_TASK: the whole wave forms the sum, also the lanes past the task's rows, whose reads
    // the others use; the condition is the same for all of them)
    if (NEURONS && sum_range.y > 0 && (WAVE_TASK ? it.n_dots == 0 : n_dots == 0)) sum = summed(r);

    if (LPR >= NHIP_WAVE) {
        // Everything but the columns is the same for all lanes.  The operands of a lane's partial
        // sum (the host has checked: at least 128 columns, stride 1) are 16 bytes apart: 32
        // loads with constant offsets from one address.  The lanes of the last tile start as
        // many steps early as it takes to end inside the row, and leave those steps out.
        constexpr int STEPS = TILE / 4, TILES = NHIP_WAVE / 4;  // per wave and pass
        constexpr int WAVES = LPR / NHIP_WAVE;                  // on one row
        __shared__ float s_tiles[WAVES > 1 ? WAVES * TILES : 1];
        const int my_wave = WAVES > 1 ? __builtin_amdgcn_readfirstlane(tid >> 6) : 0;
        const int n_dots_u = __builtin_amdgcn_readfirstlane(n_dots);
        const int row_u = __builtin_amdgcn_readfirstlane(r);
        const int dot_begin = __builtin_amdgcn_readfirstlane(it.dot_begin);
        for (int d = 0; d < n_dots_u; ++d) {
            const GemvDot dot = dots[dot_begin + d];
            const int n_cols = dot.N;
            const float* arow = A + dot.a_start + (size_t)row_u * dot.a_stride0;
            const float* xg = X + dot.x_start;
            // Rows and vectors of whole aligned quads: a lane loads 16 bytes where it loaded 4, quad 4 i + p
            // of a tile goes to lane p, and the four lanes transpose what they hold.  64 loads of 16 pieces
            // of 16 bytes keep a compute unit's address path busy: with as many rows as fill it,
            // whole steps of rate neurons are faster so (1,026 rows of 1,200 columns 13.0 -> 12.2 us, 1,538
            // of 2,000 16.9 -> 15.4), but not where a unit has a wave or two (770 rows of 1,000 11.6 both
            // ways), nor where a group takes a row (160 rows of 3,000 12.8 -> 13.0).
            const bool quads = LPR == NHIP_WAVE && n_tasks >= QUAD_MIN_TASKS &&
                               ((n_cols | (int)(reinterpret_cast<uintptr_t>(arow) >> 2) |
                                 (int)(reinterpret_cast<uintptr_t>(xg) >> 2)) & 3) == 0;
#pragma unroll 1
            for (int c0 = 0; c0 < n_cols; c0 += WAVES * TILES * TILE) {
                const int start = c0 + (my_wave * TILES + (lane >> 2)) * TILE + (lane & 3);
                const int early = max((start + TILE - n_cols) >> 2, 0);
                const int first = early < STEPS ? start - 4 * early : lane & 3;  // (nothing to sum)
                float s = 0.0f;
                if (quads && c0 + my_wave * TILES * TILE < n_cols) {  // uniform
                    const int tile = c0 + (my_wave * TILES + (lane >> 2)) * TILE;
                    float4 av[STEPS / 4], xv[STEPS / 4];
#pragma unroll
                    for (int i = 0; i < STEPS / 4; ++i) {
                        const int c = min(tile + 16 * i + 4 * (lane & 3), n_cols - 4);
                        av[i] = *reinterpret_cast<const float4*>(arow + c);
                        xv[i] = *reinterpret_cast<const float4*>(xg + c);
                    }
                    const int live = (n_cols - tile) >> 2;  // steps inside the row (none: a tile nobody adds)
#pragma unroll
                    for (int i = 0; i < STEPS / 4; ++i) {
                        transpose_quad(av[i], lane);
                        transpose_quad(xv[i], lane);
                        s = 4 * i + 0 < live ? fmaf(av[i].x, xv[i].x, s) : s;
                        s = 4 * i + 1 < live ? fmaf(av[i].y, xv[i].y, s) : s;
                        s = 4 * i + 2 < live ? fmaf(av[i].z, xv[i].z, s) : s;
                        s = 4 * i + 3 < live ? fmaf(av[i].w, xv[i].w, s) : s;
                    }
                    s = s + __shfl_xor(s, 2, NHIP_WAVE);
                    s = s + __shfl_xor(s, 1, NHIP_WAVE);
                } else if (c0 + my_wave * TILES * TILE < n_cols) {
                    float av[STEPS], xv[STEPS];
#pragma unroll
                    for (int e = 0; e < STEPS; ++e) {
                        av[e] = arow[first + 4 * e];
                        xv[e] = xg[first + 4 * e];
                    }
                    if (__any(early > 0)) {
#pragma unroll
                        for (int e = 0; e < STEPS; ++e) s = e >= early ? fmaf(av[e], xv[e], s) : s;
                    } else {
#pragma unroll
                        for (int e = 0; e < STEPS; ++e) s = fmaf(av[e], xv[e], s);
                    }
                    s = s + __shfl_xor(s, 2, NHIP_WAVE);
                    s = s + __shfl_xor(s, 1, NHIP_WAVE);
                }
                const int n_tiles = min((n_cols - c0 + TILE - 1) / TILE, WAVES * TILES);
                if (WAVES > 1) {
                    if ((lane & 3) == 0) s_tiles[my_wave * TILES + (lane >> 2)] = s;
                    __syncthreads();
                    s = s_tiles[lane];  // tile `lane` of the pass
                    __syncthreads();
                }
#pragma unroll 1
                for (int t = 0; t < n_tiles; ++t)
                    sum = sum + cf.x * __int_as_float(__builtin_amdgcn_readlane(
                        __float_as_int(s), WAVES > 1 ? t : 4 * t));
            }
        }
    } else
    for (int d0 = 0; __any(d0 < n_dots); d0 += BATCH) {
        GemvDot dot[BATCH];
        bool tiny = true;
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            dot[k] = dots[d0 + k < n_dots ? it.dot_begin + d0 + k : 0];
            tiny = tiny && (d0 + k >= n_dots || dot[k].N <= 4);
        }
        if (LPR == 1 || __all(tiny)) {
            float a[BATCH][PER_LANE], x[BATCH][PER_LANE];
#pragma unroll
            for (int k = 0; k < BATCH; ++k)
#pragma unroll
                for (int e = 0; e < PER_LANE; ++e) {
                    const int c = lir + e * LPR;
                    const bool live = d0 + k < n_dots && c < dot[k].N;
                    a[k][e] = live ? A[dot[k].a_start + (size_t)r * dot[k].a_stride0 + c] : 0.0f;
                    x[k][e] = live ? X[dot[k].x_start + (size_t)c * dot[k].x_stride0] : 0.0f;
                    if (WAVE_TASK && NEURONS && k == 0 && d0 == 0 && sum_range.y > 0 &&
                        __any(live)) {
                        // (all lanes of the wave run the sum: its reads are spread over them)
                        const float xs = summed_uniform(c);
                        if (live) {
                            x[k][e] = xs;
                            if (r == 0) Y[(size_t)dot[k].x_start + c] = xs;
                        }
                    } else if (NEURONS && k == 0 && d0 == 0 && live && sum_range.y > 0) {
                        x[k][e] = summed(c);
                        // the item's first row also stores the sum in the operand's place
                        if (r == 0) Y[(size_t)dot[k].x_start + c] = x[k][e];
                    }
                }
#pragma unroll
            for (int k = 0; k < BATCH; ++k) {
                float s;
                if (LPR == 4) {
                    s = lir < dot[k].N ? fmaf(a[k][0], x[k][0], 0.0f) : 0.0f;
                    s = s + __shfl_xor(s, 2, NHIP_WAVE);
                    s = s + __shfl_xor(s, 1, NHIP_WAVE);
                } else {
                    float p[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        p[e] = e < dot[k].N ? fmaf(a[k][e % PER_LANE], x[k][e % PER_LANE], 0.0f) : 0.0f;
                    s = (p[0] + p[2]) + (p[1] + p[3]);
                }
                if (d0 + k < n_dots) sum = sum + cf.x * s;
            }
            continue;
        }
        if (LPR == 4) {
#pragma unroll
            for (int k = 0; k < BATCH; ++k) {  // static indices keep the records in registers
                if (!__any(d0 + k < n_dots)) break;
                const bool have = d0 + k < n_dots;
                const int n_cols = have ? dot[k].N : 0;
                const float* arow = A + dot[k].a_start + (size_t)r * dot[k].a_stride0;
                const float* xg = X + dot[k].x_start;
                const size_t xs = (size_t)dot[k].x_stride0;
                for (int c0 = 0; c0 < n_cols; c0 += TILE) {
                    const int c1 = min(c0 + TILE, n_cols);
                    float s = 0.0f;
                    // partial sum `lir`: columns c0 + lir, + 4, ... below c1, CHUNK of them
                    // fetched at a time (past the end: the last column again, not used)
                    for (int cb = c0 + lir; cb < c1; cb += 4 * CHUNK) {
                        float av[CHUNK], xv[CHUNK];
#pragma unroll
                        for (int e = 0; e < CHUNK; ++e) {
                            const int c = min(cb + 4 * e, c1 - 1);
                            av[e] = arow[c];
                            xv[e] = xg[(size_t)c * xs];
                        }
#pragma unroll
                        for (int e = 0; e < CHUNK; ++e)
                            if (cb + 4 * e < c1) s = fmaf(av[e], xv[e], s);
                    }
                    s = s + __shfl_xor(s, 2, NHIP_WAVE);
                    s = s + __shfl_xor(s, 1, NHIP_WAVE);
                    sum = sum + cf.x * s;
                }
            }
        }
    }
    bool spiked = false;
    if (lir == 0 && valid) {
        const float y = sum + cf.z;
        if (!(epi_lif(EPI) && (pop.pflags & LIF_POP_NO_J)) &&
            !(EPI == EPI_NEURON && (npop.flags & LIF_POP_NO_J)))
            Y[it.y_start + (size_t)r * it.y_stride0] = y;
        if (epi_lif(EPI) && (pop.pflags & LIF_POP_ENABLED))
            spiked = lif_epilogue(epi->lif, pop, r, y, v_old, w_old);
        if (EPI == EPI_NEURON && (npop.flags & LIF_POP_ENABLED))
            neuron_epilogue(epi->lif, npop, r, y, v_old, w_old, n_old);
        if (epi_filters(EPI) && f_range.y > 0) {
            // the first target with what was fetched ahead (the arithmetic of
            // filter_epilogue), further targets of the item from memory
            epi->filter.F[(size_t)f_first.y_start + r] =
                filter_step<EPI == EPI_FILTER2>(epi->filter.targets, f_first, r, y, f_old);
            filter_epilogue<EPI == EPI_FILTER2>(epi->filter, make_int2(f_range.x + 1, f_range.y - 1), r, y);
        }
    }
    if (EPI == EPI_LIF_BITS) {
        // The rows of a wave are consecutive rows of the population from a multiple of their number on
        // (the host's word; a wave at the population's end may hold rows of others behind its own).
        const bool wanted = valid && (pop.pflags & LIF_POP_MASK);
        unsigned long long b = __ballot(wanted && lir == 0 && spiked);
        if (LPR == 4) {  // every fourth lane's bit -> sixteen bits
            b = (b | b >> 3) & 0x0303030303030303ull;
            b = (b | b >> 6) & 0x000f000f000f000full;
            b = (b | b >> 12) & 0x000000ff000000ffull;
            b = (b | b >> 24) & 0xffffull;
        }
        if (lane == 0 && wanted) {
            if (LPR == 4) reinterpret_cast<unsigned short*>(epi->lif.mask)[r >> 4] = (unsigned short)b;
            else reinterpret_cast<unsigned long long*>(epi->lif.mask)[r >> 6] = b;
        }
    }
}
