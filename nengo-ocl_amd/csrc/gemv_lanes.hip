// Input currents of neurons and the update of these neurons, a lane per neuron.
//
//   J[b] = beta_b * Yin[b] + gamma_b + alpha_b * sum_d A[b,d] @ X[b,d];  (V, W, S, N)[b] = neuron(J[b])
//
// for matrices that nothing writes (encoders) and dot products of at most 128 columns, one tile of the
// reference's summation order (clra_gemv.py:1043-1058, :1148-1153).  The kernels of gemv_tile.hip read such a
// matrix as it lies in the signal buffer, rows side by side, and turn it in LDS so that every partial sum
// of a row finds its elements: 300 vector, 190 scalar and 200 LDS instructions per 32 KB, which a wave issues for as
// long as it waits for memory (counters at 192 x 2000 x 32: 12,600 of 29,800 clocks).  Here the host has the
// matrix laid out once (nhip_lay_out_lanes): 64 rows by four columns are 1 KB in a row, lane l holds row l, so
// a 16-byte load brings one element of each of the four partial sums of the lane's row, and a step of
// the sums is four fused multiply-adds with x read from LDS by all lanes at one address.  No turning, no
// exchange between lanes, any column count, any alignment of the original.
//
// Whole steps before (gemv_stream_kernel, gemv_rows_ref_epi_kernel) -> with this kernel: 256 x 4096 x 64 63.9 -> 57.8 us
// (encoders and neurons: 272 MB in 46 us), 64 triples of 2000 x 32 with learning 44.3 -> 42.5, 48 x 2000 x 32 rate neurons
// 14.4 -> 11.0, 37 x 1501 x 50 14.5 -> 10.4, 32 x 1000 x 16 adaptive neurons 12.3 -> 9.4, 256 x 100 in a small world
// 10.7 -> 9.65, 100,000 x 1 with bits for a sparse product 17.7 -> 16.7.  The large ones are bound by what memory gives:
// ordinary loads while the memory-side cache keeps much of the matrices from step to step (whole steps with 268 MB of
// encoders, 256 x 4096 x 64: 57.7 us, non-temporal 61.1), non-temporal ones (PAST) where a step moves more (302 MB,
// 288 x 4096 x 64: 71.8 / 67.8, before this kernel 71.9; 512 x 4096 x 64 126.4 / 111.4, 115.4; 2000 x 1000 x 64 129.7 /
// 116.3, 116.4; 2000 x 4096 x 16 186.5 / 165.2, 196.6; the rule: `hipra_lanes.read_past_the_cache`).  The others
// are bound by the chain record -> parts -> x -> update: 2.3 us behind the launch's 0.9.  Two row
// blocks a wave were as fast for 272 MB (58.5) and slower where the launch is short (48 x 2000 x 32 13.1).
//
// A wave's task is up to 64 rows of one item.  Everything it needs to start is in its record (item,
// coefficients, first dot product, population): one read, then the matrix, the neurons' state and the parts of
// the input sum are under way together.  Up to 64 columns are straight-line code per number of column chunks,
// so that no load is under a branch (the compiler then waits by count).
#include "nhip_common.h"
#include "gemv_types.h"
#include "neuron_math.h"
#include "rows_side.h"

#include <type_traits>

namespace {

struct LaneTask {         // 40 words: GemvFatTask, the item's population, its deferred filter
    GemvTask task;        // pad: first part of the input sum
    GemvItem item;        // pad: number of parts of the input sum (0: X is read as it is)
    float alpha, beta, gamma, pad;
    GemvDot dot0;         // a_start: first KB of the laid-out matrix, a_stride0: column quads
    int pop[12];          // LifPop or NeuronPop
    int4 deferred;        // as LifArgs::deferred
};
typedef int lane_i16 __attribute__((ext_vector_type(16)));
typedef int lane_i8 __attribute__((ext_vector_type(8)));
struct __attribute__((packed, aligned(4))) LaneRecord { lane_i16 a, b; lane_i8 c; };
static_assert(sizeof(LaneTask) == 160 && sizeof(LaneRecord) == 160, "table");

// Matrices and what a wave reads alike for all lanes and nothing in the launch writes: through the constant
// cache, whose loads are counted apart from those of the matrix (no wait for one holds up the other).
template <typename T> using lane_const = const __attribute__((address_space(4))) T;
template <typename T>
__device__ __forceinline__ lane_const<T>* as_const(const T* p) {
    return reinterpret_cast<lane_const<T>*>(reinterpret_cast<uintptr_t>(p));
}

#define LANE_INLINE __attribute__((always_inline))

typedef float lane_f4 __attribute__((ext_vector_type(4)));
constexpr int LANE_COLS = 128;   // columns of a dot product at most
constexpr int LANE_HALF = 64;    // columns of a pass
constexpr int LANE_PARTS = 4;    // what the ranges of parts are padded to

struct LaneArgs {
    const GemvDot* dots;
    const float* TAU;
    const float* REF;
    const float* AMP;
    unsigned* mask;
    float dt, dtu, dt_inv;
    int upsample;
};

constexpr int LANE_WAVES = NHIP_WG / NHIP_WAVE;
constexpr size_t LANE_SEQ_BYTES = SEQ_MAX_OPS * sizeof(NhipSeqOp) + sizeof(int) * SEQ_MAX_ROWS * SEQ_ROW_WORDS;

// LDS written by some lanes of the wave is read by others: order it at wave scope
__device__ __forceinline__ void lane_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Task 4 g + w is wave w's of group g (behind the carried chains); the host has put the list into that order for the
// accelerator dies, and filled the last group up with tasks of no rows.  (With the number of tasks and the grid
// among the arguments, and those read where they are used, a wave made five dependent reads before its record.)
// PAST: matrices are read past the memory-side cache.
template <int EPI, bool SIDE, bool PAST>
__global__ __launch_bounds__(NHIP_WG) __attribute__((amdgpu_waves_per_eu(4)))
void gemv_lanes_kernel(const LaneTask* tasks, const lane_f4* At, float* B, const int2* parts_table, LaneArgs la,
                       RowsSide side)
{
    constexpr size_t X_BYTES = sizeof(float) * LANE_WAVES * LANE_COLS;
    static_assert(LANE_SEQ_BYTES > X_BYTES, "a carried sequence stages its records in the same LDS");
    __shared__ __attribute__((aligned(16))) char lds[SIDE ? LANE_SEQ_BYTES : X_BYTES];
    int group = blockIdx.x;
    if (SIDE) {  // the carried chains first: they take longest
        if (group < side.n_chains) {
            sequence_chain(side.ops + side.chains.first_op[group],
                           side.chains.first_op[group + 1] - side.chains.first_op[group],
                           side.chains.n_staged[group], reinterpret_cast<NhipSeqOp*>(lds),
                           reinterpret_cast<int (*)[SEQ_ROW_WORDS]>(lds + SEQ_MAX_OPS * sizeof(NhipSeqOp)),
                           threadIdx.x);
            return;
        }
        group -= side.n_chains;
    }
    const int lane = threadIdx.x & (NHIP_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* xb = reinterpret_cast<float*>(lds) + wave * LANE_COLS;  // x of the dot product at hand

    // the whole record at once (the compiler would fetch parts of it where they are used)
    lane_const<LaneRecord>* at = as_const(reinterpret_cast<const LaneRecord*>(tasks) + (LANE_WAVES * group + wave));
    LaneRecord record;
    record.a = at->a;
    record.b = at->b;
    record.c = at->c;
    asm volatile("" : "+s"(record.a), "+s"(record.b), "+s"(record.c));
    const LaneTask ft = __builtin_bit_cast(LaneTask, record);
    const GemvItem& it = ft.item;
    const int n_rows = min(ft.task.n_rows, NHIP_WAVE), row0 = ft.task.row0;
    if (n_rows <= 0) return;  // uniform; no group barrier below
    const unsigned lane_off = 16u * (unsigned)lane;
    const int row = row0 + min(lane, n_rows - 1);  // lanes past the task's end hold its last row and store nothing
    const bool mine = lane < n_rows;
    const LifPop pop = *reinterpret_cast<const LifPop*>(ft.pop);
    const NeuronPop npop = *reinterpret_cast<const NeuronPop*>(ft.pop);
    const float *X = B, *Yin = B;
    float* Y = B;
    LifArgs args{};
    args.V = args.W = args.S = args.N = args.Fdef = B;
    args.TAU = la.TAU;
    args.REF = la.REF;
    args.AMP = la.AMP;
    args.mask = la.mask;
    args.dt = la.dt;
    args.dtu = la.dtu;
    args.dt_inv = la.dt_inv;
    args.upsample = la.upsample;

    // what the end of the task needs besides its sums: requested behind the first matrix loads
    float y_old, v_in = 0.0f, w_in = 0.0f, n_in = 0.0f, s_in = 0.0f, f_in = 0.0f;
    const bool defers = EPI == EPI_LIF && (ft.deferred.w & 1) && (pop.pflags & LIF_POP_ENABLED);
    auto fetch_state = [&]() LANE_INLINE {
        if (defers) {
            s_in = args.S[(size_t)pop.s_start + row];
            f_in = args.Fdef[(size_t)ft.deferred.x + row];
        }
        y_old = Yin[it.yin_start + (size_t)row * it.yin_stride0];
        if (EPI == EPI_LIF) {
            const bool on = pop.pflags & LIF_POP_ENABLED;  // else: the buffers' first element
            v_in = args.V[on ? (size_t)pop.v_start + row : 0];
            w_in = args.W[on ? (size_t)pop.w_start + row : 0];
        } else {
            const bool on = npop.flags & LIF_POP_ENABLED;
            v_in = args.V[on && neuron_has_v(npop.kind) ? (size_t)npop.v_start + row : 0];
            w_in = args.W[on && neuron_has_w(npop.kind) ? (size_t)npop.w_start + row : 0];
            n_in = args.N[on && neuron_has_n(npop.kind) ? (size_t)npop.n_start + row : 0];
        }
    };
    // The filter step that closes the previous step, on the spikes this task is about to replace: y = b0 x - a0 y,
    // or y = b0 x (clra_nonlinearities.py:630-650).  Nothing else in the launch reads it.
    auto close_filter = [&]() LANE_INLINE {
        if (!defers || !mine) return;
        const float bx = __fmul_rn(nhip_bits(ft.deferred.z), s_in);
        args.Fdef[(size_t)ft.deferred.x + row] =
            (ft.deferred.w & 2) ? __fsub_rn(bx, __fmul_rn(nhip_bits(ft.deferred.y), f_in)) : bx;
    };
    // (...(0 + v_0[c] s_0) + v_1[c] s_1) + ... over the item's parts: every product rounded on its own and added
    // in order, what Y = 0 * Y + sum_k v_k s_k gives as a launch of its own.  (The table holds every
    // range padded to a multiple of LANE_PARTS with its last part.)
    auto input_sum = [&](int c) LANE_INLINE {
        float s = 0.0f;
        lane_const<int2>* parts = as_const(parts_table) + ft.task.pad;
        lane_const<float>* xc = as_const(X);
        auto some = [&](auto count, int q0) LANE_INLINE {  // so many parts, requested together
            constexpr int U = decltype(count)::value;
            float v[U], w[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int at = parts[q0 + u].x, scale = parts[q0 + u].y;
                w[u] = xc[scale];
                v[u] = (X + at)[(unsigned)c];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (q0 + u < it.pad) s = s + fmaf(v[u], w[u], 0.0f);
        };
        int q0 = 0;
        for (; q0 + LANE_PARTS < it.pad; q0 += 2 * LANE_PARTS) some(std::integral_constant<int, 2 * LANE_PARTS>{}, q0);
        if (q0 < it.pad) some(std::integral_constant<int, LANE_PARTS>{}, q0);
        return s;
    };

    float sum;
    // The sums of one dot product.  `before` runs behind the first loads of the matrix and leaves x in LDS.  A pass
    // of up to 64 columns is straight-line code per even number of column quads with all of them in
    // registers: no load of it is under a condition, and only the last two quads may be narrower or missing.
    constexpr int QUADS = LANE_HALF / 4;
    auto dot_product = [&](const GemvDot& dot, auto&& before) LANE_INLINE {
        lane_f4 s = {};  // the four partial sums
        const char* a0 = reinterpret_cast<const char*>(At) +
                         (((size_t)dot.a_start + (size_t)(row0 >> 6) * dot.a_stride0) << 10);
        // `last`: columns of the last quad
        auto pass = [&](auto n_quads, int q0, int quads, int last, auto&& first) LANE_INLINE {
            constexpr int NQ = decltype(n_quads)::value;
            const lane_f4* xq = reinterpret_cast<const lane_f4*>(xb) + q0;
            lane_f4 a[NQ];
#pragma unroll
            for (int i = 0; i < NQ; ++i) {  // (uniform base, the lane's own 32-bit offset)
                const int q = i < NQ - 1 ? i : min(i, quads - 1);
                const lane_f4* at_quad = reinterpret_cast<const lane_f4*>(a0 + ((size_t)(q0 + q) << 10) + lane_off);
                a[i] = PAST ? __builtin_nontemporal_load(at_quad) : *at_quad;
            }
            first();
            auto step = [&](int i, auto n_cols) LANE_INLINE {
                const lane_f4 x = xq[i];
                s.x = fmaf(a[i].x, x.x, s.x);
                if constexpr (n_cols() > 1) s.y = fmaf(a[i].y, x.y, s.y);
                if constexpr (n_cols() > 2) s.z = fmaf(a[i].z, x.z, s.z);
                if constexpr (n_cols() > 3) s.w = fmaf(a[i].w, x.w, s.w);
            };
            constexpr std::integral_constant<int, 4> whole{};
            auto last_step = [&](int i) LANE_INLINE {
                if (last == 4) step(i, whole);
                else if (last == 3) step(i, std::integral_constant<int, 3>{});
                else if (last == 2) step(i, std::integral_constant<int, 2>{});
                else step(i, std::integral_constant<int, 1>{});
            };
#pragma unroll
            for (int i = 0; i < NQ - 2; ++i) step(i, whole);
            if (quads == NQ) {
                step(NQ - 2, whole);
                last_step(NQ - 1);
            } else {
                last_step(NQ - 2);
            }
        };
        auto half = [&](int q0, int quads, int last, auto&& first) LANE_INLINE {
#define LANE_PASS(n) pass(std::integral_constant<int, n>{}, q0, quads, last, first)
            if (quads <= 8) {
                if (quads <= 4) {
                    if (quads <= 2) LANE_PASS(2);
                    else LANE_PASS(4);
                } else if (quads <= 6) LANE_PASS(6);
                else LANE_PASS(8);
            } else if (quads <= 12) {
                if (quads <= 10) LANE_PASS(10);
                else LANE_PASS(12);
            } else if (quads <= 14) LANE_PASS(14);
            else LANE_PASS(16);
#undef LANE_PASS
        };
        const int quads = (dot.N + 3) >> 2;
        const int last = ((dot.N - 1) & 3) + 1;
        if (quads <= QUADS) {
            half(0, quads, last, before);
        } else {
            pass(std::integral_constant<int, QUADS>{}, 0, QUADS, 4, before);
            half(QUADS, quads - QUADS, last, []() LANE_INLINE {});
        }
        sum = sum + ft.alpha * ((s.x + s.z) + (s.y + s.w));
    };
    auto gather = [&](const GemvDot& dot) LANE_INLINE {  // x as it lies in memory
        const float x0 = X[dot.x_start + (size_t)min(lane, dot.N - 1) * dot.x_stride0];
        const float x1 = X[dot.x_start + (size_t)min(lane + LANE_HALF, dot.N - 1) * dot.x_stride0];
        lane_sync();
        xb[lane] = x0;
        xb[lane + LANE_HALF] = x1;
        lane_sync();
    };

    // a matrix as it lies in memory (at most four columns; it need not be constant): element e of the lane's row
    auto raw_row = [&](const GemvDot& dot) LANE_INLINE {
        const float* a = B + dot.a_start + (size_t)row * dot.a_stride0;
        lane_f4 v = {};
        v.x = a[0];
        if (dot.N > 1) v.y = a[1];
        if (dot.N > 2) v.z = a[2];
        if (dot.N > 3) v.w = a[3];
        return v;
    };
    auto raw_sum = [&](const lane_f4& a, const lane_f4& x, int n) LANE_INLINE {
        lane_f4 s = {};
        s.x = fmaf(a.x, x.x, 0.0f);
        if (n > 1) s.y = fmaf(a.y, x.y, 0.0f);
        if (n > 2) s.z = fmaf(a.z, x.z, 0.0f);
        if (n > 3) s.w = fmaf(a.w, x.w, 0.0f);
        sum = sum + ft.alpha * ((s.x + s.z) + (s.y + s.w));
    };

    if (it.n_dots == 0) {
        fetch_state();
        close_filter();
        sum = it.pad > 0 ? input_sum(row) : ft.beta * y_old;
    } else {
        auto before = [&]() LANE_INLINE {
            fetch_state();
            if (it.pad > 0) {
                const float x = input_sum(min(lane, ft.dot0.N - 1));
                xb[lane] = x;
                // the task with the item's first rows stores the sum in the operand's place
                if (row0 == 0 && lane < ft.dot0.N) Y[(size_t)ft.dot0.x_start + lane] = x;
                if (ft.dot0.N > LANE_HALF) {
                    const int c = lane + LANE_HALF;
                    const float more = input_sum(min(c, ft.dot0.N - 1));
                    xb[c] = more;
                    if (row0 == 0 && c < ft.dot0.N) Y[(size_t)ft.dot0.x_start + c] = more;
                }
                lane_sync();
            } else {
                gather(ft.dot0);
            }
            close_filter();
            sum = ft.beta * y_old;
        };
        if (ft.dot0.p0 < 0) {
            const lane_f4 a = raw_row(ft.dot0);
            before();
            raw_sum(a, *reinterpret_cast<const lane_f4*>(xb), ft.dot0.N);
        } else {
            dot_product(ft.dot0, before);
        }
        // Further dot products: four at a time where their matrices are read as they lie in memory, else one
        // after the other (rare: a loop, which keeps the registers of the rest)
        for (int d = 1; d < it.n_dots; ++d) {
            const GemvDot dot = la.dots[it.dot_begin + d];
            if (dot.p0 < 0) {
                constexpr int U = 4;
                GemvDot some[U];
                lane_f4 a[U], x[U];
                lane_const<float>* xc = as_const(X);
                const int n = min(it.n_dots - d, U);
#pragma unroll
                for (int u = 0; u < U; ++u) some[u] = la.dots[it.dot_begin + d + min(u, n - 1)];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    a[u] = raw_row(some[u]);
                    x[u] = lane_f4{};
                    x[u].x = xc[some[u].x_start];
                    if (some[u].N > 1) x[u].y = xc[some[u].x_start + some[u].x_stride0];
                    if (some[u].N > 2) x[u].z = xc[some[u].x_start + 2 * some[u].x_stride0];
                    if (some[u].N > 3) x[u].w = xc[some[u].x_start + 3 * some[u].x_stride0];
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (u < n) raw_sum(a[u], x[u], some[u].N);
                d += n - 1;  // (matrices of one item are all of one kind)
                continue;
            }
            gather(dot);
            const char* a = reinterpret_cast<const char*>(At) +
                            (((size_t)dot.a_start + (size_t)(row0 >> 6) * dot.a_stride0) << 10);
            lane_f4 s = {};
#pragma unroll 1
            for (int c = 0; c < dot.N; c += 4, a += 1024) {
                const lane_f4 v = *reinterpret_cast<const lane_f4*>(a + lane_off);
                const lane_f4 x = *reinterpret_cast<const lane_f4*>(xb + c);
                s.x = fmaf(v.x, x.x, s.x);
                if (c + 1 < dot.N) s.y = fmaf(v.y, x.y, s.y);
                if (c + 2 < dot.N) s.z = fmaf(v.z, x.z, s.z);
                if (c + 3 < dot.N) s.w = fmaf(v.w, x.w, s.w);
            }
            sum = sum + ft.alpha * ((s.x + s.z) + (s.y + s.w));
        }
    }

    // an item without dot products that would copy Y onto itself is only there for its neurons
    const bool store_y = !(it.n_dots == 0 && it.pad == 0 && ft.beta == 1.0f && ft.gamma == 0.0f &&
                           it.y_start == it.yin_start && it.y_stride0 == it.yin_stride0) &&
                         !(EPI == EPI_LIF && (pop.pflags & LIF_POP_NO_J)) &&
                         !(EPI == EPI_NEURON && (npop.flags & LIF_POP_NO_J));
    const float j = sum + ft.gamma;
    if (mine && store_y) Y[it.y_start + (size_t)row * it.y_stride0] = j;
    if (EPI == EPI_LIF && (pop.pflags & LIF_POP_ENABLED)) {
        const float tau = lif_param(pop.tau, pop.pflags & 1, args.TAU, row);
        const float ref = lif_param(pop.ref, pop.pflags & 2, args.REF, row);
        const float amp = lif_param(pop.amp, pop.pflags & 4, args.AMP, row);
        float v = v_in, w = w_in;
        const bool spiked = (pop.pflags & LIF_POP_DECAY)
            ? lif_step_decay(j, v, w, nhip_bits(pop.decay), tau, ref, args.dtu)
            : lif_step(j, v, w, tau, ref, args.dtu, args.upsample);
        if (mine) {
            args.V[(size_t)pop.v_start + row] = v;
            args.W[(size_t)pop.w_start + row] = w;
        }
        const unsigned long long bits = __ballot(mine && spiked);
        if (pop.pflags & LIF_POP_BITS) {  // two 32-bit words (s_start is even)
            if (lane < 2 && 32 * lane < n_rows)
                reinterpret_cast<unsigned*>(args.S + (size_t)pop.s_start)[(row0 >> 5) + lane] =
                    (unsigned)(lane ? bits >> 32 : bits);
        } else if (mine) {
            args.S[(size_t)pop.s_start + row] = spiked ? __fmul_rn(amp, args.dt_inv) : 0.0f;
        }
        if ((pop.pflags & LIF_POP_MASK) && lane == 0)
            reinterpret_cast<unsigned long long*>(args.mask)[row0 >> 6] = bits;
    }
    if (EPI == EPI_NEURON && mine && (npop.flags & LIF_POP_ENABLED))
        neuron_epilogue(args, npop, row, j, v_in, w_in, n_in);
}

// Matrix a_start, a_stride0, M x N of A -> KB out .. of At: block (64 rows, 4 columns) after block
struct LaneMatrix { int a_start, a_stride0, M, N, out, quads, pad0, pad1; };

__global__ __launch_bounds__(NHIP_WG) void lay_out_lanes_kernel(const LaneMatrix* __restrict__ mats, const float* A,
                                                                lane_f4* At) {
    const LaneMatrix m = mats[blockIdx.y];
    const int blocks = (m.M + NHIP_WAVE - 1) / NHIP_WAVE, lane = threadIdx.x & (NHIP_WAVE - 1);
    for (int b = blockIdx.x; b < blocks; b += gridDim.x) {
        const int r = b * NHIP_WAVE + lane;
        for (int q = threadIdx.x >> 6; q < m.quads; q += NHIP_WG / NHIP_WAVE) {
            lane_f4 v = {0.0f, 0.0f, 0.0f, 0.0f};
            if (r < m.M) {
                const float* a = A + m.a_start + (size_t)r * m.a_stride0 + 4 * q;
                for (int e = 0; e < 4 && 4 * q + e < m.N; ++e) v[e] = a[e];
            }
            At[((size_t)m.out + (size_t)b * m.quads + q) * NHIP_WAVE + lane] = v;
        }
    }
}

}  // namespace

extern "C" int nhip_lay_out_lanes(void* stream, const int* matrices, int n, int max_blocks, const float* A, float* At) {
    if (n == 0) return 0;
    if (n < 0 || n > 65535 || max_blocks < 1 || !matrices || !A || !At || (reinterpret_cast<uintptr_t>(At) & 15))
        return NHIP_E_BADARG;
    NHIP_LAUNCH(lay_out_lanes_kernel, dim3(max_blocks < 1024 ? max_blocks : 1024, n), dim3(NHIP_WG), 0,
                static_cast<hipStream_t>(stream), reinterpret_cast<const LaneMatrix*>(matrices), A,
                reinterpret_cast<lane_f4*>(At));
    NHIP_LAUNCH_CHECK();
    return 0;
}

extern "C" int nhip_gemv_lanes(void* stream, int neurons, const int* tasks, int n_tasks, const int* dots,
                               const float* At, float* B, double dt, int upsample, const float* TAU, const float* REF,
                               const float* AMP, const int* parts, int* mask) {
    RowsSide side;
    if (take_carried(side) && n_tasks <= 0) return NHIP_E_BADARG;  // an empty launch cannot carry it
    if (n_tasks == 0) return 0;
    const int waves = NHIP_WG / NHIP_WAVE;
    if (n_tasks < 0 || n_tasks % waves || !tasks || !dots || !At || !B || upsample < 1 || !(dt > 0.0))
        return NHIP_E_BADARG;
    const bool past = neurons & NHIP_LANES_PAST_CACHE;
    neurons &= ~NHIP_LANES_PAST_CACHE;
    if (neurons != EPI_LIF && neurons != EPI_NEURON) return NHIP_E_BADCLASS;
    if (reinterpret_cast<uintptr_t>(At) & 15) return NHIP_E_BADARG;
    LaneArgs args{};
    args.dots = reinterpret_cast<const GemvDot*>(dots);
    args.dt = (float)dt;
    args.dtu = (float)(dt / (double)upsample);  // formed in double and rounded once, as in nhip_lif
    args.dt_inv = (float)(1.0 / dt);
    args.upsample = upsample;
    args.TAU = TAU;
    args.REF = REF;
    args.AMP = AMP;
    args.mask = reinterpret_cast<unsigned*>(mask);
    side.n_gemv_groups = n_tasks / waves;
    auto launch = [&](auto kernel) {
        NHIP_LAUNCH(kernel, dim3(side.n_gemv_groups + side.n_chains), dim3(NHIP_WG), 0,
                    static_cast<hipStream_t>(stream), reinterpret_cast<const LaneTask*>(tasks),
                    reinterpret_cast<const lane_f4*>(At), B, reinterpret_cast<const int2*>(parts), args, side);
    };
    auto of_type = [&](auto epi) {
        constexpr int E = decltype(epi)::value;
        if (side.n_chains > 0) past ? launch(gemv_lanes_kernel<E, true, true>) : launch(gemv_lanes_kernel<E, true, false>);
        else past ? launch(gemv_lanes_kernel<E, false, true>) : launch(gemv_lanes_kernel<E, false, false>);
    };
    if (neurons == EPI_LIF) of_type(std::integral_constant<int, EPI_LIF>{});
    else of_type(std::integral_constant<int, EPI_NEURON>{});
    NHIP_LAUNCH_CHECK();
    return 0;
}
