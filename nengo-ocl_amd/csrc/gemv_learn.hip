// Products with matrices that a learning rule (Oja's, the BCM rule, an outer product: PES) changes in the same step.
//
// As launches of their own, a step of such a matrix reads it for the product, reads and writes it for the
// rule, and a third launch steps the filters of the activities the rule reads (2000 x 2000: 8.0 + 10.4 + 4.7
// us).  All three need nothing but what is there before the first of them: the product takes the old
// matrix, the rule the old matrix and the old activities, and the filters only have to wait until
// nobody reads the old activities any more.  Here a wave owns a row: it requests the row once, writes it
// back with its change, and sums the old values in the reference's order; the group that is the last to
// have read its activities steps the filters.
//
// 2000 x 2000: 13.9 -> 9.1 us (counters of arrivals: 9.8; nothing requested behind a wait or a condition: 9.1; in a
// kernel trace of whole calls 9.5), whole steps 24.8 -> 19.0.  What is left, from the first group's start: record 0.5,
// vectors at 2.3, rows at 3.1 (5 TB/s from there to the last), rule and stores 1.1, sums 1.1 (both as long as LDS
// takes for 40 KB a wave's row), last group's filters 1.6.  A plain kernel that reads and writes 16.8 MB takes 4.4 us of a launch.
//
// A row in LDS lies in tiles of 128 columns, 132 words apart: the sum of a tile is four strided
// partial sums (clra_gemv.py:1043-1058, :1148-1153), a lane each, sixteen tiles side by side, and
// with that distance the 64 lanes of a step read 64 banks.  What lies past the row's end is -0 in the
// matrix and +0 in the vector, whose product changes no sum.
#include <type_traits>

#include "nhip_common.h"
#include "gemv_types.h"
#include "learn_math.h"
#include "neuron_math.h"
#include "rows_side.h"

namespace {

// Up to four rows (a wave each) of one item.
struct LearnTask {
    int a_start, a_stride0, N, x_start;  // row r of the matrix at a_start + r * a_stride0
    int y_start, y_stride0, yin_start, yin_stride0;
    float alpha, beta, gamma;
    int row0;
    int n_rows, learned;                 // learned 0: the matrix stays as it is
    int first_target, n_targets;         // filters of the item
    struct {                             // (in the record: a table of its own is another trip to memory)
        int kind, pre_start, post_start, post_stride0;
        int theta_start, theta_stride0;  // BCM: one value per row
        float alpha, beta;
    } rule;
    FilterTarget target;                 // the item's first filter
    int own_groups, own_filter;          // not zero: so many groups read the activities that this filter replaces
    int pad[2];
};
// A filter stepped when no group reads its output any more: F[f + i] = b S[s + i] - a F[f + i] (or b S[s + i])
struct LearnFilter {
    int s_start, f_start, n, has_a;
    float a, b;
    int pad0, pad1;
};
static_assert(sizeof(LearnTask) == 128 && sizeof(LearnFilter) == 32, "tables");

constexpr int LEARN_OUTER = 16;                // kind of rule besides NHIP_RULE_*: W += (alpha post) (x) pre
constexpr int LROWS = NHIP_WG / NHIP_WAVE;     // rows of a group
constexpr int LTILE = 128, LTILES = 16;        // columns of a tile, tiles of a pass
constexpr int LSTRIDE = LTILE + 4;             // words between tiles in LDS
constexpr int LCOLS = LTILE * LTILES;          // columns of a pass
constexpr int LCOUNTERS = 32, LCOUNTER_WORDS = 32;  // counters of arrivals (and one for them), words between them
typedef float learn_f4 __attribute__((ext_vector_type(4)));
typedef float learn_q4 __attribute__((ext_vector_type(4), aligned(4)));  // at any element of a row
typedef int learn_i16 __attribute__((ext_vector_type(16)));
typedef int learn_i8 __attribute__((ext_vector_type(8)));
#define LEARN_INLINE __attribute__((always_inline))

// LDS written by some lanes of a wave is read by others
__device__ __forceinline__ void learn_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int learn_lds(int c) { return (c >> 7) * LSTRIDE + (c & (LTILE - 1)); }

struct LearnLds {
    __attribute__((aligned(16))) float w[LROWS][LTILES * LSTRIDE];
    __attribute__((aligned(16))) float x[LTILES * LSTRIDE];
    __attribute__((aligned(16))) float pre[LCOLS];
    int last;
};

// The rows of a group, four columns at a time from whatever address on (rows of an odd length in
// single elements took four times the loads; 1401 x 1401, whole steps, 20.8 -> 16.4 us with what the kernel below
// says of arrivals); what is left of the last four, an element per lane.
// `read()`: called by all waves when every wave of the group has its activities.
// Nothing is requested under a condition of a lane: what lies past the row's end is read from its last quad (or
// element) and replaced.  (Behind conditions the compiler does not know how many loads are out, and waited for all
// of them, the rows too, before the vectors went to LDS.)
template <int RULE, typename Read>
__device__ __forceinline__ void learn_rows(const LearnTask& task, const float* spare, float* A, const float* X,
                                           LearnLds& lds, int wave, int lane, int tid, const float* y_at,
                                           const float* f_at, float& f_old, float& sum, Read&& read) {
    constexpr bool LEARNED = RULE != 0;
    const auto& rule = task.rule;
    constexpr int PER_LANE = LCOLS / NHIP_WAVE / 4;   // quads of a lane of its row, per pass
    constexpr int PER_THREAD = LCOLS / NHIP_WG / 4;   // quads of a thread of a vector, per pass
    const bool mine = wave < task.n_rows;  // the same for the wave; the others read the last row and keep nothing
    const int row = task.row0 + min(wave, task.n_rows - 1);
    float* arow = A + task.a_start + (size_t)row * task.a_stride0;
    const float* xg = X + task.x_start;
    const float* pre = X + (LEARNED ? rule.pre_start : task.x_start);
    int c0 = 0;
    do {
        const int n = min(task.N - c0, LCOLS);
        const int n4 = n & ~3;      // whole quads; then n & 3 elements
        const int tail = n4 + lane; // (of the first lanes)
        const int last4 = max(n4 - 4, 0), last = min(tail, n - 1);
        // (fewer than four columns: the quads come from memory that holds four)
        const float* x4 = n4 > 0 ? xg + c0 : spare;
        const float* p4 = n4 > 0 ? pre + c0 : spare;
        const float* w4 = n4 > 0 ? arow + c0 : spare;
        // the vectors first (the barrier waits for them), then the row: all of it under way together
        learn_f4 xv[PER_THREAD], pv[PER_THREAD], w[PER_LANE];
#pragma unroll
        for (int k = 0; k < PER_THREAD; ++k) {
            const int c = min(4 * (tid + k * NHIP_WG), last4);
            xv[k] = *reinterpret_cast<const learn_q4*>(x4 + c);
            if (LEARNED) pv[k] = *reinterpret_cast<const learn_q4*>(p4 + c);
        }
        const float xt = xg[c0 + last], pt = LEARNED ? pre[c0 + last] : 0.0f;
        // ... with what the row needs at its end (in every pass: what is on its way into a loop is waited for there)
        const float y_old = *y_at;
        f_old = *f_at;
        float post = 0.0f, theta = 0.0f;
        if (LEARNED) {
            post = X[rule.post_start + (size_t)row * rule.post_stride0];
            if (RULE == NHIP_RULE_BCM) theta = X[rule.theta_start + (size_t)row * rule.theta_stride0];
        }
#pragma unroll
        for (int k = 0; k < PER_LANE; ++k)
            w[k] = *reinterpret_cast<const learn_q4*>(w4 + min(4 * (lane + k * NHIP_WAVE), last4));
        const float wt = arow[c0 + last];
        if (c0 > 0) __syncthreads();  // the pass before has read its vectors
#pragma unroll
        for (int k = 0; k < PER_THREAD; ++k) {
            const int c = 4 * (tid + k * NHIP_WG);
            if (c < n4 || c >= n) {
                *reinterpret_cast<learn_f4*>(lds.x + learn_lds(c)) = c < n4 ? xv[k] : learn_f4{};
                if (LEARNED) *reinterpret_cast<learn_f4*>(lds.pre + c) = pv[k];
            }
        }
        if ((n & 3) && tid < 4) lds.x[learn_lds(tail)] = tail < n ? xt : 0.0f;
        if (c0 + LCOLS >= task.N) asm volatile("" :: "v"(post), "v"(theta), "v"(f_old), "v"(y_old), "v"(pt));  // here by now
        __syncthreads();
        if (c0 == 0) {  // (not formed sooner: it would be waited for before the rest is requested)
            float y = y_old;
            asm volatile("" : "+v"(y));
            sum = task.beta * y;
        }
        if (c0 + LCOLS >= task.N) read();
        if (mine) {
            const float scale = __fmul_rn(rule.alpha, post);  // (the outer product's)
            auto changed = [&](float p, float e) LEARN_INLINE {
                if constexpr (RULE == LEARN_OUTER) return __fadd_rn(e, __fmul_rn(scale, p));
                if constexpr (RULE == NHIP_RULE_BCM || RULE == NHIP_RULE_OJA)
                    return __fadd_rn(e, learn_element<RULE>(rule.alpha, rule.beta, 0.0f, 0.0f, p, post,
                                                            RULE == NHIP_RULE_BCM ? theta : e));
                return e;
            };
#pragma unroll
            for (int k = 0; k < PER_LANE; ++k) {
                const int c = 4 * (lane + k * NHIP_WAVE);
                if (c < n4 || c >= n)
                    *reinterpret_cast<learn_f4*>(lds.w[wave] + learn_lds(c)) =
                        c < n4 ? w[k] : learn_f4{-0.0f, -0.0f, -0.0f, -0.0f};
                if (LEARNED && c < n4) {
                    const learn_f4 p = *reinterpret_cast<const learn_f4*>(lds.pre + c);
                    learn_f4 v;
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[u] = changed(p[u], w[k][u]);
                    *reinterpret_cast<learn_q4*>(arow + c0 + c) = v;
                }
            }
            if (n & 3) {
                if (lane < 4) lds.w[wave][learn_lds(tail)] = tail < n ? wt : -0.0f;
                if (LEARNED && tail < n) arow[c0 + tail] = changed(pt, wt);
            }
            learn_wave_sync();
            const int at = (lane >> 2) * LSTRIDE + (lane & 3);  // partial sum lane & 3 of tile lane >> 2
            float s = 0.0f;
#pragma unroll
            for (int e = 0; e < LTILE / 4; ++e) s = fmaf(lds.w[wave][at + 4 * e], lds.x[at + 4 * e], s);
            s = s + __shfl_xor(s, 2, NHIP_WAVE);
            s = s + __shfl_xor(s, 1, NHIP_WAVE);
            const int n_tiles = (n + LTILE - 1) / LTILE;
#pragma unroll 1
            for (int t = 0; t < n_tiles; ++t)
                sum = sum + task.alpha * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 4 * t));
        }
        c0 += LCOLS;
    } while (c0 < task.N);
}

// Up to 64 rows of an item whose matrix nothing writes and whose vector is mostly zero (spikes): only the columns whose
// x is not zero are read, from a copy of the columns.  (A column left out would add zeros to its partial sum.)
struct ColumnsItem {
    int at_start, mp;              // column c: AT[at_start + c * mp ..], mp a multiple of 16
    int M, N, x_start;
    int y_start, y_stride0, yin_start, yin_stride0;  // of the item's first row
    float alpha, beta, gamma;
    int first_target, n_targets;
    int row0;                      // first row of this record (at_start is that of row 0)
    int all;                       // not zero: the columns whose x is zero count too (the matrix holds an infinity or a NaN)
    FilterTarget target;
    int pad[12];
};
static_assert(sizeof(ColumnsItem) == 128, "table");
struct LearnEvents {
    const ColumnsItem* items;
    const float* AT;
    int n_items;
};

constexpr int CTILES = 32, CCOLS = CTILES * LTILE;  // tiles and columns of a pass
constexpr int CBATCH = 20, CPART = 4;               // columns of a tile requested together; added together
struct ColumnsLds {
    uint2 list[CTILES][LTILE];     // active columns of a tile in order: byte offset | column % 4, x
    float tile[CTILES][NHIP_WAVE];
    int count[CTILES];
};

// A group per record.  A wave lists the active columns of its tiles; then 16, 32 or 64 lanes (as many as there are
// rows) take a tile, and request 20 columns each of two tiles together: 128 neurons of which 8 % spike have
// ten.  192 such items of 32 x 2000 beside 2,048 learned rows of 2,000: the launch 11.0 us, 16.6 with the walk of
// csrc/gemv_events.hip (a column a wave at a time) in groups of this size, 12.8 with these groups behind those
// of rows, whose requests theirs then wait behind; 22.0 with every column read (gemv_stream_kernel).  From the first
// group's start: lists at 2.2 us, columns requested at 4.3 (behind the rows' on their way), there at 4.6, added at 6.4,
// done at 7.3; the rows beside them at 6.0.
__device__ __forceinline__ void columns_group(const ColumnsItem& it, const float* __restrict__ AT, const float* X,
                                              const float* Yin, float* Y, const FilterArgs& filter, ColumnsLds& lds,
                                              int wave, int lane) {
    const int lg = it.M <= 16 ? 4 : it.M <= 32 ? 5 : 6, workers = NHIP_WAVE >> lg;  // lanes of a tile; tiles at once
    const int me = lane >> lg, at_row = lane & ((1 << lg) - 1);
    const char* at = reinterpret_cast<const char*>(AT + it.at_start + it.row0 + min(at_row, it.M - 1));
    const unsigned col_bytes = 4u * (unsigned)it.mp;
    const int row = it.row0 + min(lane, it.M - 1);
    const float* y_at = Yin + it.yin_start + (size_t)row * it.yin_stride0;
    const float* f_at = filter.F + (it.n_targets > 0 ? (size_t)it.target.y_start + row : 0);
    float y_old = 0.0f, f_old = 0.0f, sum = 0.0f;
    int base = 0;
    do {
        const int n_cols = min(it.N - base, CCOLS), n_tiles = (n_cols + LTILE - 1) / LTILE;
        const int per_wave = (n_tiles + LROWS - 1) / LROWS;
        const int t_lo = min(wave * per_wave, n_tiles), t_hi = min(t_lo + per_wave, n_tiles);
        for (int t0 = t_lo; t0 < t_hi; t0 += 4) {  // (up to 2,048 columns: once)
            float xv[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                xv[u] = X[it.x_start + base + min(t0 * LTILE + u * NHIP_WAVE + lane, n_cols - 1)];
            y_old = *y_at;  // (the first wave's, which has tiles)
            f_old = *f_at;
            int found = 0;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int t = t0 + (u >> 1), c = t0 * LTILE + u * NHIP_WAVE + lane;
                if (t >= t_hi) break;  // uniform
                const bool active = c < n_cols && (it.all || (__float_as_uint(xv[u]) & 0x7fffffffu) != 0u);
                const unsigned long long b = __ballot(active);
                if ((u & 1) == 0) found = 0;
                const int before = found + __builtin_amdgcn_mbcnt_hi((unsigned)(b >> 32),
                                                                     __builtin_amdgcn_mbcnt_lo((unsigned)b, 0));
                if (active)
                    lds.list[t][before] = make_uint2((unsigned)(base + c) * col_bytes | (unsigned)(c & 3),
                                                     __float_as_uint(xv[u]));
                found += __popcll(b);
                if ((u & 1) && lane == 0) lds.count[t] = found;
            }
        }
        learn_wave_sync();
        for (int t0 = t_lo; t0 < t_hi; t0 += 2 * workers) {
            const int ta = t0 + me, tb = ta + workers;
            const int na = ta < t_hi ? lds.count[ta] : 0, nb = tb < t_hi ? lds.count[tb] : 0;
            const uint2* la = lds.list[min(ta, CTILES - 1)];
            const uint2* lb = lds.list[min(tb, CTILES - 1)];
            float a[CBATCH], b[CBATCH];
            // (entries that are not there: the first column, and no sum takes it)
            auto request = [&](const uint2* list, int n, int k, float (&v)[CBATCH]) LEARN_INLINE {
#pragma unroll
                for (int u = 0; u < CBATCH; ++u) {
                    const unsigned off = list[min(k + u, LTILE - 1)].x & ~3u;  // (read whether it is there or not)
                    v[u] = *reinterpret_cast<const float*>(at + (k + u < n ? off : 0u));
                }
            };
            float s[4];
            auto add = [&](const uint2* list, int n, int k, const float (&v)[CBATCH]) LEARN_INLINE {
#pragma unroll
                for (int p = 0; p < CBATCH; p += CPART)
                    if (__any(k + p < n))
#pragma unroll
                        for (int u = p; u < p + CPART; ++u) {
                            const uint2 e = list[min(k + u, LTILE - 1)];
                            const int j = k + u < n ? (int)(e.x & 3u) : 4;
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const float next = fmaf(v[u], __uint_as_float(e.y), s[q]);
                                s[q] = j == q ? next : s[q];
                            }
                        }
            };
            auto finish = [&](int t, const uint2* list, int n, float (&v)[CBATCH]) LEARN_INLINE {
                s[0] = s[1] = s[2] = s[3] = 0.0f;
                add(list, n, 0, v);
                for (int k = CBATCH; __any(k < n); k += CBATCH) {
                    request(list, n, k, v);
                    add(list, n, k, v);
                }
                if (t < t_hi) lds.tile[t][at_row] = it.alpha * ((s[0] + s[2]) + (s[1] + s[3]));
            };
            request(la, na, 0, a);
            request(lb, nb, 0, b);
            finish(ta, la, na, a);
            finish(tb, lb, nb, b);
        }
        __syncthreads();
        if (wave == 0) {
            if (base == 0) sum = it.beta * y_old;
#pragma unroll
            for (int h = 0; h < CTILES; h += 16) {
                float v[16];
#pragma unroll
                for (int t = 0; t < 16; ++t) v[t] = lds.tile[h + t][lane];  // (16 reads at once)
#pragma unroll
                for (int t = 0; t < 16; ++t)
                    if (h + t < n_tiles) sum = sum + v[t];
            }
        }
        base += CCOLS;
        if (base < it.N) __syncthreads();  // read, before the next pass
    } while (base < it.N);
    if (wave == 0 && lane < it.M) {
        const float y = sum + it.gamma;
        Y[it.y_start + (size_t)row * it.y_stride0] = y;
        if (it.n_targets > 0) {
            filter.F[(size_t)it.target.y_start + row] = filter_step<true>(filter.targets, it.target, row, y, f_old);
            filter_epilogue<true>(filter, make_int2(it.first_target + 1, it.n_targets - 1), row, y);
        }
    }
}

// EVENTS: there are such items (their groups before those of rows: they take longer)
template <bool EVENTS>
__global__ __launch_bounds__(NHIP_WG) void gemv_learn_kernel(
    const LearnTask* tasks, float* A, const float* X, const float* Yin, float* Y,
    FilterArgs filter, const LearnFilter* filters, int n_filters, int* arrived, LearnEvents events, RowsSide side)
{
    static_assert(sizeof(ColumnsLds) <= sizeof(LearnLds), "one piece of LDS for both");
    __shared__ LearnLds lds;
    const int tid = threadIdx.x, lane = tid & (NHIP_WAVE - 1);
    if ((int)blockIdx.x < side.n_chains) {  // a carried sequence first: it takes longer than a group's rows
        static_assert(sizeof(lds.w) >= SEQ_MAX_OPS * sizeof(NhipSeqOp) + sizeof(int) * SEQ_MAX_ROWS * SEQ_ROW_WORDS,
                      "a carried sequence stages its records in the same LDS");
        const int c = blockIdx.x;
        sequence_chain(side.ops + side.chains.first_op[c], side.chains.first_op[c + 1] - side.chains.first_op[c],
                       side.chains.n_staged[c], reinterpret_cast<NhipSeqOp*>(lds.w),
                       reinterpret_cast<int (*)[SEQ_ROW_WORDS]>(
                           reinterpret_cast<char*>(lds.w) + SEQ_MAX_OPS * sizeof(NhipSeqOp)), tid);
        return;
    }
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int group = (int)blockIdx.x - side.n_chains;
    if (EVENTS && group < events.n_items) {
        typedef const __attribute__((address_space(4))) learn_i16 const_i16;
        const const_i16* at = reinterpret_cast<const const_i16*>(
            reinterpret_cast<uintptr_t>(events.items + group));
        learn_i16 w0 = at[0], w1 = at[1];
        asm volatile("" : "+s"(w0), "+s"(w1));
        struct Words { learn_i16 a, b; };
        const Words words = {w0, w1};
        columns_group(__builtin_bit_cast(ColumnsItem, words), events.AT, X, Yin, Y, filter,
                      *reinterpret_cast<ColumnsLds*>(&lds), wave, lane);
        return;
    }
    if (EVENTS) group -= events.n_items;
    // (constant address space: the whole record, and those of the filters, at once)
    typedef const __attribute__((address_space(4))) learn_i16 const_i16;
    const const_i16* at = reinterpret_cast<const const_i16*>(reinterpret_cast<uintptr_t>(tasks + group));
    learn_i16 w0 = at[0], w1 = at[1], fw = learn_i16{};
    if (n_filters > 0) fw = *reinterpret_cast<const const_i16*>(reinterpret_cast<uintptr_t>(filters));  // (two at least)
    asm volatile("" : "+s"(w0), "+s"(w1), "+s"(fw));
    struct Words { learn_i16 a, b; };
    const Words words = {w0, w1};
    const LearnTask task = __builtin_bit_cast(LearnTask, words);
    const bool mine = wave < task.n_rows;
    const int row = task.row0 + min(wave, task.n_rows - 1);
    // the old y, the filters of the row (a lane each, the first one's record being here already)
    const float* y_at = Yin + task.yin_start + (size_t)row * task.yin_stride0;
    FilterTarget target = task.target;
    const float* f_at = filter.F + (task.n_targets > 0 ? (size_t)target.y_start + row : 0);
    float f_first = 0.0f;
    if (task.n_targets > 1 && lane < task.n_targets) target = filter.targets[task.first_target + lane];
    float sum = 0.0f;
    // Every wave of the group has its activities in registers and LDS: the last group to say so may replace
    // them.  Nobody waits; nothing that another group wrote is read.  (Said here, while the rows are
    // still on their way, the last group's trips for the filters lie beside the other groups' rows.)
    // Additions to one word go one after the other, about 12 ns each: 500 groups that all told it of
    // themselves were what the launch waited for, their first waves' rows behind the answer (2000 x 2000:
    // 13.9 -> 9.8 us).  So a group tells one of LCOUNTERS words, each in a line of its own; the last there tells
    // the word behind them.
    auto read = [&]() LEARN_INLINE {
        if ((n_filters > 0 || task.own_groups > 0) && tid == 0) {
            const int n_groups = side.n_gemv_groups, mine = group % LCOUNTERS;
            auto tell = [&](int counter, int expected) {  // the last of `expected`? (it clears the word for the next launch)
                int* word = arrived + counter * LCOUNTER_WORDS;
                if (__hip_atomic_fetch_add(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != expected - 1) return 0;
                __hip_atomic_store(word, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return 1;
            };
            lds.last = task.own_groups > 0 ? tell(LCOUNTERS + 1 + task.own_filter, task.own_groups)
                                           : tell(mine, (n_groups - mine + LCOUNTERS - 1) / LCOUNTERS) &&
                                                 tell(LCOUNTERS, min(n_groups, LCOUNTERS));
        }
    };
    auto rows = [&](auto rule) LEARN_INLINE {
        learn_rows<decltype(rule)::value>(task, reinterpret_cast<const float*>(tasks), A, X, lds, wave, lane, tid, y_at,
                                          f_at, f_first, sum, read);
    };
    if (!task.learned) rows(std::integral_constant<int, 0>{});
    else if (task.rule.kind == LEARN_OUTER) rows(std::integral_constant<int, LEARN_OUTER>{});
    else if (task.rule.kind == NHIP_RULE_BCM) rows(std::integral_constant<int, NHIP_RULE_BCM>{});
    else rows(std::integral_constant<int, NHIP_RULE_OJA>{});
    if (mine) {
        const float y = sum + task.gamma;
        if (lane == 0) Y[task.y_start + (size_t)row * task.y_stride0] = y;
        float f_old = f_first;
        if (task.n_targets > 1 && lane < task.n_targets) f_old = filter.F[(size_t)target.y_start + row];
        if (lane < task.n_targets)
            filter.F[(size_t)target.y_start + row] = filter_step<true>(filter.targets, target, row, y, f_old);
        for (int q = lane + NHIP_WAVE; q < task.n_targets; q += NHIP_WAVE)
            filter_epilogue<true>(filter, make_int2(task.first_target + q, 1), row, y);
    }
    const bool own = task.own_groups > 0;  // activities of its item's groups alone: their last one replaces those
    if (!own && n_filters == 0) return;
    typedef const __attribute__((address_space(4))) learn_i8 const_i8;
    learn_i8 f2 = learn_i8{}, f3 = learn_i8{};
    if (n_filters > 2) {
        const const_i8* more = reinterpret_cast<const const_i8*>(reinterpret_cast<uintptr_t>(filters));
        f2 = more[2];
        f3 = more[min(3, n_filters - 1)];
    }
    __syncthreads();
    if (lds.last == 0) return;
    struct TwoFilters { LearnFilter a, b; };
    const TwoFilters here = __builtin_bit_cast(TwoFilters, fw);
    // Q filters by T threads, of which this one is t: in quads, and what is left behind the last quad an element a
    // thread; all of it requested together.
    auto step = [&](const auto& f, int t, auto threads) LEARN_INLINE {
        constexpr int T = decltype(threads)::value, U = 2;  // quads of a thread, of each filter
        constexpr int Q = sizeof(f) / sizeof(f[0]);
        const auto stepped = [](const LearnFilter& f, float s, float old) LEARN_INLINE {
            const float bx = __fmul_rn(f.b, s);
            return f.has_a ? __fsub_rn(bx, __fmul_rn(f.a, old)) : bx;
        };
        float st[Q], vt[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int i = (f[q].n & ~3) + t;
            st[q] = vt[q] = 0.0f;
            if (i < f[q].n) {
                st[q] = X[f[q].s_start + (size_t)i];
                vt[q] = filter.F[f[q].f_start + (size_t)i];
            }
        }
        int longest = 0;
#pragma unroll
        for (int q = 0; q < Q; ++q) longest = max(longest, f[q].n);
        for (int i0 = 4 * t; i0 < longest; i0 += 4 * U * T) {
            learn_f4 s[Q][U], v[Q][U];
#pragma unroll
            for (int q = 0; q < Q; ++q)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int i = i0 + 4 * u * T;
                    s[q][u] = v[q][u] = learn_f4{};
                    if (i + 4 <= f[q].n) {
                        s[q][u] = *reinterpret_cast<const learn_q4*>(X + f[q].s_start + (size_t)i);
                        v[q][u] = *reinterpret_cast<const learn_q4*>(filter.F + f[q].f_start + (size_t)i);
                    }
                }
#pragma unroll
            for (int q = 0; q < Q; ++q)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int i = i0 + 4 * u * T;
                    if (i + 4 <= f[q].n) {
                        learn_f4 y;
#pragma unroll
                        for (int e = 0; e < 4; ++e) y[e] = stepped(f[q], s[q][u][e], v[q][u][e]);
                        *reinterpret_cast<learn_q4*>(filter.F + f[q].f_start + (size_t)i) = y;
                    }
                }
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int i = (f[q].n & ~3) + t;
            if (i < f[q].n) filter.F[f[q].f_start + (size_t)i] = stepped(f[q], st[q], vt[q]);
        }
    };
    // The first two or four (the activities of both sides, the BCM rule's third) by all threads, the others by a wave
    // each.  (Two after the other by all threads, elements behind the last quad after those: 18 filters of up to 257
    // elements beside 21 groups, the launch 17.0 us, now 8.6; whole steps of the BCM rule on 2000 x 2000 14.5 -> 12.7,
    // on 92 x 92 9.5 -> 8.7, of Oja's 12.9 -> 12.3 and 8.7 -> 8.5.  With the records of more than two filters
    // requested at the kernel's begin 12.9, 8.9, 12.5, 8.7.)
    constexpr std::integral_constant<int, NHIP_WG> group_threads{};
    if (own || n_filters <= 2) {
        LearnFilter both[2] = {here.a, here.b};
        if (own) both[0] = filters[task.own_filter];
        if (own || n_filters < 2) both[1].n = 0;
        step(both, tid, group_threads);
        return;
    }
    LearnFilter first[4] = {here.a, here.b, __builtin_bit_cast(LearnFilter, f2), __builtin_bit_cast(LearnFilter, f3)};
    if (n_filters < 4) first[3].n = 0;
    step(first, tid, group_threads);
    for (int k = 4 + wave; k < n_filters; k += 4 * LROWS) {
        LearnFilter more[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            more[q] = filters[min(k + q * LROWS, n_filters - 1)];
            if (k + q * LROWS >= n_filters) more[q].n = 0;
        }
        step(more, lane, std::integral_constant<int, NHIP_WAVE>{});
    }
}

// Matrix a_start, a_stride0, M x N of A -> its columns, mp floats apart, from `out` of AT on; the records of the items
// first_record .. are told where it holds an infinity or a NaN (products of those with zeros count)
struct LearnColumns { int a_start, a_stride0, M, N, out, mp, first_record, n_records; };

__global__ __launch_bounds__(NHIP_WG) void lay_out_columns_kernel(const LearnColumns* __restrict__ mats, const float* A,
                                                                  float* AT, ColumnsItem* records) {
    constexpr int T = NHIP_WAVE;  // rows and columns of a block
    __shared__ float block[T][T + 1];
    const LearnColumns m = mats[blockIdx.y];
    const int lane = threadIdx.x & (T - 1), wave = threadIdx.x >> 6;
    bool odd = false;
    for (int c0 = blockIdx.x * T; c0 < m.N; c0 += gridDim.x * T)
        for (int r0 = 0; r0 < m.mp; r0 += T) {
            __syncthreads();
            for (int r = wave; r < T; r += NHIP_WG / T) {
                const bool inside = r0 + r < m.M && c0 + lane < m.N;
                const float v = inside ? A[m.a_start + (size_t)(r0 + r) * m.a_stride0 + c0 + lane] : 0.0f;
                odd |= (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u;
                block[r][lane] = v;
            }
            __syncthreads();
            for (int c = wave; c < T; c += NHIP_WG / T)
                if (c0 + c < m.N && r0 + lane < m.mp)
                    AT[(size_t)m.out + (size_t)(c0 + c) * m.mp + r0 + lane] = block[lane][c];
        }
    if (odd)
        for (int i = 0; i < m.n_records; ++i) records[m.first_record + i].all = 1;
}

template <typename Launch>
int learn_launch(void* stream, const int* tasks, int n_tasks, float* A, const float* X, const float* Yin, float* Y,
                 const int* targets, float* F, const int* filters, int n_filters, int* arrived, int n_more,
                 Launch&& launch) {
    RowsSide side;
    if (take_carried(side) && n_tasks <= 0) return NHIP_E_BADARG;  // an empty launch cannot carry it
    if (n_tasks == 0) return 0;
    if (n_tasks < 0 || !tasks || !A || !X || !Yin || !Y || !targets || !F || n_filters < 0)
        return NHIP_E_BADARG;
    if (n_filters > 0 && (!filters || !arrived)) return NHIP_E_BADARG;
    if (((reinterpret_cast<uintptr_t>(tasks) & 63) | (reinterpret_cast<uintptr_t>(filters) & 63)) != 0) return NHIP_E_BADARG;
    side.n_gemv_groups = n_tasks;
    FilterArgs filter{};
    filter.targets = reinterpret_cast<const FilterTarget*>(targets);
    filter.F = F;
    launch(dim3(n_tasks + n_more + side.n_chains), filter, side);
    NHIP_LAUNCH_CHECK();
    return 0;
}

}  // namespace

extern "C" int nhip_gemv_learn(void* stream, const int* tasks, int n_tasks, float* A,
                               const float* X, const float* Yin, float* Y, const int* targets, float* F,
                               const int* filters, int n_filters, int* arrived) {
    return learn_launch(stream, tasks, n_tasks, A, X, Yin, Y, targets, F, filters, n_filters, arrived, 0,
                        [&](dim3 grid, const FilterArgs& filter, const RowsSide& side) {
        NHIP_LAUNCH(gemv_learn_kernel<false>, grid, dim3(NHIP_WG), 0, static_cast<hipStream_t>(stream),
                    reinterpret_cast<const LearnTask*>(tasks), A, X, Yin, Y, filter,
                    reinterpret_cast<const LearnFilter*>(filters), n_filters, arrived, LearnEvents{}, side);
    });
}

extern "C" int nhip_gemv_learn_events(void* stream, const int* tasks, int n_tasks, float* A, const float* X,
                                      const float* Yin, float* Y, const int* targets, float* F, const int* filters,
                                      int n_filters, int* arrived, const int* items, int n_items, const float* AT) {
    if (n_items < 0 || (n_items > 0 && (!items || !AT)) || (reinterpret_cast<uintptr_t>(items) & 63)) {
        RowsSide none;
        take_carried(none);  // (whatever becomes of the launch)
        return NHIP_E_BADARG;
    }
    return learn_launch(stream, tasks, n_tasks, A, X, Yin, Y, targets, F, filters, n_filters, arrived, n_items,
                        [&](dim3 grid, const FilterArgs& filter, const RowsSide& side) {
        NHIP_LAUNCH(gemv_learn_kernel<true>, grid, dim3(NHIP_WG), 0, static_cast<hipStream_t>(stream),
                    reinterpret_cast<const LearnTask*>(tasks), A, X, Yin, Y, filter,
                    reinterpret_cast<const LearnFilter*>(filters), n_filters, arrived,
                    (LearnEvents{reinterpret_cast<const ColumnsItem*>(items), AT, n_items}), side);
    });
}

extern "C" int nhip_lay_out_columns(void* stream, const int* matrices, int n, int max_cols, const float* A, float* AT,
                                    int* records) {
    if (n == 0) return 0;
    if (n < 0 || n > 65535 || max_cols < 1 || !matrices || !A || !AT || !records) return NHIP_E_BADARG;
    const int blocks = (max_cols + NHIP_WAVE - 1) / NHIP_WAVE;
    NHIP_LAUNCH(lay_out_columns_kernel, dim3(blocks < 1024 ? blocks : 1024, n), dim3(NHIP_WG), 0,
                static_cast<hipStream_t>(stream), reinterpret_cast<const LearnColumns*>(matrices), A, AT,
                reinterpret_cast<ColumnsItem*>(records));
    NHIP_LAUNCH_CHECK();
    return 0;
}
