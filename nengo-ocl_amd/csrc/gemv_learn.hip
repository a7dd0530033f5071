// Products with matrices that Oja's or the BCM rule changes in the same step.
//
// As launches of their own, a step of such a matrix reads it for the product, reads and writes it for the
// rule, and a third launch steps the filters of the activities the rule reads (2000 x 2000: 8.0 + 10.4 + 4.7
// us).  All three need nothing but what is there before the first of them: the product takes the old
// matrix, the rule the old matrix and the old activities, and the filters only have to wait until
// nobody reads the old activities any more.  Here a wave owns a row: it requests the row once, writes it
// back with its change, and sums the old values in the reference's order; the group that is the last to
// have read its activities steps the filters.  2000 x 2000: 14.2 us; with the rule in the task's record and
// the arrivals told while the rows are on their way 13.8 (1003 x 1003, BCM, whole steps: 17.4 -> 17.0).
// Bound by launch and latency of one round of groups: without the stores it takes 1.5 us less, without
// the filters' tail 1.9, without the sums as long.
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
};
// A filter stepped when no group reads its output any more: F[f + i] = b S[s + i] - a F[f + i] (or b S[s + i])
struct LearnFilter {
    int s_start, f_start, n, has_a;
    float a, b;
    int pad0, pad1;
};
static_assert(sizeof(LearnTask) == 96 && sizeof(LearnFilter) == 32, "tables");

constexpr int LROWS = NHIP_WG / NHIP_WAVE;     // rows of a group
constexpr int LTILE = 128, LTILES = 16;        // columns of a tile, tiles of a pass
constexpr int LSTRIDE = LTILE + 4;             // words between tiles in LDS
constexpr int LCOLS = LTILE * LTILES;          // columns of a pass
typedef float learn_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int learn_lds(int c) { return (c >> 7) * LSTRIDE + (c & (LTILE - 1)); }

// VEC 4: rows, vectors and their starts are made of aligned quads; 1: any
// `read()`: called by all waves when every wave of the group has its activities, what it requested
// before (`early`) included.
template <int VEC, typename Read>
__device__ __forceinline__ void learn_rows(const LearnTask& task, float* A, const float* X,
                                           float (*s_w)[LTILES * LSTRIDE], float* s_x, float* s_pre,
                                           int wave, int lane, int tid, float early, float& sum, Read&& read) {
    const auto& rule = task.rule;
    const bool learned = task.learned != 0;
    constexpr int PER_LANE = LCOLS / NHIP_WAVE / VEC;   // accesses of a lane to its row, per pass
    constexpr int PER_THREAD = LCOLS / NHIP_WG / VEC;   // accesses of a thread to a vector, per pass
    typedef std::conditional_t<VEC == 4, learn_f4, float> vec;
    auto element = [](vec& v, int u) -> float& {
        if constexpr (VEC == 4) return reinterpret_cast<float*>(&v)[u];
        else return v;
    };
    const bool mine = wave < task.n_rows;  // the same for the wave; the others only meet the barriers
    const int row = task.row0 + wave;
    float* arow = A + task.a_start + (size_t)row * task.a_stride0;
    const float* xg = X + task.x_start;
    const float* pre = X + rule.pre_start;
    float post = 0.0f, theta = 0.0f;
    if (learned && mine) {
        post = X[rule.post_start + (size_t)row * rule.post_stride0];
        if (rule.kind == NHIP_RULE_BCM) theta = X[rule.theta_start + (size_t)row * rule.theta_stride0];
    }
#pragma unroll 1
    for (int c0 = 0; c0 < task.N; c0 += LCOLS) {
        const int n = min(task.N - c0, LCOLS);
        // the vectors first (the barrier waits for them), then the row: all of it under way together
        vec xv[PER_THREAD], pv[PER_THREAD], w[PER_LANE];
#pragma unroll
        for (int k = 0; k < PER_THREAD; ++k) {
            const int c = VEC * (tid + k * NHIP_WG);
            xv[k] = vec{};
            pv[k] = vec{};
            if (c < n) {
                xv[k] = *reinterpret_cast<const vec*>(xg + c0 + c);
                if (learned) pv[k] = *reinterpret_cast<const vec*>(pre + c0 + c);
            }
        }
        if (mine) {
#pragma unroll
            for (int k = 0; k < PER_LANE; ++k) {
                const int c = VEC * (lane + k * NHIP_WAVE);
#pragma unroll
                for (int u = 0; u < VEC; ++u) element(w[k], u) = -0.0f;
                if (c < n) w[k] = *reinterpret_cast<const vec*>(arow + c0 + c);
            }
        }
        if (c0 > 0) __syncthreads();  // the pass before has read its vectors
#pragma unroll
        for (int k = 0; k < PER_THREAD; ++k) {
            const int c = VEC * (tid + k * NHIP_WG);
            *reinterpret_cast<vec*>(s_x + learn_lds(c)) = xv[k];
            if (learned) *reinterpret_cast<vec*>(s_pre + c) = pv[k];
        }
        if (c0 + LCOLS >= task.N) asm volatile("" :: "v"(post), "v"(theta), "v"(early), "v"(sum));  // here by now
        __syncthreads();
        if (c0 + LCOLS >= task.N) read();
        if (mine) {
#pragma unroll
            for (int k = 0; k < PER_LANE; ++k) {
                const int c = VEC * (lane + k * NHIP_WAVE);
                *reinterpret_cast<vec*>(s_w[wave] + learn_lds(c)) = w[k];
                if (learned && c < n) {
                    vec p = *reinterpret_cast<const vec*>(s_pre + c);
#pragma unroll
                    for (int u = 0; u < VEC; ++u) {
                        float& e = element(w[k], u);
                        const float change = rule.kind == NHIP_RULE_BCM
                            ? learn_element<NHIP_RULE_BCM>(rule.alpha, rule.beta, 0.0f, 0.0f, element(p, u), post, theta)
                            : learn_element<NHIP_RULE_OJA>(rule.alpha, rule.beta, 0.0f, 0.0f, element(p, u), post, e);
                        e = __fadd_rn(e, change);
                    }
                    *reinterpret_cast<vec*>(arow + c0 + c) = w[k];
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int at = (lane >> 2) * LSTRIDE + (lane & 3);  // partial sum lane & 3 of tile lane >> 2
            float s = 0.0f;
#pragma unroll
            for (int e = 0; e < LTILE / 4; ++e) s = fmaf(s_w[wave][at + 4 * e], s_x[at + 4 * e], s);
            s = s + __shfl_xor(s, 2, NHIP_WAVE);
            s = s + __shfl_xor(s, 1, NHIP_WAVE);
            const int n_tiles = (n + LTILE - 1) / LTILE;
#pragma unroll 1
            for (int t = 0; t < n_tiles; ++t)
                sum = sum + task.alpha * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 4 * t));
        }
    }
}

__global__ __launch_bounds__(NHIP_WG) void gemv_learn_kernel(
    const LearnTask* __restrict__ tasks, int vec4, float* A, const float* X, const float* Yin, float* Y,
    FilterArgs filter, const LearnFilter* __restrict__ filters, int n_filters, int* arrived, RowsSide side)
{
    __shared__ __attribute__((aligned(16))) float s_w[LROWS][LTILES * LSTRIDE];
    __shared__ __attribute__((aligned(16))) float s_x[LTILES * LSTRIDE];
    __shared__ __attribute__((aligned(16))) float s_pre[LCOLS];
    __shared__ int s_last;
    const int tid = threadIdx.x, lane = tid & (NHIP_WAVE - 1);
    if ((int)blockIdx.x < side.n_chains) {  // a carried sequence first: it takes longer than a group's rows
        static_assert(sizeof(s_w) >= SEQ_MAX_OPS * sizeof(NhipSeqOp) + sizeof(int) * SEQ_MAX_ROWS * SEQ_ROW_WORDS,
                      "a carried sequence stages its records in the same LDS");
        const int c = blockIdx.x;
        sequence_chain(side.ops + side.chains.first_op[c], side.chains.first_op[c + 1] - side.chains.first_op[c],
                       side.chains.n_staged[c], reinterpret_cast<NhipSeqOp*>(s_w),
                       reinterpret_cast<int (*)[SEQ_ROW_WORDS]>(
                           reinterpret_cast<char*>(s_w) + SEQ_MAX_OPS * sizeof(NhipSeqOp)), tid);
        return;
    }
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const LearnTask task = tasks[blockIdx.x - side.n_chains];
    const bool mine = wave < task.n_rows;
    const int row = task.row0 + min(wave, task.n_rows - 1);
    // what the row needs at its end, requested now: the old y, the filters of the row (a lane each)
    const float y_old = Yin[task.yin_start + (size_t)row * task.yin_stride0];
    FilterTarget target = {};
    float f_old = 0.0f;
    if (lane < task.n_targets) {
        target = filter.targets[task.first_target + lane];
        f_old = filter.F[(size_t)target.y_start + row];
    }
    float sum = task.beta * y_old;
    // Every wave of the group has its activities in registers and LDS: the last group to say so may replace
    // them.  Nobody waits; nothing that another group wrote is read.  (Said here, while the rows are
    // still on their way, the last group's trips for the filters lie beside the other groups' rows.)
    auto read = [&] {
        if (n_filters > 0 && tid == 0)
            s_last = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                     (int)gridDim.x - side.n_chains - 1;
    };
    if (vec4 && ((task.a_start | task.a_stride0 | task.N | task.x_start |
                  (task.learned ? task.rule.pre_start : 0)) & 3) == 0)
        learn_rows<4>(task, A, X, s_w, s_x, s_pre, wave, lane, tid, f_old, sum, read);
    else
        learn_rows<1>(task, A, X, s_w, s_x, s_pre, wave, lane, tid, f_old, sum, read);
    if (mine) {
        const float y = sum + task.gamma;
        if (lane == 0) Y[task.y_start + (size_t)row * task.y_stride0] = y;
        if (lane < task.n_targets)
            filter.F[(size_t)target.y_start + row] = filter_step<true>(filter.targets, target, row, y, f_old);
        for (int q = lane + NHIP_WAVE; q < task.n_targets; q += NHIP_WAVE)
            filter_epilogue<true>(filter, make_int2(task.first_target + q, 1), row, y);
    }
    if (n_filters == 0) return;
    __syncthreads();
    if (s_last == 0) return;
    if (tid == 0) *arrived = 0;  // for the next launch
    for (int k = 0; k < n_filters; k += 2) {  // two at a time (the activities of both sides)
        const LearnFilter f[2] = {filters[k], filters[min(k + 1, n_filters - 1)]};
        const int n[2] = {f[0].n, k + 1 < n_filters ? f[1].n : 0};
        constexpr int U = 8;  // elements of a thread requested together, of each filter
        for (int i0 = tid; i0 < max(n[0], n[1]); i0 += U * NHIP_WG) {
            float sv[2][U], fv[2][U];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int i = i0 + u * NHIP_WG;
                    sv[q][u] = i < n[q] ? X[f[q].s_start + (size_t)i] : 0.0f;
                    fv[q][u] = i < n[q] ? filter.F[f[q].f_start + (size_t)i] : 0.0f;
                }
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int i = i0 + u * NHIP_WG;
                    if (i >= n[q]) break;
                    const float bx = __fmul_rn(f[q].b, sv[q][u]);
                    filter.F[f[q].f_start + (size_t)i] =
                        f[q].has_a ? __fsub_rn(bx, __fmul_rn(f[q].a, fv[q][u])) : bx;
                }
        }
    }
}

}  // namespace

extern "C" int nhip_gemv_learn(void* stream, const int* tasks, int n_tasks, float* A,
                               const float* X, const float* Yin, float* Y, const int* targets, float* F,
                               const int* filters, int n_filters, int* arrived) {
    RowsSide side;
    if (take_carried(side) && n_tasks <= 0) return NHIP_E_BADARG;  // an empty launch cannot carry it
    if (n_tasks == 0) return 0;
    if (n_tasks < 0 || !tasks || !A || !X || !Yin || !Y || !targets || !F || n_filters < 0)
        return NHIP_E_BADARG;
    if (n_filters > 0 && (!filters || !arrived)) return NHIP_E_BADARG;
    const int vec4 = ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(X)) & 15) == 0;
    side.n_gemv_groups = n_tasks;
    FilterArgs filter{};
    filter.targets = reinterpret_cast<const FilterTarget*>(targets);
    filter.F = F;
    NHIP_LAUNCH(gemv_learn_kernel, dim3(n_tasks + side.n_chains), dim3(NHIP_WG), 0,
                static_cast<hipStream_t>(stream), reinterpret_cast<const LearnTask*>(tasks),
                vec4, A, X, Yin, Y, filter,
                reinterpret_cast<const LearnFilter*>(filters), n_filters, arrived, side);
    NHIP_LAUNCH_CHECK();
    return 0;
}
