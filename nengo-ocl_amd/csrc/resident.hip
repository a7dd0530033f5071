// Many timesteps of a small network in one launch.
//
// A step of a network of a few hundred neurons is a handful of short launches, each a chain of
// dependent reads of records, states and operands from memory and the start of a launch on top:
// 8.5 us a step for two populations of 100 neurons, whatever the kernels do inside.  Here one work-group
// copies everything such a network consists of -- signals, work lists, parameters -- into its LDS,
// runs n steps there, and copies back what the steps wrote.  The host (hipra_resident.py) sorts the
// operations into phases that touch different memory, with a barrier between them, and gives every wave a
// program of its own.  Operations are the block functions of the ordinary launches on LDS instead of
// memory; the three that make up most steps of such networks have a form of their own, since a wave
// alone on its SIMD is bound by the number of instructions (5 clocks each, 13 where one waits for the
// other): the same arithmetic with everything that can be known beforehand resolved by the host.
// Whole steps, two launches replayed as a graph -> this one: two populations of 100 neurons 8.5 -> 2.55 us, of
// 1000 8.7 -> 6.65; 16 populations of 20 with 10 inputs each 10.9 -> 5.6.  An operation costs a wave 0.2-0.4 us to
// fetch, 64 neurons 0.75 us (0.93 where both waves of a SIMD have some, 1.35 and more with sums of inputs), a
// row of 100 columns 1.1 us.
#include <cstdint>
#include <type_traits>

#include "nhip_common.h"
#include "gemv_rows.h"
#include "sequence_ops.h"

namespace {

constexpr int RES_WG = 512, RES_WAVES = RES_WG / NHIP_WAVE;
constexpr int RES_LDS_WORDS = 39 * 1024;  // 156 KB

// words [lds, lds + words) of the LDS image mirror `words` words at `ptr`; both on 16-byte boundaries
struct ResSpan {
    unsigned long long ptr;
    int words, lds, write_back, pad;
};

// kinds of the GEMV with its epilogue: 16 rows of four lanes per task, up to 64 rows of one item
// per task (dot products of at most 4 columns), one row per task (at least 128 columns)
enum { RES_ROWS4 = 16, RES_ROWS1 = 32, RES_LONG = 48 };  // + EPI_NONE, EPI_LIF, EPI_FILTER2, EPI_NEURON
// currents of at most one dot product of at most 4 columns and their LIF neurons, 64 per task; rows of
// one dot product and their filters, 16 per task; first-order filters, 64 elements per task
enum { RES_LIF = 64, RES_DECODE = 65, RES_FILTER = 66 };

struct ResOp {
    int kind;          // NHIP_SEQ_*, or one of the kinds above + the epilogue; 0: nothing
    int n_tasks;       // wave tasks of the operation; this wave takes first, first + stride, ...
    int first;
    int last;          // a barrier follows
    int n_rows;        // rows of the work list
    int lanes;         // sequence operations: lanes per row (at most 64)
    int i0, upsample;  // opcode of a unary function
    int stride, pad;
    int p[8];          // word offsets into the LDS image
    double d0;         // dt
    unsigned long long global;  // address outside the image (probe samples, table of inputs)
    int q[4];          // epilogue: pops or targets, parts, sum ranges
    int pad2[2];
};
static_assert(sizeof(ResSpan) == 24 && sizeof(ResOp) == 112, "tables");

struct ResLif {   // 24 words: up to 64 neurons of one population
    int n_rows, n_cols, yin, yin_stride;   // word offsets of the task's first row
    int a, a_stride, x, x_stride;
    float alpha, beta, gamma, tau;
    float ref, spike;                      // spike: the output of a neuron that spikes
    int y, v;                              // y: where the current goes, < 0: nowhere
    int w, s, sum_first, sum_n;            // the vector operand as a sum of parts
    int store_sum, pad[3];
};
struct ResDecode {  // 12 words: one row
    int a, x, n, y;
    int yin, first_target, n_targets, row;
    float alpha, beta, gamma;
    int pad;
};
struct ResFilter { int x, y; float a, b; };  // y = b x - a y; a NaN stands for y = b x (host: a is never NaN)
static_assert(sizeof(ResLif) == 96 && sizeof(ResDecode) == 48 && sizeof(ResFilter) == 16, "tables");

// The sums of gemv_rows_ref_block<1, EPI_LIF, true, true> and lif_epilogue.
__device__ __forceinline__ void res_lif(const ResOp& op, float* image, int lane) {
    float* sig = image + op.p[4];
    const float dtu = (float)(op.d0 / (double)op.upsample);
    for (int t = op.first; t < op.n_tasks; t += op.stride) {
        const ResLif d = reinterpret_cast<const ResLif*>(image + op.p[0])[t];
        const int r = min(lane, d.n_rows - 1);
        const int n_cols = __builtin_amdgcn_readfirstlane(d.n_cols);
        float v = sig[d.v + r], w = sig[d.w + r];
        float sum = d.beta * sig[d.yin + r * d.yin_stride];
        if (n_cols > 0) {
            float x[4], p[4];
            const int n_parts = __builtin_amdgcn_readfirstlane(d.sum_n);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = e < n_cols ? sig[d.x + e * d.x_stride] : 0.0f;
            if (n_parts > 0) {
                const int2* parts = reinterpret_cast<const int2*>(image + op.q[1]) + d.sum_first;
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = 0.0f;
                // lane k forms the products of part k, which are added in order
                for (int q0 = 0; q0 < n_parts; q0 += NHIP_WAVE) {
                    const int m = min(n_parts - q0, NHIP_WAVE);
                    const int2 part = parts[q0 + min(lane, m - 1)];
                    const float scale = sig[part.y];
                    float own[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) own[e] = e < n_cols ? fmaf(sig[part.x + e], scale, 0.0f) : 0.0f;
                    for (int k = 0; k < m; ++k)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (e < n_cols)
                                x[e] = x[e] + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(own[e]), k));
                }
                if (d.store_sum && lane == 0) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (e < n_cols) sig[d.x + e] = x[e];
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                p[e] = e < n_cols ? fmaf(sig[d.a + r * d.a_stride + e], x[e], 0.0f) : 0.0f;
            sum = sum + d.alpha * ((p[0] + p[2]) + (p[1] + p[3]));
        }
        const float j = sum + d.gamma;
        const bool spiked = lif_step(j, v, w, d.tau, d.ref, dtu, op.upsample);
        if (lane < d.n_rows) {
            if (d.y >= 0) sig[d.y + r] = j;
            sig[d.v + r] = v;
            sig[d.w + r] = w;
            sig[d.s + r] = spiked ? d.spike : 0.0f;
        }
    }
}

// The sums of gemv_rows_ref_block<4, EPI_FILTER2>.
__device__ __forceinline__ void res_decode(const ResOp& op, float* image, int lane) {
    constexpr int TILE = 128, CHUNK = 8;
    float* sig = image + op.p[4];
    for (int t = op.first; t < op.n_tasks; t += op.stride) {
        const int slot = 16 * t + (lane >> 2), k = lane & 3;
        const ResDecode d = reinterpret_cast<const ResDecode*>(image + op.p[0])[min(slot, op.n_rows - 1)];
        const FilterTarget* targets = reinterpret_cast<const FilterTarget*>(image + op.q[0]);
        float sum = d.beta * sig[d.yin];
        for (int c0 = 0; c0 < d.n; c0 += TILE) {
            const int c1 = min(c0 + TILE, d.n);
            const float* a = sig + d.a;
            const float* x = sig + d.x;
            float s = 0.0f;
            auto chunk = [&](auto width, int c) {  // so many steps of the partial sum, all of them inside
                constexpr int W = decltype(width)::value;
                float av[W], xv[W];
#pragma unroll
                for (int e = 0; e < W; ++e) {
                    av[e] = a[c + 4 * e];
                    xv[e] = x[c + 4 * e];
                }
#pragma unroll
                for (int e = 0; e < W; ++e) s = fmaf(av[e], xv[e], s);
            };
            int c = c0 + k;
            for (; c + 4 * (4 * CHUNK - 1) < c1; c += 16 * CHUNK) chunk(std::integral_constant<int, 4 * CHUNK>{}, c);
            if (c + 4 * (2 * CHUNK - 1) < c1) {
                chunk(std::integral_constant<int, 2 * CHUNK>{}, c);
                c += 8 * CHUNK;
            }
            if (c + 4 * (CHUNK - 1) < c1) {
                chunk(std::integral_constant<int, CHUNK>{}, c);
                c += 4 * CHUNK;
            }
            if (c + 4 * (CHUNK / 2 - 1) < c1) {
                chunk(std::integral_constant<int, CHUNK / 2>{}, c);
                c += 2 * CHUNK;
            }
            for (; c < c1; c += 4) s = fmaf(a[c], x[c], s);
            s = s + __shfl_xor(s, 2, NHIP_WAVE);
            s = s + __shfl_xor(s, 1, NHIP_WAVE);
            sum = sum + d.alpha * s;
        }
        if (k == 0 && slot < op.n_rows) {
            const float y = sum + d.gamma;
            sig[d.y] = y;
            for (int q = 0; q < d.n_targets; ++q) {
                const FilterTarget target = targets[d.first_target + q];
                float* f = sig + target.y_start + d.row;
                *f = filter_step<true>(targets, target, d.row, y, *f);
            }
        }
    }
}

__device__ __forceinline__ void res_filter(const ResOp& op, float* image, int lane) {
    float* sig = image + op.p[4];
    for (int t = op.first; t < op.n_tasks; t += op.stride) {
        const int i = NHIP_WAVE * t + lane;
        if (i >= op.n_rows) return;
        const ResFilter f = reinterpret_cast<const ResFilter*>(image + op.p[0])[i];
        const float bx = __fmul_rn(f.b, sig[f.x]);
        sig[f.y] = isnan(f.a) ? bx : __fsub_rn(bx, __fmul_rn(f.a, sig[f.y]));
    }
}

template <int LPR, int EPI, bool WIDE, bool WAVE_TASK>
__device__ __forceinline__ void res_rows(const ResOp& op, float* image, int lane) {
    float* sig = image + op.p[4];
    EpilogueArgs epi{};
    if (EPI == EPI_LIF || EPI == EPI_NEURON) {
        LifArgs& lif = epi.lif;
        lif.pops = reinterpret_cast<const LifPop*>(image + op.q[0]);
        lif.dt = (float)op.d0;
        lif.dtu = (float)(op.d0 / (double)op.upsample);  // formed in double and rounded once, as in nhip_lif
        lif.dt_inv = (float)(1.0 / op.d0);
        lif.upsample = op.upsample;
        lif.V = lif.W = lif.S = lif.N = sig;
        lif.TAU = lif.REF = lif.AMP = sig;
        lif.parts = reinterpret_cast<const int2*>(image + op.q[1]);
        lif.sum_ranges = op.i0 ? reinterpret_cast<const int2*>(image + op.q[2]) : nullptr;
    }
    if (epi_filters(EPI)) {
        epi.filter.item_targets = reinterpret_cast<const int2*>(image + op.q[2]);
        epi.filter.targets = reinterpret_cast<const FilterTarget*>(image + op.q[0]);
        epi.filter.F = sig;
    }
    for (int t = op.first; t < op.n_tasks; t += op.stride)
        gemv_rows_ref_block<LPR, EPI, WIDE, WAVE_TASK>(
            reinterpret_cast<const GemvItem*>(image + op.p[0]), reinterpret_cast<const float4*>(image + op.p[1]),
            reinterpret_cast<const GemvDot*>(image + op.p[2]), reinterpret_cast<const GemvTask*>(image + op.p[3]),
            op.n_rows, sig, sig, sig, sig, t >> 2, ((t & 3) << 6) | lane, &epi);
}

// rows of a sequence operation; at most 64 lanes per row: their block functions need no barrier
#define RES_SEQ(ROW, CALL)                                                                        \
    for (int t = op.first; t < op.n_tasks; t += op.stride) {                                      \
        const int L = op.lanes, row = t * (NHIP_WAVE / L) + ln / L, lane = ln & (L - 1);          \
        if (row < op.n_rows) {                                                                    \
            const ROW& d = reinterpret_cast<const ROW*>(image + op.p[0])[row];                    \
            (void)d;                                                                              \
            CALL;                                                                                 \
        }                                                                                         \
    }

struct ResPrograms { int first[RES_WAVES + 1]; };  // wave w runs ops[first[w] .. first[w + 1])

__global__ __launch_bounds__(RES_WG) void resident_kernel(const ResSpan* __restrict__ spans, int n_spans,
                                                          const ResOp* __restrict__ ops, ResPrograms programs,
                                                          int n_steps) {
    __shared__ __attribute__((aligned(16))) float image[RES_LDS_WORDS];
    const int tid = threadIdx.x, ln = tid & (NHIP_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int s = 0; s < n_spans; ++s) {
        const ResSpan sp = spans[s];
        const float4* src = reinterpret_cast<const float4*>(static_cast<uintptr_t>(sp.ptr));
        float4* dst = reinterpret_cast<float4*>(image + sp.lds);
        for (int i = tid; i < (sp.words >> 2); i += RES_WG) dst[i] = src[i];
        if (tid < (sp.words & 3))
            image[sp.lds + (sp.words & ~3) + tid] = reinterpret_cast<const float*>(src)[(sp.words & ~3) + tid];
    }
    __syncthreads();
    const int k0 = programs.first[wave], k1 = programs.first[wave + 1];
    for (int step = 0; step < n_steps; ++step) {
#pragma unroll 1
        for (int k = k0; k < k1; ++k) {
            const ResOp op = ops[k];
            switch (op.kind) {
                case RES_ROWS4 + EPI_NONE: res_rows<4, EPI_NONE, false, false>(op, image, ln); break;
                case RES_ROWS4 + EPI_LIF: res_rows<4, EPI_LIF, false, false>(op, image, ln); break;
                case RES_ROWS4 + EPI_NEURON: res_rows<4, EPI_NEURON, false, false>(op, image, ln); break;
                case RES_ROWS4 + EPI_FILTER2: res_rows<4, EPI_FILTER2, false, false>(op, image, ln); break;
                case RES_ROWS1 + EPI_NONE: res_rows<1, EPI_NONE, true, true>(op, image, ln); break;
                case RES_ROWS1 + EPI_LIF: res_rows<1, EPI_LIF, true, true>(op, image, ln); break;
                case RES_ROWS1 + EPI_NEURON: res_rows<1, EPI_NEURON, true, true>(op, image, ln); break;
                case RES_ROWS1 + EPI_FILTER2: res_rows<1, EPI_FILTER2, true, true>(op, image, ln); break;
                case RES_LONG + EPI_NONE: res_rows<NHIP_WAVE, EPI_NONE, true, false>(op, image, ln); break;
                case RES_LONG + EPI_FILTER2: res_rows<NHIP_WAVE, EPI_FILTER2, true, false>(op, image, ln); break;
                case RES_LIF: res_lif(op, image, ln); break;
                case RES_DECODE: res_decode(op, image, ln); break;
                case RES_FILTER: res_filter(op, image, ln); break;
                case NHIP_SEQ_RESET:
                    RES_SEQ(int4, reset_block(d, image + op.p[1], lane, L))
                    break;
                case NHIP_SEQ_COPY:
                    RES_SEQ(CopyDesc, copy_block(d, image + op.p[1], image + op.p[2], lane, L))
                    break;
                case NHIP_SEQ_SLICEDCOPY:
                    RES_SEQ(SlicedDesc, slicedcopy_block(d, image + op.p[1], image + op.p[2],
                                                         reinterpret_cast<const int*>(image + op.p[3]),
                                                         reinterpret_cast<const int*>(image + op.p[4]), lane, L))
                    break;
                case NHIP_SEQ_ELEMENTWISE_INC:
                    RES_SEQ(EwDesc, elementwise_inc_block(d, image + op.p[1], image + op.p[2], image + op.p[3],
                                                          lane, L))
                    break;
                case NHIP_SEQ_LINEARFILTER:
                    RES_SEQ(LfDesc, linearfilter_block(d, reinterpret_cast<int2*>(image + op.p[1]), image + op.p[2],
                                                       image + op.p[3], image + op.p[4], image + op.p[5],
                                                       image + op.p[6], image + op.p[7], row, lane, L))
                    break;
                case NHIP_SEQ_TIMEUPDATE:
                    timeupdate_block(image + op.p[0], image + op.p[1], op.d0, ln);
                    break;
                case NHIP_SEQ_PRESENTINPUT:
                    RES_SEQ(PiDesc, presentinput_block(d, (float)op.d0, image + op.p[1], image + op.p[2],
                                                       reinterpret_cast<const float*>(static_cast<uintptr_t>(op.global)),
                                                       lane, L))
                    break;
                case NHIP_SEQ_DIRECT_UNARY:
                    RES_SEQ(int4, direct_unary_block(op.i0, d, image + op.p[1], image + op.p[2], lane, L))
                    break;
                case NHIP_SEQ_PROBES:
                    RES_SEQ(ProbeDesc, probes_block(d, image + op.p[1], reinterpret_cast<int*>(image + op.p[2]),
                                                    image + op.p[3], image + op.p[4],
                                                    reinterpret_cast<float*>(static_cast<uintptr_t>(op.global)), row,
                                                    lane, L))
                    break;
                default: break;
            }
            if (op.last) __syncthreads();  // (every program has as many)
        }
    }
    for (int s = 0; s < n_spans; ++s) {
        const ResSpan sp = spans[s];
        if (!sp.write_back) continue;
        const float4* src = reinterpret_cast<const float4*>(image + sp.lds);
        float4* dst = reinterpret_cast<float4*>(static_cast<uintptr_t>(sp.ptr));
        for (int i = tid; i < (sp.words >> 2); i += RES_WG) dst[i] = src[i];
        if (tid < (sp.words & 3))
            reinterpret_cast<float*>(dst)[(sp.words & ~3) + tid] = image[sp.lds + (sp.words & ~3) + tid];
    }
}

}  // namespace

extern "C" int nhip_resident(void* stream, const void* spans, int n_spans, const void* ops, const int* first_op,
                             int n_waves, int n_steps) {
    if (n_steps == 0) return 0;
    if (!spans || !ops || !first_op || n_spans <= 0 || n_waves != RES_WAVES || n_steps < 0) return NHIP_E_BADARG;
    ResPrograms programs;
    for (int w = 0; w <= RES_WAVES; ++w) {
        programs.first[w] = first_op[w];
        if (first_op[w] < 0 || (w > 0 && first_op[w] < first_op[w - 1])) return NHIP_E_BADARG;
    }
    NHIP_LAUNCH(resident_kernel, dim3(1), dim3(RES_WG), 0, static_cast<hipStream_t>(stream),
                static_cast<const ResSpan*>(spans), n_spans, static_cast<const ResOp*>(ops), programs, n_steps);
    NHIP_LAUNCH_CHECK();
    return 0;
}
