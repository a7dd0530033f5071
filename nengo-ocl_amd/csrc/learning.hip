// Weight-update rules that write a per-connection delta matrix: BCM, Oja, Voja.
// (PES is an outer product and runs through the element-wise kernel.)  Every rule
// is one pass over the delta matrix; a block is a run of consecutive elements of
// one connection's delta, handled by one 256-thread group, so that the row-major
// delta and weight / encoder matrices stream coalesced while the pre / post
// vectors come from cache.
#include "nhip_common.h"
#include "learn_math.h"

namespace {

#define NHIP_STREAM(s) static_cast<hipStream_t>(s)

struct LearnDesc {
    int pre_start, pre_stride0, post_start, post_stride0;
    int aux_start, aux_stride0, delta_start, delta_stride0;
    int shape1, offset, count, alpha_bits;
    int beta_bits, learn_start, scale_start, scale_stride0;
};

typedef float learn_f4 __attribute__((ext_vector_type(4)));

// Bound by the stream of the matrix, if its loads are all under way together: a thread takes four
// elements of a block of 1024, as one 16-byte access where rows, strides and starts allow that and
// otherwise 256 elements apart, and requests everything it needs before it forms the first change.
// One 2000 x 2000 matrix, Oja in place: 12.5 -> 11.0 us on average, 8.6 -> 6.6 us at best (32 MB: 4.9
// TB/s); an element at a time, each waited for before the next was requested, was the slower one.
template <int RULE>
__global__ __launch_bounds__(NHIP_WG) void learning_kernel(const LearnDesc* __restrict__ desc,
                                                           int inc, int aligned, const float* PRE,
                                                           const float* POST, const float* AUX,
                                                           float* DELTA, const float* LEARN,
                                                           const float* SCALE) {
    const LearnDesc d = desc[blockIdx.x];
    const float alpha = nhip_bits(d.alpha_bits), beta = nhip_bits(d.beta_bits);
    const float* pre = PRE + d.pre_start;
    const float* post = POST + d.post_start;
    const float* aux = AUX + d.aux_start;
    float* delta = DELTA + d.delta_start;
    const float learn = RULE == NHIP_RULE_VOJA ? LEARN[d.learn_start] : 0.0f;
    const float* scale = RULE == NHIP_RULE_VOJA ? SCALE + d.scale_start : nullptr;
    const int i0 = d.offset / d.shape1, j0 = d.offset - i0 * d.shape1;  // once per block
    // inc: the change is added to the matrix DELTA points at (which may be the weights or
    // encoders AUX is: each element is read, then written, by one thread only)
    const bool in_place = RULE != NHIP_RULE_BCM && aux == delta && d.aux_stride0 == d.delta_stride0;
    int quad_bits = d.shape1 | d.offset | d.count | d.delta_start | d.delta_stride0;
    if (RULE != NHIP_RULE_BCM) quad_bits |= d.aux_start | d.aux_stride0;
    if (aligned && (quad_bits & 3) == 0) {  // uniform
        const bool pre_quads = d.pre_stride0 == 1 && (d.pre_start & 3) == 0;
        for (int k = 4 * threadIdx.x; k < d.count; k += 4 * NHIP_WG) {
            int i, j;
            nhip_row_col(i0, j0, k, d.shape1, d.count, i, j);
            learn_f4* dst = reinterpret_cast<learn_f4*>(delta + (size_t)i * d.delta_stride0 + j);
            learn_f4 x, m, now = {0.0f, 0.0f, 0.0f, 0.0f};
            if (RULE == NHIP_RULE_BCM) m = aux[(size_t)i * d.aux_stride0];
            else m = *reinterpret_cast<const learn_f4*>(aux + (size_t)i * d.aux_stride0 + j);
            if (inc) now = in_place ? m : *dst;
            if (pre_quads) {
                x = *reinterpret_cast<const learn_f4*>(pre + j);
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) x[u] = pre[(size_t)(j + u) * d.pre_stride0];
            }
            const float y = post[(size_t)i * d.post_stride0];
            const float sc = RULE == NHIP_RULE_VOJA ? scale[(size_t)i * d.scale_stride0] : 0.0f;
            learn_f4 out;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                out[u] = learn_element<RULE>(alpha, beta, learn, sc, x[u], y, m[u]);
                if (inc) out[u] = __fadd_rn(now[u], out[u]);
            }
            *dst = out;
        }
        return;
    }
    for (int k0 = threadIdx.x; k0 < d.count; k0 += 4 * NHIP_WG) {
        float x[4], y[4], m[4], sc[4], now[4];
        float* dst[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {  // (past the end: the last element again, not written)
            int i, j;
            nhip_row_col(i0, j0, min(k0 + u * NHIP_WG, d.count - 1), d.shape1, d.count, i, j);
            dst[u] = delta + (size_t)i * d.delta_stride0 + j;
            x[u] = pre[(size_t)j * d.pre_stride0];
            y[u] = post[(size_t)i * d.post_stride0];
            m[u] = aux[(size_t)i * d.aux_stride0 + (RULE == NHIP_RULE_BCM ? 0 : j)];
            sc[u] = RULE == NHIP_RULE_VOJA ? scale[(size_t)i * d.scale_stride0] : 0.0f;
            now[u] = inc ? *dst[u] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (k0 + u * NHIP_WG >= d.count) break;
            const float out = learn_element<RULE>(alpha, beta, learn, sc[u], x[u], y[u], m[u]);
            *dst[u] = inc ? __fadd_rn(now[u], out) : out;
        }
    }
}

}  // namespace

extern "C" int nhip_learning_rule(void* stream, int rule, int inc, const int* desc, int n_blocks,
                                  const float* PRE, const float* POST, const float* AUX,
                                  float* DELTA, const float* LEARN, const float* SCALE) {
    if (n_blocks == 0) return 0;
    if (n_blocks < 0 || !desc || !PRE || !POST || !AUX || !DELTA) return NHIP_E_BADARG;
    const LearnDesc* d = reinterpret_cast<const LearnDesc*>(desc);
    const dim3 grid(n_blocks), block(NHIP_WG);
    const int aligned = ((reinterpret_cast<uintptr_t>(PRE) | reinterpret_cast<uintptr_t>(AUX) |
                          reinterpret_cast<uintptr_t>(DELTA)) & 15) == 0;
    switch (rule) {
    case NHIP_RULE_BCM:
        NHIP_LAUNCH(learning_kernel<NHIP_RULE_BCM>, grid, block, 0, NHIP_STREAM(stream), d,
                           inc, aligned, PRE, POST, AUX, DELTA, LEARN, SCALE);
        break;
    case NHIP_RULE_OJA:
        NHIP_LAUNCH(learning_kernel<NHIP_RULE_OJA>, grid, block, 0, NHIP_STREAM(stream), d,
                           inc, aligned, PRE, POST, AUX, DELTA, LEARN, SCALE);
        break;
    case NHIP_RULE_VOJA:
        if (!LEARN || !SCALE) return NHIP_E_BADARG;
        NHIP_LAUNCH(learning_kernel<NHIP_RULE_VOJA>, grid, block, 0, NHIP_STREAM(stream),
                           d, inc, aligned, PRE, POST, AUX, DELTA, LEARN, SCALE);
        break;
    default:
        return NHIP_E_BADARG;
    }
    NHIP_LAUNCH_CHECK();
    return 0;
}
