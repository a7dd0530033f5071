// Sparse matrix-vector products of a timestep: Y[b] (=|+=) A[b] @ X[b] for many
// sparse matrices in one launch.
//
// The reference keeps each matrix in CSR or ELLPACK and launches one kernel per
// matrix with one work-item per row (clra_gemv.py:1570-1646, :1649-1755).  Here all
// matrices of a step share one launch and one layout made for 64-wide waves:
// rows are cut into slices of 64 and padded to the longest row of the slice, rounded
// up to a multiple of 4; inside a slice elements 4q .. 4q+3 of row r sit side by side
// at slice_start + 256 q + 4 r (sliced ELLPACK with slice height 64, four elements of
// a row per 16 bytes).  A wave owns a slice, lane r owns row r: a load of values or
// column indices is one 16-byte access per lane and one contiguous 1-KiB run per wave
// (a quarter of the address work of 4-byte accesses), and each row is still summed
// strictly in column order (one fused multiply-add per stored element, starting from
// the old y when incrementing), which is the order of the reference's CSR kernel, so
// results are bit-identical to a sequential float32 restatement.  Only the gather
// from X is irregular; X is a few MB at most and stays in cache.  Where the host found
// a run of SPMV_WINDOW consecutive elements of X that holds a good part of a slice's
// column indices (band matrices, rings), the wave first copies that run into LDS and
// takes the elements inside it from there: only the lanes whose column lies outside
// go to the cache, which spares it one look-up per line and instruction.
#include <type_traits>
#include "nhip_common.h"
#include "neuron_math.h"
#include "sequence_ops.h"

namespace {

// First-order filters stepped on the fresh rows of a product (the synapse of a connection
// through a sparse matrix): per slice {first target, number of targets, first row of the
// slice in its matrix, 0}; targets as for the dense products.  slice_epi == nullptr: none.
struct SpmvEpi {
    const int4* slice_epi;
    const FilterTarget* targets;
    float* F;
};

// A sequence armed with nhip_gemv_tile_carry rides in extra work-groups behind those of the
// product (256 threads run a chain; further waves of such a group end at once: a barrier
// waits for the waves that are still running).
struct SpmvSide {
    const NhipSeqOp* ops;
    SeqChains chains;
    int n_chains;       // 0: none
    int n_groups;       // groups of the product itself
};

__device__ __forceinline__ void spmv_side_chain(const SpmvSide& side, void* lds) {
    if (threadIdx.x >= NHIP_WG) return;
    const int c = blockIdx.x - side.n_groups;
    NhipSeqOp* s_ops = reinterpret_cast<NhipSeqOp*>(lds);
    int (*s_rows)[SEQ_ROW_WORDS] = reinterpret_cast<int (*)[SEQ_ROW_WORDS]>(
        reinterpret_cast<char*>(lds) + SEQ_MAX_OPS * sizeof(NhipSeqOp));
    sequence_chain(side.ops + side.chains.first_op[c],
                   side.chains.first_op[c + 1] - side.chains.first_op[c], side.chains.n_staged[c],
                   s_ops, s_rows, threadIdx.x);
}

__device__ __forceinline__ void spmv_filter_rows(const SpmvEpi& epi, int s, int lane, float y) {
    const int4 e = epi.slice_epi[s];
    for (int q = 0; q < e.y; ++q) {
        const FilterTarget t = epi.targets[e.x + q];
        float* f = epi.F + (size_t)t.y_start + e.z + lane;
        const float bx = __fmul_rn(nhip_bits(t.b_bits), y);
        *f = t.na ? __fsub_rn(bx, __fmul_rn(nhip_bits(t.a_bits), *f)) : bx;
    }
}

struct SpmvSlice {
    int data_start;  // offset of the slice in `cols` / `vals`
    int width;       // stored elements per row of the slice (longest row, rounded up to 4)
    int len_start;   // offset of the slice's row lengths in `row_len`
    int n_rows;      // rows in the slice (<= 64)
    int x_start;     // element offsets of the item's X and of the slice's first Y row
    int y_start;
    int inc;         // 1: Y += A X, 0: Y = A X
    int window;      // first element (relative to x_start, multiple of 4) of the run of X kept in LDS; < 0: none
};

constexpr int SPMV_WINDOW = 1024;  // elements of X a wave keeps in LDS (4 KiB)

typedef int spmv_i4 __attribute__((ext_vector_type(4)));
typedef float spmv_f4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(NHIP_WG) void spmv_sell_kernel(
    const SpmvSlice* __restrict__ slices, int n_slices, const int* __restrict__ row_len,
    const int* __restrict__ cols, const float* __restrict__ vals, const float* X, float* Y,
    SpmvEpi epi, SpmvSide side)
{
    const int lane = threadIdx.x & (NHIP_WAVE - 1);
    const int s = blockIdx.x * (NHIP_WG / NHIP_WAVE) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __shared__ __attribute__((aligned(16))) float s_x[NHIP_WG / NHIP_WAVE][SPMV_WINDOW];
    static_assert(sizeof(s_x) >= SEQ_MAX_OPS * sizeof(NhipSeqOp) + sizeof(int) * SEQ_MAX_ROWS * SEQ_ROW_WORDS,
                  "a carried sequence stages its records in the same LDS");
    if (side.n_chains > 0 && (int)blockIdx.x >= side.n_groups) return spmv_side_chain(side, s_x);
    // waves past the last slice have no work but still meet the group barrier below
    const bool has_slice = s < n_slices;
    SpmvSlice sl = slices[has_slice ? s : 0];
    if (!has_slice) { sl.n_rows = 0; sl.width = 0; sl.window = -1; }
    float* wx = s_x[__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)];
    if (sl.window >= 0) {
        const spmv_f4* src = reinterpret_cast<const spmv_f4*>(X + sl.x_start + sl.window) + lane;
#pragma unroll
        for (int i = 0; i < SPMV_WINDOW / (4 * NHIP_WAVE); ++i)
            reinterpret_cast<spmv_f4*>(wx)[i * NHIP_WAVE + lane] = src[i * NHIP_WAVE];
    }
    __syncthreads();  // every wave of the group arrives here exactly once
    const unsigned win_lo = sl.window >= 0 ? (unsigned)sl.window : 0u;
    const unsigned win_n = sl.window >= 0 ? (unsigned)SPMV_WINDOW : 0u;
    const bool live = lane < sl.n_rows;
    const int len = live ? row_len[sl.len_start + lane] : 0;
    const float* x = X + sl.x_start;
    float acc = (live && sl.inc) ? Y[(size_t)sl.y_start + lane] : 0.0f;
    const int n_quads = sl.width >> 2;  // the host pads the width to a multiple of 4
    if (n_quads > 0) {
        const spmv_i4* c = reinterpret_cast<const spmv_i4*>(cols + (size_t)sl.data_start) + lane;
        const spmv_f4* v = reinterpret_cast<const spmv_f4*>(vals + (size_t)sl.data_start) + lane;
        // values and column indices of the next two quads are requested before the
        // gathers from X of the current one (past the end: the last again, unused)
        const int q1 = min(1, n_quads - 1);
        spmv_i4 ci = __builtin_nontemporal_load(c), ci1 = __builtin_nontemporal_load(c + (size_t)q1 * NHIP_WAVE);
        spmv_f4 vi = __builtin_nontemporal_load(v), vi1 = __builtin_nontemporal_load(v + (size_t)q1 * NHIP_WAVE);
        for (int q = 0; q < n_quads; ++q) {
            const int qn = min(q + 2, n_quads - 1);
            const spmv_i4 cn = __builtin_nontemporal_load(c + (size_t)qn * NHIP_WAVE);
            const spmv_f4 vn = __builtin_nontemporal_load(v + (size_t)qn * NHIP_WAVE);
            const int k0 = 4 * q;
            float xi[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const unsigned w = (unsigned)ci[u] - win_lo;  // position inside the run kept in LDS
                xi[u] = (k0 + u < len) ? (w < win_n ? wx[w] : x[ci[u]]) : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (k0 + u < len) acc = fmaf(vi[u], xi[u], acc);
            ci = ci1; vi = vi1;
            ci1 = cn; vi1 = vn;
        }
    }
    if (live) {  // no wave without a slice is live
        Y[(size_t)sl.y_start + lane] = acc;
        if (epi.slice_epi) spmv_filter_rows(epi, s, lane, acc);
    }
}

// ---- products whose X is mostly zero (spikes) -------------------------------------------
// One bit per element of X ("is not +0.0"), made by a launch of its own (or, for an X of at most
// SPMV_MASK_INLINE_COLS elements, by every work-group for itself), is kept in LDS by every
// work-group; for a stored element whose bit is clear the operand is the constant +0.0
// instead of a look-up in the cache.  The sum is formed as above, term by term, so the
// result has the bits of the kernel above whatever X and the matrix hold.  Groups are
// persistent, and their waves take one of two things until none is left:
//   a quarter of a slice, four lanes per row (spmv_skip_rows), while that is what keeps the waves
//     busy: 2,000 rows of 100 6.4 us, against 20.4 by whole slices (one lane per row is bound by its chain
//     of loads, bits and look-ups); 100,000 rows of 100 24.5 against 30.6 (4.1 of them the launch for
//     the bits).  Quarters are dealt out over the groups first and the waves of a group second.
//   a whole slice, a lane per row (spmv_skip_slice), where the slices are enough for all waves: a
//     load is then one run of 1 KiB, and a wave starts a chain of loads once per slice instead
//     of four times.  1,000,000 rows of 100 139 us (5.9 TB/s), by quarters 161; rows of 20 43 and 52, of 4
//     21 and 35.  Which one: see `spmv_takes_slices`.
// Every group's own copy of the bits made from X costs 400 KB of reads per compute unit at
// 100,000 elements (30.4 us in all instead of 24.5): hence the limit below.
constexpr int SPMV_SKIP_WG = 1024;
constexpr int SPMV_MASK_WORDS = 36864;  // 144 KiB of LDS: X of up to 1,179,648 elements
constexpr int SPMV_MASK_U = 16;
// X of at most so many elements: every group forms the bits itself, without a launch for them
constexpr int SPMV_MASK_INLINE_COLS = 32768;

// Sixteen rows of a slice by one wave, four lanes per row: lane j of a row holds its quads j,
// j + 4, ..., U of them at a time, so a row of 100 elements is two requests deep instead of
// the seven it takes a lane alone, and four times as many waves have requests in flight.  The sum
// still runs through the row element by element: each quad's lane adds its four products to the
// sum the quad before left, which reaches it by an exchange inside the four lanes.  All the
// bits of a batch are read first, then all the elements of X that are needed, then it is
// summed: a batch waits for memory twice and not once per element.  What is stored past a row's
// end is not looked at, value or column: such an element counts as +0 times -0, which changes no
// sum.  (The loads of a batch past the last quad take that one again: past the row's end too.)
// ONE: every element of X that is not +0.0 is `one` (spikes of one amplitude): the bits are all
// there is to know, and X is not looked up at all.
template <int U, bool ONE>
__device__ __forceinline__ float spmv_skip_rows(const spmv_i4* c, const spmv_f4* v, int n_quads,
                                                int len, int j, const float* x,
                                                const unsigned* s_mask, float one, float acc) {
    auto request = [&](int q, spmv_i4 (&cq)[U], spmv_f4 (&vq)[U]) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const size_t at = (size_t)min(q + 4 * i + j, n_quads - 1) * NHIP_WAVE;
            cq[i] = __builtin_nontemporal_load(c + at);
            vq[i] = __builtin_nontemporal_load(v + at);
        }
    };
    auto add = [&](int q, const spmv_i4 (&cq)[U], const spmv_f4 (&vq)[U]) {
        unsigned word[U][4];
        float xi[U][4];
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const bool stored = 4 * (q + 4 * i + j) + u < len;
                word[i][u] = s_mask[stored ? (unsigned)cq[i][u] >> 5 : 0u];
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const unsigned col = (unsigned)cq[i][u];
                const bool stored = 4 * (q + 4 * i + j) + u < len;
                const bool set = stored & ((word[i][u] >> (col & 31u)) & 1u);
                xi[i][u] = stored ? 0.0f : -0.0f;
                if (ONE) xi[i][u] = set ? one : xi[i][u];
                else if (set) xi[i][u] = x[col];
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < U; ++i) {
            if (q + 4 * i >= n_quads) break;  // uniform
            float w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) w[u] = 4 * (q + 4 * i + j) + u < len ? vq[i][u] : 0.0f;
#define SPMV_LINK(J, CTRL)                                                               \
            {                                                                            \
                _Pragma("unroll") for (int u = 0; u < 4; ++u) acc = fmaf(w[u], xi[i][u], acc); \
                acc = __int_as_float(__builtin_amdgcn_update_dpp(                        \
                    0, __float_as_int(acc), CTRL, 0xF, 0xF, true));                      \
            }
            SPMV_LINK(0, 0x00)  // the sum of lane 0 of the four to all of them, then lane 1's, ...
            SPMV_LINK(1, 0x55)
            SPMV_LINK(2, 0xAA)
            SPMV_LINK(3, 0xFF)
#undef SPMV_LINK
        }
    };
    spmv_i4 ca[U], cb[U];
    spmv_f4 va[U], vb[U];
    request(0, ca, va);
#pragma unroll 1
    for (int q = 0; q < n_quads; q += 8 * U) {
        if (n_quads > 4 * U) request(q + 4 * U, cb, vb);
        __builtin_amdgcn_sched_barrier(0);
        add(q, ca, va);
        if (q + 4 * U >= n_quads) break;
        request(q + 8 * U, ca, va);
        __builtin_amdgcn_sched_barrier(0);
        add(q + 4 * U, cb, vb);
    }
    return acc;
}

// A slice by one wave, lane r its row r; SPMV_SLICE_U quads of a row are in flight per lane while
// the ones before are summed.  ONE and what lies past a row's end: as above.
constexpr int SPMV_SLICE_U = 4;
template <bool ONE>
__device__ __forceinline__ float spmv_skip_slice(const spmv_i4* c, const spmv_f4* v, int n_quads,
                                                 int len, const float* x, const unsigned* s_mask,
                                                 float one, float acc) {
    constexpr int U = SPMV_SLICE_U;
    spmv_i4 ci[U];
    spmv_f4 vi[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
        ci[i] = spmv_i4{0, 0, 0, 0};
        vi[i] = spmv_f4{0.0f, 0.0f, 0.0f, 0.0f};
        if (i < n_quads) {  // the same for all lanes
            ci[i] = __builtin_nontemporal_load(c + (size_t)i * NHIP_WAVE);
            vi[i] = __builtin_nontemporal_load(v + (size_t)i * NHIP_WAVE);
        }
    }
    for (int q = 0; q < n_quads; q += U) {
        // the next U quads are requested before the look-ups of the current ones
        spmv_i4 cn[U];
        spmv_f4 vn[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            cn[i] = ci[i];
            vn[i] = vi[i];
            if (q + U + i < n_quads) {
                cn[i] = __builtin_nontemporal_load(c + (size_t)(q + U + i) * NHIP_WAVE);
                vn[i] = __builtin_nontemporal_load(v + (size_t)(q + U + i) * NHIP_WAVE);
            }
        }
        float xi[U][4];
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const unsigned col = (unsigned)ci[i][u];
                const bool stored = 4 * (q + i) + u < len;
                const bool set = stored && ((s_mask[col >> 5] >> (col & 31u)) & 1u);
                xi[i][u] = 0.0f;
                if (ONE) xi[i][u] = set ? one : 0.0f;
                else if (set) xi[i][u] = x[col];
            }
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (4 * (q + i) + u < len) acc = fmaf(vi[i][u], xi[i][u], acc);
#pragma unroll
        for (int i = 0; i < U; ++i) {
            ci[i] = cn[i];
            vi[i] = vn[i];
        }
    }
    return acc;
}

// Whole slices or quarters, for a grid of `n_waves` waves.  Measured (kernel time in us, slices /
// quarters; n rows and columns, rows of 32, 60, 100; 4,096 waves; one amplitude):
//   n = 160,000 (0.61 slices per wave)  17.5/17.6  24.7/21.8   33.8/32.5
//       220,000 (0.84)                  18.7/20.3  27.0/27.2   38.1/41.6
//       260,000 (0.99)                  20.4/22.3  30.2/30.5   43.3/47.3
//       300,000 (1.14)                  28.0/24.3  40.5/33.3   60.0/52.0   (a second, nearly empty round)
//       400,000 (1.53)                  30.0/28.7  42.6/42.9   63.6/67.6
//       500,000 (1.91)                  32.6/34.0  47.9/51.3   73.3/81.3
//       700,000 (2.67)                  41.5/44.1  63.5/69.2   98.8/112.2
//     1,000,000 (3.81)                  54.1/60.4  86.7/99.9  138.8/161.1
// Shorter rows are mostly the start of a task, which quarters pay four times: rows of 12, n =
// 100,000 12.8/12.4, 150,000 12.1/13.8, 300,000 16.7/18.4; of 24, 100,000 15.2/14.3, 120,000 15.4/15.3,
// 200,000 16.5/18.7.  (Short: by the width of the first slice.  A choice by one slice is the
// same for every group, and either form is right for any.)
constexpr int SPMV_SHORT_WIDTH = 24;
__device__ __forceinline__ bool spmv_takes_slices(int n_slices, int width, int n_waves) {
    if (width <= SPMV_SHORT_WIDTH) return 9LL * n_slices >= 4LL * n_waves;
    return n_slices <= n_waves ? 5LL * n_slices >= 4LL * n_waves : 2LL * n_slices >= 3LL * n_waves;
}

// smallest and largest bits of the elements of X that are not +0.0
__device__ __forceinline__ void spmv_wave_range(unsigned& lo, unsigned& hi) {
#pragma unroll
    for (int off = NHIP_WAVE / 2; off > 0; off >>= 1) {
        lo = min(lo, (unsigned)__shfl_xor((int)lo, off, NHIP_WAVE));
        hi = max(hi, (unsigned)__shfl_xor((int)hi, off, NHIP_WAVE));
    }
}

// a bit per element; with `ranges` also {smallest, largest} bits of the set ones of every 64
__global__ __launch_bounds__(NHIP_WG) void spmv_mask_kernel(const float* __restrict__ X, int n,
                                                            unsigned* __restrict__ mask,
                                                            unsigned* __restrict__ ranges,
                                                            int n_words) {
    const int i = blockIdx.x * NHIP_WG + threadIdx.x;
    const unsigned bits = i < n ? __float_as_uint(X[i]) : 0u;
    const unsigned long long b = __ballot(bits != 0u);
    unsigned lo = bits != 0u ? bits : 0xffffffffu, hi = bits;
    spmv_wave_range(lo, hi);
    if ((threadIdx.x & (NHIP_WAVE - 1)) == 0 && 2 * (i >> 6) < n_words) {
        // (words past the last element of X, up to a multiple of 4, are written as zero)
        mask[2 * (i >> 6)] = (unsigned)b;
        mask[2 * (i >> 6) + 1] = (unsigned)(b >> 32);
        if (ranges) {
            ranges[2 * (i >> 6)] = lo;
            ranges[2 * (i >> 6) + 1] = hi;
        }
    }
}

__global__ __launch_bounds__(SPMV_SKIP_WG) void spmv_sell_skip_kernel(
    const SpmvSlice* __restrict__ slices, int n_slices, const int* __restrict__ row_len,
    const int* __restrict__ cols, const float* __restrict__ vals, const float* X, float* Y,
    const unsigned* __restrict__ mask, const unsigned* __restrict__ ranges, int x_start, int n_cols,
    SpmvEpi epi, SpmvSide side)
{
    __shared__ __attribute__((aligned(16))) unsigned s_mask[SPMV_MASK_WORDS];
    __shared__ unsigned s_one[SPMV_SKIP_WG / NHIP_WAVE], s_mixed[SPMV_SKIP_WG / NHIP_WAVE];
    if (side.n_chains > 0 && (int)blockIdx.x >= side.n_groups) return spmv_side_chain(side, s_mask);
    const int lane = threadIdx.x & (NHIP_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int WAVES = SPMV_SKIP_WG / NHIP_WAVE;
    const int stride = side.n_groups * WAVES;
    unsigned lo = 0xffffffffu, hi = 0u;  // smallest and largest bits of a set element
    if (mask) {
        const int n_mask_quads = (n_cols + 127) / 128;
        for (int i = threadIdx.x; i < n_mask_quads; i += SPMV_SKIP_WG) {
            reinterpret_cast<spmv_i4*>(s_mask)[i] = reinterpret_cast<const spmv_i4*>(mask)[i];
            if (!ranges) continue;
            const spmv_i4 r = reinterpret_cast<const spmv_i4*>(ranges)[i];
            lo = min(lo, min((unsigned)r[0], (unsigned)r[2]));
            hi = max(hi, max((unsigned)r[1], (unsigned)r[3]));
        }
    } else {
        // the bits straight from X: a wave forms one 64-bit word per 64 elements, the
        // elements of SPMV_MASK_U words requested together
        const unsigned* bits = reinterpret_cast<const unsigned*>(X + x_start);
        const int n_words = (n_cols + NHIP_WAVE - 1) / NHIP_WAVE;
#pragma unroll 1
        for (int w0 = wave; w0 < n_words; w0 += WAVES * SPMV_MASK_U) {
            unsigned e[SPMV_MASK_U];
#pragma unroll
            for (int j = 0; j < SPMV_MASK_U; ++j) {
                const int i = (w0 + j * WAVES) * NHIP_WAVE + lane;
                const unsigned b = bits[min(i, n_cols - 1)];
                e[j] = i < n_cols ? b : 0u;
            }
#pragma unroll
            for (int j = 0; j < SPMV_MASK_U; ++j) {
                const unsigned long long b = __ballot(e[j] != 0u);
                const int w = w0 + j * WAVES;
                if (lane == 0 && w < n_words)
                    reinterpret_cast<unsigned long long*>(s_mask)[w] = b;
                lo = min(lo, e[j] != 0u ? e[j] : 0xffffffffu);
                hi = max(hi, e[j]);
            }
        }
    }
    const bool values_known = ranges || !mask;  // (else: look-ups)
    if (values_known) {
        // the wave's set elements: one value (0: there are none), or several
        const unsigned long long some = __ballot(hi != 0u);
        const unsigned one_w = some ? __builtin_amdgcn_readlane(hi, __ffsll(some) - 1) : 0u;
        const unsigned long long other = __ballot(hi != 0u && (lo != hi || hi != one_w));
        if (lane == 0) {
            s_one[wave] = one_w;
            s_mixed[wave] = other != 0ull;
        }
    }
    const bool whole = spmv_takes_slices(n_slices, slices[0].width, stride);  // uniform over the grid
    __syncthreads();  // the only barrier; every thread reaches it
    bool one_value = false;  // all set elements have the same bits (or there are none)
    float one = 0.0f;
    if (values_known) {
        const unsigned w = lane < WAVES ? s_one[lane] : 0u;
        const unsigned long long some = __ballot(w != 0u);
        const unsigned first = some ? __builtin_amdgcn_readlane(w, __ffsll(some) - 1) : 0u;
        one_value = __ballot(lane < WAVES && (s_mixed[lane] != 0u || (w != 0u && w != first))) == 0ull;
        one = __uint_as_float(first);
    }
    auto take_slices = [&](auto one_tag) {
        for (int s = blockIdx.x * WAVES + wave; s < n_slices; s += stride) {
            const SpmvSlice sl = slices[s];
            const bool live = lane < sl.n_rows;
            const int len = live ? row_len[sl.len_start + lane] : 0;
            float acc = (live && sl.inc) ? Y[(size_t)sl.y_start + lane] : 0.0f;
            const spmv_i4* c = reinterpret_cast<const spmv_i4*>(cols + (size_t)sl.data_start) + lane;
            const spmv_f4* v = reinterpret_cast<const spmv_f4*>(vals + (size_t)sl.data_start) + lane;
            const float* x = X + sl.x_start;
            acc = spmv_skip_slice<decltype(one_tag)::value>(c, v, sl.width >> 2, len, x, s_mask, one,
                                                            acc);
            if (live) {
                Y[(size_t)sl.y_start + lane] = acc;
                if (epi.slice_epi) spmv_filter_rows(epi, s, lane, acc);
            }
        }
    };
    if (whole) {
        if (one_value) take_slices(std::true_type());
        else take_slices(std::false_type());
        return;
    }
    for (int t = wave * side.n_groups + blockIdx.x; t < 4 * n_slices; t += stride) {
        const int s = t >> 2, row = 16 * (t & 3) + (lane >> 2), j = lane & 3;
        const SpmvSlice sl = slices[s];
        if (16 * (t & 3) >= sl.n_rows) continue;  // uniform: a short last slice
        const bool live = row < sl.n_rows;
        const int len = live ? row_len[sl.len_start + row] : 0;
        float acc = (live && sl.inc) ? Y[(size_t)sl.y_start + row] : 0.0f;
        const int n_quads = sl.width >> 2;
        const spmv_i4* c = reinterpret_cast<const spmv_i4*>(cols + (size_t)sl.data_start) + row;
        const spmv_f4* v = reinterpret_cast<const spmv_f4*>(vals + (size_t)sl.data_start) + row;
        const float* x = X + sl.x_start;
        // (all of these conditions are the same for all lanes)
        if (n_quads > 4 && one_value)
            acc = spmv_skip_rows<4, true>(c, v, n_quads, len, j, x, s_mask, one, acc);
        else if (n_quads > 4)
            acc = spmv_skip_rows<4, false>(c, v, n_quads, len, j, x, s_mask, one, acc);
        else if (n_quads > 0 && one_value)
            acc = spmv_skip_rows<1, true>(c, v, n_quads, len, j, x, s_mask, one, acc);
        else if (n_quads > 0)
            acc = spmv_skip_rows<1, false>(c, v, n_quads, len, j, x, s_mask, one, acc);
        if (live && j == 0) {
            Y[(size_t)sl.y_start + row] = acc;
            if (epi.slice_epi) spmv_filter_rows(epi, s, row, acc);
        }
    }
}

// ---- spikes that the launch of the neurons has left as bits ------------------------------
// All spikes have the value `one` (nhip_gemv_rows_lif_bits), so a launch for the bits, look-ups of X and
// a look at the values it holds fall away.  The layout is one of its own, which leaves a few instructions per
// stored element (the kernel above is bound by them: 100 elements of a row cost it as much at 6
// bytes each as at 8):
//  - column indices of 24 bits, or of 16 where X has fewer than 65,536 elements;
//  - rows are padded to whole quads for every lane of a row, with a column past X's end, whose bit is
//    clear, and the value -0: such an element adds -0, which changes no sum, so nothing asks
//    where a row ends;
//  - LANES (1, 2, 4) per row, as many as fill the waves: a lane holds every LANES-th quad of its row,
//    and the sum goes from lane to lane, quad by quad, as in spmv_skip_rows -- which every lane of
//    the row computes, so fewer lanes are fewer instructions.
// A wave's record and first elements are on their way before the bits are.
// A step with its product, in calls of 1,000 (the launch of the neurons included; before: bits in a launch of
// their own, or by every group for itself, 32-bit indices, four lanes per row): 100,000 rows of 100 25.4 -> 17.3
// us (the product 18.9 -> 12.6, of 70 MB: 5.6 TB/s), of 20 16.3 -> 9.3; 180,000 of 60 27.9 -> 18.4; 10,000 rows of
// 100 11.1 -> 10.2; 2,000 of 30 9.1 -> 8.9; 1,000,000 rows of 20 64.9 -> 49.2.
template <int BITS> struct SpmvBitCols;
template <> struct SpmvBitCols<16> {
    struct quad { int w[2]; };
    static constexpr int WORDS = 2;
    static __device__ __forceinline__ unsigned raw(const quad& q, int u) {
        return (u & 1) ? (unsigned)q.w[u >> 1] >> 16 : (unsigned)q.w[u >> 1];
    }
};
template <> struct SpmvBitCols<24> {
    struct quad { int w[3]; };
    static constexpr int WORDS = 3;
    static __device__ __forceinline__ unsigned raw(const quad& q, int u) {
        switch (u) {
            case 0: return (unsigned)q.w[0];
            case 1: return __builtin_amdgcn_alignbit((unsigned)q.w[1], (unsigned)q.w[0], 24);
            case 2: return __builtin_amdgcn_alignbit((unsigned)q.w[2], (unsigned)q.w[1], 16);
            default: return (unsigned)q.w[2] >> 8;
        }
    }
};

template <typename T>
__device__ __forceinline__ T spmv_uniform(const T* p) {
    static_assert(sizeof(T) == 16, "four words");
    typedef const __attribute__((address_space(4))) spmv_i4* scalar;
    return __builtin_bit_cast(T, *(scalar)reinterpret_cast<uintptr_t>(p));
}

template <int LANES, int BITS>
__global__ __launch_bounds__(SPMV_SKIP_WG) void spmv_sell_bits_kernel(
    const SpmvSlice* __restrict__ slices, int n_slices, const int* __restrict__ cols,
    const float* __restrict__ vals, float* Y, const unsigned* __restrict__ mask, int n_cols, float one,
    SpmvEpi epi, SpmvSide side)
{
    __shared__ __attribute__((aligned(16))) unsigned s_mask[SPMV_MASK_WORDS];
    if (side.n_chains > 0 && (int)blockIdx.x >= side.n_groups) return spmv_side_chain(side, s_mask);
    typedef SpmvBitCols<BITS> Cols;
    typedef typename Cols::quad quad;
    constexpr int WAVES = SPMV_SKIP_WG / NHIP_WAVE, U = 4, ROWS = NHIP_WAVE / LANES;
    const int lane = threadIdx.x & (NHIP_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane % LANES, stride = side.n_groups * WAVES, n_tasks = LANES * n_slices;
    const unsigned one_bits = __float_as_uint(one);
    // quads k .. k + U - 1 of every lane of the row; past the last one: that one again (WHOLE: there are U)
    auto request = [&](auto whole, const SpmvSlice& sl, int row, int k, quad (&c)[U], spmv_f4 (&v)[U]) {
        const int m = sl.width / (4 * LANES);  // quads per lane (the host pads the width)
        const char* cs = reinterpret_cast<const char*>(cols) + (size_t)(sl.data_start >> 2) * sizeof(quad);
        const char* vs = reinterpret_cast<const char*>(vals + (size_t)sl.data_start);
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int q = decltype(whole)::value ? k + i : min(k + i, m - 1);
            const unsigned at = (unsigned)(LANES * q + j) * NHIP_WAVE + row;
            const int* cp = reinterpret_cast<const int*>(cs + at * (unsigned)sizeof(quad));
#pragma unroll
            for (int w = 0; w < Cols::WORDS; ++w) c[i].w[w] = __builtin_nontemporal_load(cp + w);
            v[i] = __builtin_nontemporal_load(reinterpret_cast<const spmv_f4*>(vs + at * 16u));
        }
    };
    float acc = 0.0f;
    auto add = [&](auto whole, int n, const quad (&c)[U], const spmv_f4 (&v)[U]) {  // n quads of every lane
        float x[U][4];
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                x[i][u] = __uint_as_float(s_mask[(Cols::raw(c[i], u) >> 5) & ((1u << (BITS - 5)) - 1u)]);
        __builtin_amdgcn_sched_barrier(0);  // (every look-up of the batch before the first is waited for)
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u)  // the bit, spread over the word: the value or +0
                x[i][u] = __uint_as_float((unsigned)__builtin_amdgcn_sbfe((int)__float_as_uint(x[i][u]),
                                                                          Cols::raw(c[i], u), 1) & one_bits);
#pragma unroll
        for (int i = 0; i < U; ++i) {
            if (!decltype(whole)::value && i >= n) break;  // uniform
#define SPMV_LINK(CTRL)                                                                      \
            {                                                                                \
                _Pragma("unroll") for (int u = 0; u < 4; ++u) acc = fmaf(v[i][u], x[i][u], acc); \
                if (LANES > 1)                                                               \
                    acc = __int_as_float(__builtin_amdgcn_update_dpp(                        \
                        0, __float_as_int(acc), CTRL, 0xF, 0xF, true));                      \
            }
            if (LANES == 4) {  // the sum of lane 0 of the four to all of them, then lane 1's, ...
                SPMV_LINK(0x00) SPMV_LINK(0x55) SPMV_LINK(0xAA) SPMV_LINK(0xFF)
            } else if (LANES == 2) {
                SPMV_LINK(0xA0) SPMV_LINK(0xF5)
            } else {
                SPMV_LINK(0xE4)
            }
#undef SPMV_LINK
        }
    };
    constexpr std::true_type all{};
    constexpr std::false_type part{};

    int t = wave * side.n_groups + blockIdx.x;
    // the bits are asked for first: what they are waited for with is only asked for behind them
    // (one quad more than the bits: the column of the padding is X's first past its end)
    const int n_mask_quads = (n_cols + 127) / 128;
    spmv_i4 bits = {0, 0, 0, 0};
    if ((int)threadIdx.x < n_mask_quads) bits = reinterpret_cast<const spmv_i4*>(mask)[threadIdx.x];
    SpmvSlice sl = slices[min(t / LANES, n_slices - 1)];
    int row = ROWS * (t % LANES) + lane / LANES;
    quad ca[U], cb[U];
    spmv_f4 va[U], vb[U];
    if (sl.width > 0) request(part, sl, row, 0, ca, va);  // (uniform; a wave without a task: of the last slice)
    // what the row needs at its end is requested now as well: its old sum and its first filter's old value
    int4 filters = make_int4(0, 0, 0, 0);
    FilterTarget f_first = {};
    float y_old = 0.0f, f_old = 0.0f;
    auto request_ends = [&](int s) {
        // (tables that no launch writes, at addresses that are the wave's: scalar loads, which
        // wait for nothing but themselves)
        if (epi.slice_epi) filters = spmv_uniform(epi.slice_epi + s);
        if (filters.y > 0) f_first = spmv_uniform(epi.targets + filters.x);
        y_old = f_old = 0.0f;
        if (row < sl.n_rows) {
            if (sl.inc) y_old = Y[(size_t)sl.y_start + row];
            if (filters.y > 0) f_old = epi.F[(size_t)f_first.y_start + filters.z + row];
        }
    };
    request_ends(min(t / LANES, n_slices - 1));
    if ((int)threadIdx.x <= n_mask_quads) reinterpret_cast<spmv_i4*>(s_mask)[threadIdx.x] = bits;
    for (int i = threadIdx.x + SPMV_SKIP_WG; i <= n_mask_quads; i += SPMV_SKIP_WG)
        reinterpret_cast<spmv_i4*>(s_mask)[i] =
            i < n_mask_quads ? reinterpret_cast<const spmv_i4*>(mask)[i] : spmv_i4{0, 0, 0, 0};
    __syncthreads();  // the only barrier; every thread reaches it
    while (t < n_tasks) {
        const int m = sl.width / (4 * LANES);
        const bool live = row < sl.n_rows;
        acc = y_old;
        int k = 0;
#pragma unroll 1
        for (; k + 3 * U <= m; k += 2 * U) {  // a batch is requested before the one ahead of it is summed
            request(all, sl, row, k + U, cb, vb);
            __builtin_amdgcn_sched_barrier(0);
            add(all, U, ca, va);
            request(all, sl, row, k + 2 * U, ca, va);
            __builtin_amdgcn_sched_barrier(0);
            add(all, U, cb, vb);
        }
        for (; k < m; k += 2 * U) {  // up to three batches are left, the last of them in part
            const bool more = k + U < m, yet_more = k + 2 * U < m;
            if (more) {
                request(part, sl, row, k + U, cb, vb);
                __builtin_amdgcn_sched_barrier(0);
                add(all, U, ca, va);
                if (yet_more) {
                    request(part, sl, row, k + 2 * U, ca, va);
                    __builtin_amdgcn_sched_barrier(0);
                    add(all, U, cb, vb);
                } else {
                    add(part, m - k - U, cb, vb);
                }
            } else {
                add(part, m - k, ca, va);
            }
        }
        if (live && j == 0) {
            Y[(size_t)sl.y_start + row] = acc;
            if (filters.y > 0) {
                epi.F[(size_t)f_first.y_start + filters.z + row] =
                    filter_step<false>(epi.targets, f_first, row, acc, f_old);
                filter_epilogue<false>(FilterArgs{nullptr, epi.targets, epi.F, nullptr},
                                       make_int2(filters.x + 1, filters.y - 1), filters.z + row, acc);
            }
        }
        t += stride;
        if (t >= n_tasks) break;
        sl = slices[t / LANES];
        row = ROWS * (t % LANES) + lane / LANES;
        if (sl.width > 0) request(part, sl, row, 0, ca, va);
        request_ends(t / LANES);
    }
}

// a sequence armed by nhip_gemv_tile_carry is the calling launch's, whatever becomes of it
SpmvSide take_side() {
    SpmvSide side{};
    const NhipCarried armed = nhip_carried;
    nhip_carried = NhipCarried{};
    if (armed.n_chains > 0) {
        side.ops = static_cast<const NhipSeqOp*>(armed.ops);
        for (int c = 0; c <= NHIP_SEQ_MAX_CHAINS; ++c) side.chains.first_op[c] = armed.first_op[c];
        for (int c = 0; c < NHIP_SEQ_MAX_CHAINS; ++c) side.chains.n_staged[c] = armed.n_staged[c];
        side.n_chains = armed.n_chains;
    }
    return side;
}

int launch_plain(void* stream, const int* slices, int n_slices, const int* row_len,
                 const int* cols, const float* vals, const float* X, float* Y, SpmvEpi epi) {
    SpmvSide side = take_side();
    if (n_slices == 0) return side.n_chains > 0 ? NHIP_E_BADARG : 0;  // nothing to ride in
    if (n_slices < 0 || !slices || !row_len || !cols || !vals || !X || !Y) return NHIP_E_BADARG;
    // the kernel reads `cols`, `vals` and the runs of X it keeps in LDS 16 bytes at a time
    if ((reinterpret_cast<uintptr_t>(cols) | reinterpret_cast<uintptr_t>(vals) |
         reinterpret_cast<uintptr_t>(X)) & 15)
        return NHIP_E_BADARG;
    const int wpg = NHIP_WG / NHIP_WAVE;
    side.n_groups = (n_slices + wpg - 1) / wpg;
    NHIP_LAUNCH(spmv_sell_kernel, dim3(side.n_groups + side.n_chains), dim3(NHIP_WG), 0,
                       static_cast<hipStream_t>(stream),
                       reinterpret_cast<const SpmvSlice*>(slices), n_slices, row_len, cols, vals, X,
                       Y, epi, side);
    NHIP_LAUNCH_CHECK();
    return 0;
}

// Groups of a product of spikes with so many tasks for waves at most.
bool skip_groups(SpmvSide& side, int most) {
    static int n_cu = 0;
    if (n_cu == 0) {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess)
            return false;
        n_cu = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    }
    // a group takes a whole compute unit (its LDS holds the bits of X), so the groups of a
    // carried sequence need compute units of their own: with one product group per compute
    // unit they would only start when the product is over
    side.n_groups = min(n_cu > side.n_chains ? n_cu - side.n_chains : n_cu, most);
    return true;
}

// The product, behind a launch for the bits of X where X is long.
int launch_skip(void* stream, const int* slices, int n_slices, const int* row_len,
                const int* cols, const float* vals, const float* X, float* Y, int x_start,
                int n_cols, unsigned* mask, unsigned* ranges, SpmvEpi epi) {
    SpmvSide side = take_side();
    if (n_slices == 0) return side.n_chains > 0 ? NHIP_E_BADARG : 0;  // nothing to ride in
    if (n_slices < 0 || !slices || !row_len || !cols || !vals || !X || !Y || !mask || x_start < 0 ||
        n_cols <= 0)
        return NHIP_E_BADARG;
    if (n_cols > 32 * SPMV_MASK_WORDS) return NHIP_E_TOOBIG;
    if ((reinterpret_cast<uintptr_t>(cols) | reinterpret_cast<uintptr_t>(vals) |
         reinterpret_cast<uintptr_t>(mask) | reinterpret_cast<uintptr_t>(ranges)) & 15)
        return NHIP_E_BADARG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool bits_in_kernel = n_cols <= SPMV_MASK_INLINE_COLS;
    if (!bits_in_kernel) {
        const int n_mask_quads = (n_cols + 127) / 128;        // 128 bits per 16 bytes
        const int n_mask_threads = n_mask_quads * 128;        // one thread per bit, whole quads
        NHIP_LAUNCH_FIRST(spmv_mask_kernel,
                          dim3(n_mask_threads / NHIP_WG + (n_mask_threads % NHIP_WG != 0)),
                          dim3(NHIP_WG), 0, s, X + x_start, n_cols, mask, ranges,
                          4 * n_mask_quads);
        NHIP_LAUNCH_CHECK();
    }
    if (!skip_groups(side, 4 * n_slices)) return NHIP_E_BADARG;
    const dim3 grid(side.n_groups + side.n_chains);
    if (bits_in_kernel)
        NHIP_LAUNCH(spmv_sell_skip_kernel, grid, dim3(SPMV_SKIP_WG), 0, s,
                    reinterpret_cast<const SpmvSlice*>(slices), n_slices, row_len, cols, vals, X, Y,
                    nullptr, nullptr, x_start, n_cols, epi, side);
    else
        NHIP_LAUNCH_LAST(spmv_sell_skip_kernel, grid, dim3(SPMV_SKIP_WG), 0, s,
                         reinterpret_cast<const SpmvSlice*>(slices), n_slices, row_len, cols, vals,
                         X, Y, mask, ranges, x_start, n_cols, epi, side);
    NHIP_LAUNCH_CHECK();
    return 0;
}

}  // namespace

extern "C" int nhip_spmv_sell(void* stream, const int* slices, int n_slices, const int* row_len,
                              const int* cols, const float* vals, const float* X, float* Y) {
    return launch_plain(stream, slices, n_slices, row_len, cols, vals, X, Y, SpmvEpi{});
}

// The product for an X that is mostly zero.  All slices must read the same X:
// `n_cols` elements at X + x_start, n_cols <= 32 * SPMV_MASK_WORDS.  `mask` is a workspace
// of (n_cols + 127) / 128 * 4 words that the call may fill with one bit per element of X and then
// read.  One launch, or two where X has more than SPMV_MASK_INLINE_COLS elements.
extern "C" int nhip_spmv_sell_skip(void* stream, const int* slices, int n_slices,
                                   const int* row_len, const int* cols, const float* vals,
                                   const float* X, float* Y, int x_start, int n_cols,
                                   unsigned* mask) {
    return launch_skip(stream, slices, n_slices, row_len, cols, vals, X, Y, x_start, n_cols, mask,
                       nullptr, SpmvEpi{});
}

// The same, with filters (slice_epi != nullptr) or without, and with `ranges`, a second workspace of
// the size of `mask`, for the values that the set elements of an X of more than
// SPMV_MASK_INLINE_COLS elements span: without it such an X is always looked up.
extern "C" int nhip_spmv_sell_spikes(void* stream, const int* slices, int n_slices,
                                     const int* row_len, const int* cols, const float* vals,
                                     const float* X, float* Y, const int* slice_epi,
                                     const int* targets, float* F, int x_start, int n_cols,
                                     unsigned* mask, unsigned* ranges) {
    if (!ranges || (slice_epi && (!targets || !F))) return NHIP_E_BADARG;
    const SpmvEpi epi = slice_epi ? SpmvEpi{reinterpret_cast<const int4*>(slice_epi),
                                            reinterpret_cast<const FilterTarget*>(targets), F}
                                  : SpmvEpi{};
    return launch_skip(stream, slices, n_slices, row_len, cols, vals, X, Y, x_start, n_cols, mask,
                       ranges, epi);
}

// The product of spikes whose bits are in `mask` already (nhip_gemv_rows_lif_bits) and all have
// the value `one`, on the layout of spmv_sell_bits_kernel.
extern "C" int nhip_spmv_sell_bits(void* stream, const int* slices, int n_slices, const int* cols,
                                   const float* vals, float* Y, const int* slice_epi, const int* targets,
                                   float* F, int n_cols, const unsigned* mask, float one, int lanes,
                                   int index_bits) {
    SpmvSide side = take_side();
    if (n_slices == 0) return side.n_chains > 0 ? NHIP_E_BADARG : 0;  // nothing to ride in
    if (n_slices < 0 || !slices || !cols || !vals || !Y || !mask || n_cols <= 0 ||
        (slice_epi && (!targets || !F)))
        return NHIP_E_BADARG;
    if (n_slices > (1 << 28) || n_cols > 32 * SPMV_MASK_WORDS - 128 || (index_bits == 16 && n_cols > 0xffff))
        return NHIP_E_TOOBIG;
    if ((reinterpret_cast<uintptr_t>(vals) | reinterpret_cast<uintptr_t>(mask)) & 15) return NHIP_E_BADARG;
    const SpmvEpi epi = slice_epi ? SpmvEpi{reinterpret_cast<const int4*>(slice_epi),
                                            reinterpret_cast<const FilterTarget*>(targets), F}
                                  : SpmvEpi{};
    if (!skip_groups(side, lanes * n_slices)) return NHIP_E_BADARG;
    auto launch = [&](auto kernel) {
        NHIP_LAUNCH(kernel, dim3(side.n_groups + side.n_chains), dim3(SPMV_SKIP_WG), 0,
                    static_cast<hipStream_t>(stream), reinterpret_cast<const SpmvSlice*>(slices), n_slices,
                    cols, vals, Y, mask, n_cols, one, epi, side);
        return 0;
    };
    const int kind = 100 * lanes + index_bits;
    if (kind == 116) launch(spmv_sell_bits_kernel<1, 16>);
    else if (kind == 216) launch(spmv_sell_bits_kernel<2, 16>);
    else if (kind == 416) launch(spmv_sell_bits_kernel<4, 16>);
    else if (kind == 124) launch(spmv_sell_bits_kernel<1, 24>);
    else if (kind == 224) launch(spmv_sell_bits_kernel<2, 24>);
    else if (kind == 424) launch(spmv_sell_bits_kernel<4, 24>);
    else return NHIP_E_BADCLASS;
    NHIP_LAUNCH_CHECK();
    return 0;
}

// Either product with first-order filters stepped on its fresh rows: `slice_epi` holds
// {first target, number of targets, first row of the slice in its matrix, 0} per slice,
// `targets` {y_start, a bits, b bits, number of denominator coefficients} as for the dense
// products, `F` the buffer of the filter outputs.  mask == nullptr: the ordinary product.
extern "C" int nhip_spmv_sell_filter(void* stream, const int* slices, int n_slices,
                                     const int* row_len, const int* cols, const float* vals,
                                     const float* X, float* Y, const int* slice_epi,
                                     const int* targets, float* F, int x_start, int n_cols,
                                     unsigned* mask) {
    if (!slice_epi || !targets || !F) return NHIP_E_BADARG;
    const SpmvEpi epi{reinterpret_cast<const int4*>(slice_epi),
                      reinterpret_cast<const FilterTarget*>(targets), F};
    if (mask)
        return launch_skip(stream, slices, n_slices, row_len, cols, vals, X, Y, x_start, n_cols,
                           mask, nullptr, epi);
    return launch_plain(stream, slices, n_slices, row_len, cols, vals, X, Y, epi);
}
