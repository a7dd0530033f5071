// Rows of constant matrices times vectors, each row with its first- and second-order filters: decoders.
//
//   y = beta Yin + gamma + alpha A x;  F = filter(y)   for every row, one dot product each
//
// in the reference's order (clra_gemv.py:1043-1058, :1148-1153): per tile of 128 columns four partial sums of every
// fourth column, (s0 + s2) + (s1 + s3), tiles in order onto beta Yin, gamma last.  A lane carries one partial sum of
// one tile.  The kernels of gemv_rows.h read matrix and vector element by element, 32 loads each in four or more
// rounds of 16 pieces of 16 bytes, behind a chain of records (task, item, dot product, filters): 3.3 us inside
// a launch of 1,169 rows of 100 columns, 4.0 for 1,600 rows of 2,000, most of them between the records and the last product.
// Here the matrices are laid out once (nhip_lay_out_dots): the elements of a lane's partial sum lie in quads, a quad
// of all lanes of a row side by side, so eight 16-byte loads bring a tile; and a row's (or a group's) record holds
// everything there is to know about it, so matrix, vector, old output and old filter value are requested together.
// What lies past a row's end is -0 in the copy and +0 in the vector, whose product changes no sum.
//
// Measured, first wave to last: 1,169 rows of 100 columns 4.0 -> 2.6 us, 544 of 1,000 3.8 -> 2.2, 1,600 of 2,000 (with
// second-order filters) 5.2 -> 3.4; 37 x 50 rows of 1,501 columns 4.5 (active columns only) -> 4.1. What is left: record 0.3,
// matrix and vector 1.0, sums 0.4-0.7, filters 0.3. Whole steps of 100 x 2000 x 48 rate neurons (38 MB of decoders) 27.9 ->
// 19.3 us together with gemv_lanes.hip, 200 x 3000 x 20 33.9 -> 25.6.
#include "nhip_common.h"
#include "gemv_types.h"
#include "neuron_math.h"
#include "rows_side.h"

#include <type_traits>

namespace {

typedef float dots_f4 __attribute__((ext_vector_type(4)));
typedef int dots_i16 __attribute__((ext_vector_type(16)));
#define DOTS_INLINE __attribute__((always_inline))

constexpr int DTILE = 128, DSTRIDE = DTILE + 4;  // columns of a tile, its words in LDS
constexpr int DQUADS = 8, DSTEPS = 32;           // quads and elements of a lane's partial sum of a tile
constexpr size_t DOTS_SEQ_BYTES = SEQ_MAX_OPS * sizeof(NhipSeqOp) + sizeof(int) * SEQ_MAX_ROWS * SEQ_ROW_WORDS;

// One row of at most 256 columns.  n_targets < 0: no row (the list is filled up to whole groups).
struct DotRow {
    int a, x, N, n_targets;       // a: 64 bytes of the copy
    int y, yin, first_target, row;
    float alpha, beta, gamma;
    int pad;
    FilterTarget target;          // the first one
};
// Rows of one item that a group takes: row0 .. row0 + n_rows.
struct DotGroup {
    int a, row_units, N, x_start;  // copy of the item's first row, 64-byte units from row to row
    int x_stride0, row0, n_rows, n_targets;
    int y_start, y_stride0, yin_start, yin_stride0;
    float alpha, beta, gamma;
    int first_target;
    FilterTarget target;
    int x_bits;                    // not zero: X is a bit per element (32 to a word), this the float of a set one
    int pad[11];
};
static_assert(sizeof(DotRow) == 64 && sizeof(DotGroup) == 128, "tables");

__device__ __forceinline__ float dots_quad_sum(float s) {  // (s0 + s2) + (s1 + s3) in all four lanes
    s = s + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x4E, 0xF, 0xF, true));
    return s + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ void dots_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A carried sequence in the groups before those of the rows (it takes longer than they do).
#define DOTS_SIDE(lds, group)                                                                            \
    if (SIDE) {                                                                                          \
        if (group < side.n_chains) {                                                                     \
            sequence_chain(side.ops + side.chains.first_op[group],                                       \
                           side.chains.first_op[group + 1] - side.chains.first_op[group],                \
                           side.chains.n_staged[group], reinterpret_cast<NhipSeqOp*>(lds),               \
                           reinterpret_cast<int (*)[SEQ_ROW_WORDS]>(lds + SEQ_MAX_OPS * sizeof(NhipSeqOp)), threadIdx.x); \
            return;                                                                                      \
        }                                                                                                \
        group -= side.n_chains;                                                                          \
    }

// Rows of at most TP * 128 columns (TP 1 or 2), 4 * TP lanes each, of whatever items.  EQ: quads of a tile at most;
// every partial sum of the launch has `full` elements at least, `most` at most.
template <int TP, int EQ, int EPI, bool SIDE>
__global__ __launch_bounds__(NHIP_WG) __attribute__((amdgpu_waves_per_eu(4)))
void dot_rows_kernel(const DotRow* __restrict__ rows, const dots_f4* __restrict__ At, float* B,
                     const FilterTarget* __restrict__ targets, int full, int most, RowsSide side)
{
    constexpr int L = 4 * TP;
    int group = blockIdx.x;
    if constexpr (SIDE) {
        __shared__ __attribute__((aligned(16))) char lds[DOTS_SEQ_BYTES];
        DOTS_SIDE(lds, group)
    }
    const int tid = threadIdx.x, lis = tid & (L - 1), j = tid & 3, t = lis >> 2;
    const DotRow d = rows[(size_t)group * (NHIP_WG / L) + tid / L];
    const dots_f4* ap = At + (size_t)d.a * 4 + lis;
    const float* xp = B + d.x + t * DTILE + j;
    dots_f4 a[EQ];
    float x[4 * EQ];
    const int left = d.N - (t * DTILE + j);  // columns from the lane's first on
#pragma unroll
    for (int q = 0; q < EQ; ++q) a[q] = ap[q * L];
#pragma unroll
    for (int e = 0; e < 4 * EQ; ++e) {
        if (e < full) x[e] = xp[4 * e];  // uniform
        else if (e < most) x[e] = B[4 * e < left ? d.x + t * DTILE + j + 4 * e : 0];
        else x[e] = 0.0f;
    }
    const float y_old = B[d.yin];
    const float f_old = B[d.n_targets > 0 ? d.target.y_start + d.row : 0];
    float s = 0.0f;
#pragma unroll
    for (int e = 0; e < 4 * EQ; ++e) {
        if (e < full) s = fmaf(a[e >> 2][e & 3], x[e], s);
        else if (e < most) s = fmaf(a[e >> 2][e & 3], 4 * e < left ? x[e] : 0.0f, s);
    }
    s = dots_quad_sum(s);
    float sum = d.beta * y_old;
    sum = sum + d.alpha * s;
    if (TP == 2) {
        const float next = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x104, 0xF, 0xF, true));
        if (d.N > DTILE) sum = sum + d.alpha * next;  // lane i: the value of lane i + 4
    }
    if (lis == 0 && d.n_targets >= 0) {
        const float y = sum + d.gamma;
        B[d.y] = y;
        if (d.n_targets > 0) {
            B[d.target.y_start + d.row] = filter_step<EPI == EPI_FILTER2>(targets, d.target, d.row, y, f_old);
            for (int q = 1; q < d.n_targets; ++q) {
                const FilterTarget more = targets[d.first_target + q];
                float* f = B + more.y_start + d.row;
                *f = filter_step<EPI == EPI_FILTER2>(targets, more, d.row, y, *f);
            }
        }
    }
}

// Rows of any length, 4 * TP lanes each, 64 / TP of one item to a group, which stages their vector in LDS: a pass of
// TP tiles after the other.  (Element by element from memory the vector of 2,000 columns costs a wave 32 loads of 16
// pieces; a group's address path was what 1,600 such rows waited for.)
template <int TP, int EPI, bool SIDE>
__global__ __launch_bounds__(NHIP_WG) __attribute__((amdgpu_waves_per_eu(4)))
void dot_items_kernel(const DotGroup* groups, const dots_f4* __restrict__ At, float* B,
                      const FilterTarget* __restrict__ targets, RowsSide side)
{
    constexpr int L = 4 * TP, ROWS = NHIP_WG / L, COLS = TP * DTILE, XL = COLS / NHIP_WG;
    constexpr size_t X_BYTES = sizeof(float) * (TP * DSTRIDE + ROWS * TP);
    __shared__ __attribute__((aligned(16))) char lds[SIDE && DOTS_SEQ_BYTES > X_BYTES ? DOTS_SEQ_BYTES : X_BYTES];
    int group = blockIdx.x;
    DOTS_SIDE(lds, group)
    const int tid = threadIdx.x, slot = tid / L, lis = tid & (L - 1), j = tid & 3, t = lis >> 2;
    float* xs = reinterpret_cast<float*>(lds);
    float* ts = xs + TP * DSTRIDE + slot * TP;  // alpha times the tile sums of the lane's row
    // (constant address space: the whole record in two reads, with no wait for other loads)
    typedef const __attribute__((address_space(4))) dots_i16 const_i16;
    const const_i16* at = reinterpret_cast<const const_i16*>(reinterpret_cast<uintptr_t>(groups + group));
    dots_i16 w0 = at[0], w1 = at[1];
    asm volatile("" : "+s"(w0), "+s"(w1));
    struct Words { dots_i16 a, b; };
    const Words words = {w0, w1};
    const DotGroup d = __builtin_bit_cast(DotGroup, words);
    const int row = d.row0 + min(slot, d.n_rows - 1);
    const char* a0 = reinterpret_cast<const char*>(At) + ((size_t)d.a << 6) + (size_t)d.row0 * (size_t)(d.row_units << 6);
    const unsigned a_row = (unsigned)(row - d.row0) * ((unsigned)d.row_units << 6);
    float y_old = 0.0f, f_old = 0.0f, sum = 0.0f;
    for (int c0 = 0; c0 < d.N; c0 += COLS) {
        // (a lane whose tile the row does not reach reads what the row's first lane reads)
        const unsigned off = a_row + 16u * (unsigned)(c0 + t * DTILE < d.N ? lis : 0);
        const char* base = a0 + (size_t)(c0 / COLS) * (DQUADS * L * 16);
        dots_f4 a[DQUADS];
        float xv[XL];
#pragma unroll
        for (int i = 0; i < XL; ++i) {
            const int c = c0 + tid + i * NHIP_WG;
            const int from = min(c, d.N - 1);
            xv[i] = B[d.x_start + (d.x_bits ? (size_t)(from >> 5) : (size_t)from * d.x_stride0)];
            if (d.x_bits)  // uniform
                xv[i] = __float_as_int(xv[i]) >> (from & 31) & 1 ? nhip_bits(d.x_bits) : 0.0f;
        }
#pragma unroll
        for (int q = 0; q < DQUADS; ++q) a[q] = *reinterpret_cast<const dots_f4*>(base + q * (L * 16) + off);
        if (c0 == 0) {
            y_old = B[d.yin_start + (size_t)row * d.yin_stride0];
            f_old = B[d.n_targets > 0 ? d.target.y_start + row : 0];
        } else {
            __syncthreads();  // the pass before has read its vector
        }
#pragma unroll
        for (int i = 0; i < XL; ++i) {
            const int c = tid + i * NHIP_WG;
            xs[(c >> 7) * DSTRIDE + (c & (DTILE - 1))] = c0 + c < d.N ? xv[i] : 0.0f;
        }
        __syncthreads();
        const float* xp = xs + t * DSTRIDE + j;
        float s = 0.0f;
#pragma unroll
        for (int e = 0; e < DSTEPS; ++e) s = fmaf(a[e >> 2][e & 3], xp[4 * e], s);
        s = dots_quad_sum(s);
        if (j == 0) ts[t] = d.alpha * s;
        dots_sync();  // (the lanes of a row are one wave's)
        if (c0 == 0) sum = d.beta * y_old;
        const int n_tiles = min(TP, (d.N - c0 + DTILE - 1) / DTILE);  // uniform
#pragma unroll 4
        for (int k = 0; k < n_tiles; ++k) sum = sum + ts[k];
    }
    if (lis == 0 && slot < d.n_rows) {
        const float y = sum + d.gamma;
        B[d.y_start + (size_t)row * d.y_stride0] = y;
        if (d.n_targets > 0) {
            B[d.target.y_start + row] = filter_step<EPI == EPI_FILTER2>(targets, d.target, row, y, f_old);
            for (int q = 1; q < d.n_targets; ++q) {
                const FilterTarget more = targets[d.first_target + q];
                float* f = B + more.y_start + row;
                *f = filter_step<EPI == EPI_FILTER2>(targets, more, row, y, *f);
            }
        }
    }
}

// Matrix a_start, a_stride0, M x N -> its copy from 64-byte unit `out` on: row after row `row_units` units, pass after
// pass, quads of all lanes of a row side by side
struct DotMatrix { int a_start, a_stride0, M, N, out, lanes, quads, row_units; };

__global__ __launch_bounds__(NHIP_WG) void lay_out_dots_kernel(const DotMatrix* __restrict__ mats, const float* A,
                                                               dots_f4* At) {
    const DotMatrix m = mats[blockIdx.y];
    const int pass_cols = m.lanes / 4 * DTILE, passes = (m.N + pass_cols - 1) / pass_cols;
    for (int r = blockIdx.x; r < m.M; r += gridDim.x)
        for (int i = threadIdx.x; i < passes * m.quads * m.lanes; i += NHIP_WG) {
            const int lane = i % m.lanes, q = i / m.lanes % m.quads, pass = i / m.lanes / m.quads;
            const int c = pass * pass_cols + (lane >> 2) * DTILE + (lane & 3) + 16 * q;
            dots_f4 v;
            for (int k = 0; k < 4; ++k)
                v[k] = c + 4 * k < m.N ? A[m.a_start + (size_t)r * m.a_stride0 + c + 4 * k] : -0.0f;
            At[((size_t)m.out + (size_t)r * m.row_units) * 4 + i] = v;
        }
}

}  // namespace

extern "C" int nhip_lay_out_dots(void* stream, const int* matrices, int n, int max_rows, const float* A, float* At) {
    if (n == 0) return 0;
    if (n < 0 || n > 65535 || max_rows < 1 || !matrices || !A || !At || (reinterpret_cast<uintptr_t>(At) & 63))
        return NHIP_E_BADARG;
    NHIP_LAUNCH(lay_out_dots_kernel, dim3(max_rows < 1024 ? max_rows : 1024, n), dim3(NHIP_WG), 0,
                static_cast<hipStream_t>(stream), reinterpret_cast<const DotMatrix*>(matrices), A,
                reinterpret_cast<dots_f4*>(At));
    NHIP_LAUNCH_CHECK();
    return 0;
}

extern "C" int nhip_gemv_dots(void* stream, int tiles, int quads, int order, const int* records, int n_groups,
                              const float* At, float* B, const int* targets, int full, int most) {
    RowsSide side;
    if (take_carried(side) && n_groups <= 0) return NHIP_E_BADARG;  // an empty launch cannot carry it
    if (n_groups == 0) return 0;
    if (n_groups < 0 || !records || !At || !B || !targets || order < 1 || order > 2 || full < 0 || full > most)
        return NHIP_E_BADARG;
    if ((reinterpret_cast<uintptr_t>(At) & 63) || (reinterpret_cast<uintptr_t>(records) & 63)) return NHIP_E_BADARG;
    if (tiles <= 2 && most > 4 * quads) return NHIP_E_BADARG;
    side.n_gemv_groups = n_groups;
    const dim3 grid(n_groups + side.n_chains);
    const dots_f4* at = reinterpret_cast<const dots_f4*>(At);
    const FilterTarget* t = reinterpret_cast<const FilterTarget*>(targets);
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto rows = [&](auto kernel) {
        NHIP_LAUNCH(kernel, grid, dim3(NHIP_WG), 0, s, reinterpret_cast<const DotRow*>(records), at, B, t, full, most, side);
    };
    auto items = [&](auto kernel) {
        NHIP_LAUNCH(kernel, grid, dim3(NHIP_WG), 0, s, reinterpret_cast<const DotGroup*>(records), at, B, t, side);
    };
    bool known = true;
    auto pick = [&](auto epi, auto carried) {
        constexpr int E = decltype(epi)::value;
        constexpr bool C = decltype(carried)::value;
        if (tiles == 1 && quads == 2) rows(dot_rows_kernel<1, 2, E, C>);
        else if (tiles == 1 && quads == 4) rows(dot_rows_kernel<1, 4, E, C>);
        else if (tiles == 1 && quads == 8) rows(dot_rows_kernel<1, 8, E, C>);
        else if (tiles == 2 && quads == 8) rows(dot_rows_kernel<2, 8, E, C>);
        else if (tiles == 4) items(dot_items_kernel<4, E, C>);
        else if (tiles == 8) items(dot_items_kernel<8, E, C>);
        else if (tiles == 16) items(dot_items_kernel<16, E, C>);
        else known = false;
    };
    auto of_order = [&](auto epi) {
        if (side.n_chains > 0) pick(epi, std::true_type{});
        else pick(epi, std::false_type{});
    };
    if (order == 2) of_order(std::integral_constant<int, EPI_FILTER2>{});
    else of_order(std::integral_constant<int, EPI_FILTER>{});
    if (!known) return NHIP_E_BADCLASS;
    NHIP_LAUNCH_CHECK();
    return 0;
}
